// The host side of the C ABI (md_api.hip) on a stand-in for the device: device
// memory is host memory with a budget, launches move states and touch the
// arrays they would write.  Built under AddressSanitizer, so a launch on freed
// memory ends the program.  Prints "<case> passed" for the case in argv[1].
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <map>
#include <string>
#include <vector>

#include "md_device.h"
#include "moldyn_hip.h"

using namespace md;

static size_t g_budget = (size_t)1 << 32, g_live = 0;
static std::map<void*, size_t> g_size;
static hipError_t g_last = hipSuccess;
static int g_builds = 0, g_failed_allocs = 0;

extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
    if (n > g_budget || g_live > g_budget - n) {
        ++g_failed_allocs;
        *p = nullptr;
        return g_last = hipErrorOutOfMemory;
    }
    *p = malloc(n);
    g_size[*p] = n;
    g_live += n;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    if (p) {
        g_live -= g_size.at(p);
        g_size.erase(p);
        free(p);
    }
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return (*p = malloc(n)) ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipHostFree(void* p) { return free(p), hipSuccess; }
hipError_t hipHostGetDevicePointer(void** d, void* h, unsigned) { return *d = h, hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { return memcpy(d, s, n), hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
    return memcpy(d, s, n), hipSuccess;
}
hipError_t hipMemsetAsync(void* p, int v, size_t n, hipStream_t) { return memset(p, v, n), hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return *s = nullptr, hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipErrorNotSupported; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t*) { return hipErrorNotSupported; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return *e = nullptr, hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t*, hipGraph_t, hipGraphNode_t*, char*, size_t) {
    return hipErrorNotSupported;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipErrorNotSupported; }
hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipGetDeviceCount(int* n) { return *n = 1, hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { return *v = 256, hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
    memset(p, 0, sizeof *p);
    strcpy(p->gcnArchName, "gfx950");
    return hipSuccess;
}
const char* hipGetErrorString(hipError_t e) { return e == hipSuccess ? "no error" : "error"; }
hipError_t hipGetLastError(void) {
    const hipError_t e = g_last;
    g_last = hipSuccess;
    return e;
}
}

namespace md {

static hipError_t launched() { return hipGetLastError(); }

// every atom of [a0, a1): visit(slot, atom - a0)
template <typename F>
static void each_atom(const DevState& d, int n_groups, const StateIO& io, F visit) {
    for (int g = 0; g < n_groups; ++g)
        for (int64_t k = 0; k < d.groups[g].count; ++k) {
            const int64_t a = d.groups[g].first_atom + k;
            if (a >= io.a0 && a < io.a1) visit(d.groups[g].start + k, a - io.a0);
        }
}
hipError_t launch_put_state(const DevState& d, bool, int n_groups, const StateIO& io, hipStream_t) {
    each_atom(d, n_groups, io, [&](int64_t s, int64_t o) {
        for (int b = 0; b < 2; ++b) {
            Rec<float>& r = ((Rec<float>*)d.rec[b])[s];
            r = Rec<float>{};
            if (io.x) r.x = io.x[3 * o], r.y = io.x[3 * o + 1], r.z = io.x[3 * o + 2];
            if (io.v) r.vx = io.v[3 * o], r.vy = io.v[3 * o + 1], r.vz = io.v[3 * o + 2];
        }
        d.pot[s] = d.vir[s] = 0.0;
    });
    return launched();
}
hipError_t launch_put_forces(const DevState& d, bool, int n_groups, const StateIO& io, hipStream_t) {
    each_atom(d, n_groups, io, [&](int64_t s, int64_t o) {
        Rec<float>& r = ((Rec<float>*)d.rec[0])[s];
        if (io.f) r.fx = (float)io.f[3 * o], r.fy = (float)io.f[3 * o + 1], r.fz = (float)io.f[3 * o + 2];
        d.pot[s] = io.pot ? io.pot[o] : 0.0;
        d.vir[s] = io.vir ? io.vir[o] : 0.0;
    });
    return launched();
}
hipError_t launch_get_state(const DevState& d, bool, int n_groups, const StateIO& io, hipStream_t) {
    each_atom(d, n_groups, io, [&](int64_t s, int64_t o) {
        const Rec<float>& r = ((const Rec<float>*)d.rec[0])[s];
        if (io.x) io.x[3 * o] = r.x, io.x[3 * o + 1] = r.y, io.x[3 * o + 2] = r.z;
        if (io.v) io.v[3 * o] = r.vx, io.v[3 * o + 1] = r.vy, io.v[3 * o + 2] = r.vz;
        if (io.f) io.f[3 * o] = r.fx, io.f[3 * o + 1] = r.fy, io.f[3 * o + 2] = r.fz;
        if (io.pot) io.pot[o] = d.pot[s];
        if (io.vir) io.vir[o] = d.vir[s];
    });
    return launched();
}
hipError_t launch_build(const DevState& d, bool, hipStream_t) {
    ++g_builds;
    const size_t n = (size_t)d.n_slots;
    d.ncount[0] = d.ncount[n - 1] = 0;
    d.nbr[0] = d.nbr[n * d.list_cap - 1] = 0;
    d.cell_hdr[0][0] = d.cell_hdr[1][0] = 0;
    d.cell_slots[0][0] = d.cell_slots[1][(size_t)d.cell_plane * d.cell_cap - 1] = 0;
    return launched();
}
hipError_t launch_step(const DevState&, bool, int, hipStream_t) { return launched(); }
hipError_t launch_pack(const DevState&, bool, int, hipStream_t) { return launched(); }
hipError_t launch_dpos(const DevState&, int, hipStream_t) { return launched(); }
hipError_t launch_prof_init(const DevState&, hipStream_t) { return launched(); }
hipError_t launch_prime(const DevState&, const RepParams&, double*, int, MlpStat*, RepCtrl*, hipStream_t) {
    return launched();
}
hipError_t launch_epilogue(const DevState& d, int par, RepCtrl* c, RepStats* s, hipStream_t) {
    memcpy(c, d.ctrl + (size_t)par * d.n_reps, sizeof(RepCtrl) * d.n_reps);
    *s = *d.stats;
    return launched();
}
hipError_t launch_finalize(const DevState&, int, bool, bool, hipStream_t) { return launched(); }
hipError_t launch_drift(const DevState&, int, hipStream_t) { return launched(); }
hipError_t launch_allpairs(const DevState&, int, bool, hipStream_t) { return launched(); }
hipError_t launch_ap_force(const DevState&, int, bool, hipStream_t) { return launched(); }
hipError_t launch_ap_finish(const DevState&, int, hipStream_t) { return launched(); }
hipError_t launch_insert_all(const DevState&, bool, int, hipStream_t) { return launched(); }
hipError_t launch_force_eval(const DevState&, bool, int, hipStream_t) { return launched(); }
hipError_t launch_reduce_state(const DevState&, bool, int, hipStream_t) { return launched(); }
hipError_t launch_scale(const DevState&, bool, int64_t, int64_t, double, int, hipStream_t) { return launched(); }
hipError_t launch_wrap(const DevState&, bool, int, hipStream_t) { return launched(); }
hipError_t launch_mlp_desc(const DevState&, int, bool, int, hipStream_t) { return launched(); }
hipError_t launch_mlp_net(const DevState&, int, hipStream_t) { return launched(); }
hipError_t launch_mlp_force(const DevState&, int, bool, hipStream_t) { return launched(); }
hipError_t launch_mlp_convert(const DevState&, hipStream_t) { return launched(); }
hipError_t launch_init_blank(const DevState&, bool, const GroupInfo*, int, int64_t, hipStream_t) { return launched(); }
hipError_t launch_init_lattice(void*, bool, int64_t, int64_t, bool, const double*, const int64_t*, double,
                               hipStream_t) {
    return launched();
}
hipError_t launch_init_mb(void*, bool, int64_t, int64_t, double, uint64_t, hipStream_t) { return launched(); }

}  // namespace md

#define CHECK(cond)                                                                  \
    do {                                                                             \
        if (!(cond)) {                                                               \
            fprintf(stderr, "FAILED line %d: %s\n", __LINE__, #cond);                 \
            exit(1);                                                                 \
        }                                                                            \
    } while (0)

static md_ctx* context(int64_t n, std::vector<double>& x, std::vector<double>& v) {
    md_ctx* c = nullptr;
    const double mass = 66.335, box[3] = {30.0, 30.0, 30.0};
    CHECK(md_create(&c, 1, &n, &mass, box) == MD_OK);
    x.resize((size_t)n * 3);
    v.resize((size_t)n * 3);
    for (size_t i = 0; i < x.size(); ++i) {
        x[i] = (double)(i % 29) + 1e-6 * (double)i;
        v[i] = -1e-3 * (double)i;
    }
    CHECK(md_upload_state(c, x.data(), v.data(), box) == MD_OK);
    return c;
}

// Options whose lists do not fit are refused each time they are set, nothing
// runs on the lists that were given back, and options that fit are taken.
static void lists() {
    std::vector<double> x, v;
    md_ctx* c = context(4096, x, v);
    md_options o;
    CHECK(md_get_options(c, &o) == MD_OK);
    CHECK(md_update_force(c) == MD_OK && g_builds == 1);
    o.list_capacity = 1 << 28;
    for (int k = 0; k < 2; ++k) {
        CHECK(md_set_options(c, &o) == MD_ERR_NOMEM);
        CHECK(md_update_force(c) != MD_OK && g_builds == 1);
        CHECK(md_step(c, 0.002, nullptr, nullptr, 1) != MD_OK);
        md_stats st;
        CHECK(md_get_stats(c, &st) == MD_OK);
    }
    std::vector<double> x2(x.size()), v2(v.size());
    CHECK(md_download_state(c, x2.data(), v2.data(), nullptr, nullptr, nullptr, nullptr) == MD_OK);
    CHECK(x2 == x && v2 == v);
    o.list_capacity = 64;
    CHECK(md_set_options(c, &o) == MD_OK);
    CHECK(md_update_force(c) == MD_OK && g_builds == 2);
    md_destroy(c);
    CHECK(g_live == 0);
}

// A layout that does not fit is refused each time, and a context without one
// runs nothing until it has one again.
static void layout() {
    std::vector<double> x, v;
    md_ctx* c = context(2000, x, v);
    md_options o;
    CHECK(md_get_options(c, &o) == MD_OK);
    const size_t budget = g_budget;
    o.block_size = 128;
    g_budget = (size_t)1 << 20;
    const double box[3] = {30.0, 30.0, 30.0};
    for (int k = 0; k < 2; ++k) {
        CHECK(md_set_options(c, &o) == MD_ERR_NOMEM);
        CHECK(md_update_force(c) != MD_OK && md_step(c, 0.002, nullptr, nullptr, 1) != MD_OK);
        CHECK(md_upload_state(c, x.data(), v.data(), box) != MD_OK);
        CHECK(md_download_state(c, x.data(), nullptr, nullptr, nullptr, nullptr, nullptr) != MD_OK);
        CHECK(md_apply_boundary_conditions(c) != MD_OK && md_init_velocities(c, 0, 0, 100.0, 1) != MD_OK);
    }
    CHECK(g_builds == 0);
    g_budget = budget;
    CHECK(md_set_options(c, &o) == MD_OK);
    CHECK(md_upload_state(c, x.data(), v.data(), box) == MD_OK && md_update_force(c) == MD_OK && g_builds == 1);
    md_destroy(c);
    CHECK(g_live == 0);
}

// States move as well on a device without room for staging: everything in and
// out again, with the last piece not a whole one.
static void staging() {
    const int64_t n = 60001;
    const size_t budget = g_budget;
    const double mass = 66.335, box[3] = {30.0, 30.0, 30.0};
    std::vector<double> x(3 * n), v(3 * n), f(3 * n), pot(n), vir(n);
    for (int64_t i = 0; i < n; ++i) {
        for (int k = 0; k < 3; ++k) {
            x[3 * i + k] = 1e-4 * (double)i + k;
            v[3 * i + k] = -1e-3 * (double)(3 * i + k);
            f[3 * i + k] = (double)(float)(0.25 * (double)i + k);
        }
        pot[i] = 3.0 * (double)i;
        vir[i] = -1.0 * (double)i;
    }
    for (int room = 0; room < 2; ++room) {
        md_ctx* e = nullptr;
        CHECK(md_create(&e, 1, &n, &mass, box) == MD_OK);
        if (!room) g_budget = g_live;
        const int failed = g_failed_allocs;
        CHECK(md_upload_state(e, x.data(), v.data(), box) == MD_OK);
        CHECK(md_upload_forces(e, f.data(), pot.data(), vir.data()) == MD_OK);
        std::vector<double> x2(3 * n), v2(3 * n), f2(3 * n), p2(n), w2(n);
        CHECK(md_download_state(e, x2.data(), v2.data(), f2.data(), p2.data(), w2.data(), nullptr) == MD_OK);
        CHECK(x2 == x && v2 == v && f2 == f && p2 == pot && w2 == vir);
        CHECK((g_failed_allocs > failed) == !room);
        CHECK(md_update_force(e) == MD_OK);  // a refused staging is no error of a later launch
        g_budget = budget;
        md_destroy(e);
    }
    CHECK(g_live == 0);
}

// Device memory of a list context per slot: records, step records, drifted
// positions, type, potential and virial, a list of 8 entries and its length, and
// two cells of 8 slots and a header in both grid buffers; small arrays aside.
static void footprint() {
    const int64_t n = 1 << 20;
    md_ctx* c = nullptr;
    const double mass = 66.335, box[3] = {400.0, 400.0, 400.0};
    CHECK(md_create(&c, 1, &n, &mass, box) == MD_OK);
    md_stats st;
    CHECK(md_get_stats(c, &st) == MD_OK);
    const size_t per = 2 * sizeof(Rec<float>) + 2 * sizeof(CRec) + sizeof(double4) + 1 + 2 * sizeof(double) +
                       sizeof(int32_t) * (st.list_capacity + 1) + 2 * 2 * (8 + sizeof(int32_t) * st.cell_capacity);
    printf("%.2f bytes per slot, %zu expected\n", (double)g_live / n, per);
    CHECK(g_live <= per * n + ((size_t)4 << 20));
    md_destroy(c);
}

int main(int argc, char** argv) {
    const std::string what = argc > 1 ? argv[1] : "";
    if (what == "lists") lists();
    else if (what == "layout") layout();
    else if (what == "staging") staging();
    else if (what == "footprint") footprint();
    else return 2;
    printf("%s passed\n", what.c_str());
    return 0;
}
