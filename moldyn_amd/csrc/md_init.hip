// md_init.hip -- the reference's initialisers on the device: a blank state
// (initialize_particles, solver/src/initializer/position.rs:116-137), the
// U / FCC lattices (position.rs:24-104) and Maxwell-Boltzmann velocities
// with pair negation (velocity.rs:6-29), written straight into the records;
// and the transfer of whole states between the records and the caller's arrays
// (N x 3 doubles, type-major).
#include "md_common.h"

namespace md {

// every slot of both record buffers: position 0 (NaN on padding slots),
// velocity and force 0, the group's type (initialize_particles)
template <typename FT>
__global__ __launch_bounds__(256) void k_init_blank(Rec<FT>* __restrict__ r0, Rec<FT>* __restrict__ r1,
                                                    const GroupInfo* __restrict__ groups, int n_groups,
                                                    int64_t n_slots) {
    const int64_t s = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (s >= n_slots) return;
    int g = 0;
    while (g + 1 < n_groups && s >= groups[g + 1].start) ++g;
    const GroupInfo& G = groups[g];
    const double p = s - G.start < G.count ? 0.0 : __builtin_nan("");
    Rec<FT> r{};
    r.x = r.y = r.z = p;
    r.vx = r.vy = r.vz = 0.0;
    r.fx = r.fy = r.fz = (FT)0;
    r.type = (uint32_t)G.type;
    r0[s] = r;
    r1[s] = r;
}

// UnitCell::{U, FCC}: site k of cell (x, y, z), cell = x gy gz + y gz + z, at
// start + (X + o_k) a with o_0 = 0 and the FCC face centres o_1..o_3
template <typename FT>
__global__ __launch_bounds__(256) void k_init_lattice(Rec<FT>* __restrict__ rec, int64_t slot0, int64_t sites,
                                                      int fcc, double s0, double s1, double s2, int64_t gy,
                                                      int64_t gz, double a) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= sites) return;
    const int64_t cell = fcc ? i / 4 : i;
    const int k = fcc ? (int)(i % 4) : 0;
    const double X = (double)(cell / (gy * gz)), Y = (double)((cell / gz) % gy), Z = (double)(cell % gz);
    const double ox = (k == 2 || k == 3) ? 0.5 : 0.0;
    const double oy = (k == 1 || k == 3) ? 0.5 : 0.0;
    const double oz = (k == 1 || k == 2) ? 0.5 : 0.0;
    Rec<FT>& r = rec[slot0 + i];
    r.x = s0 + (X + ox) * a;
    r.y = s1 + (Y + oy) * a;
    r.z = s2 + (Z + oz) * a;
}

// SplitMix64 output number k (0-based) of the stream seeded with `seed`
__device__ __forceinline__ uint64_t sm64_at(uint64_t seed, uint64_t k) {
    uint64_t z = seed + (k + 1) * 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

__device__ __forceinline__ double open01_at(uint64_t seed, uint64_t k) {
    return ((double)(sm64_at(seed, k) >> 11) + 0.5) * (1.0 / 9007199254740992.0);
}

// standard normal number j of the sequence: Box-Muller pair j / 2 from
// uniforms 2 (j / 2) and 2 (j / 2) + 1, cosine for even j, sine for odd j
__device__ __forceinline__ double normal_at(uint64_t seed, uint64_t j) {
    const uint64_t p = j >> 1;
    const double u1 = open01_at(seed, 2 * p), u2 = open01_at(seed, 2 * p + 1);
    const double r = sqrt(-2.0 * log(u1));
    const double th = 6.283185307179586 * u2;
    return (j & 1) ? r * sin(th) : r * cos(th);
}

// particle i < n / 2 gets sigma (N_3i, N_3i+1, N_3i+2), particle i + n / 2
// its negation; an odd last particle keeps its velocity
template <typename FT>
__global__ __launch_bounds__(256) void k_init_mb(Rec<FT>* __restrict__ rec, int64_t slot0, int64_t n, double sigma,
                                                 uint64_t seed) {
    const int64_t h = n / 2;
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= h) return;
    const double vx = sigma * normal_at(seed, 3 * (uint64_t)i);
    const double vy = sigma * normal_at(seed, 3 * (uint64_t)i + 1);
    const double vz = sigma * normal_at(seed, 3 * (uint64_t)i + 2);
    Rec<FT>& a = rec[slot0 + i];
    a.vx = vx;
    a.vy = vy;
    a.vz = vz;
    Rec<FT>& b = rec[slot0 + i + h];
    b.vx = -vx;
    b.vy = -vy;
    b.vz = -vz;
}

// ---------------------------------------------------------------- state transfer
//
// The caller's arrays cross the host link as they are, and a thread per slot
// moves its record between them and the record buffers: bound by the link (and
// by the host's page faults on fresh arrays), not by these kernels.  Building
// and unpacking the padded 64- or 80-byte records on the host took one pass of
// a single core and a copy per buffer (1,000,000 atoms: upload 31 ms, download
// of everything 25 ms; 1.7 and 9 ms now, most of the download being page faults
// on the caller's new arrays; 256 replicas of 2,300,000 atoms: 70 and 56 ms, 3.6
// and 17.6 ms now).

// the group of slot s (groups are in slot order)
__device__ __forceinline__ const GroupInfo& group_of(const GroupInfo* __restrict__ groups, int n_groups, int64_t s) {
    int lo = 0, hi = n_groups;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (groups[mid].start <= s) lo = mid;
        else hi = mid;
    }
    return groups[lo];  // of the groups that start there the last, the one that is not empty
}

template <typename FT>
__global__ __launch_bounds__(256) void k_put_state(DevState d, int n_groups, StateIO io) {
    const int64_t s = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (s >= d.n_slots) return;
    const GroupInfo& G = group_of(d.groups, n_groups, s);
    const int64_t k = s - G.start, a = G.first_atom + k;
    const bool pad = k >= G.count;
    if (pad ? io.a0 != 0 : (a < io.a0 || a >= io.a1)) return;
    Rec<FT> r{};
    r.type = (uint32_t)G.type;
    if (pad) {
        r.x = r.y = r.z = __builtin_nan("");
    } else {
        const int64_t o = 3 * (a - io.a0);
        if (io.x) {
            r.x = io.x[o];
            r.y = io.x[o + 1];
            r.z = io.x[o + 2];
        }
        if (io.v) {
            r.vx = io.v[o];
            r.vy = io.v[o + 1];
            r.vz = io.v[o + 2];
        }
    }
    ((Rec<FT>*)d.rec[0])[s] = r;
    ((Rec<FT>*)d.rec[1])[s] = r;
    d.pot[s] = 0.0;
    d.vir[s] = 0.0;
}

template <typename FT>
__global__ __launch_bounds__(256) void k_put_forces(DevState d, int n_groups, StateIO io) {
    const int64_t s = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (s >= d.n_slots) return;
    const GroupInfo& G = group_of(d.groups, n_groups, s);
    const int64_t k = s - G.start, a = G.first_atom + k;
    if (k >= G.count || a < io.a0 || a >= io.a1) return;
    Rec<FT>& r = ((Rec<FT>*)d.rec[ctrl_in(d, G.rep).cur & 1])[s];
    const int64_t o = a - io.a0;
    r.fx = io.f ? (FT)io.f[3 * o] : (FT)0;
    r.fy = io.f ? (FT)io.f[3 * o + 1] : (FT)0;
    r.fz = io.f ? (FT)io.f[3 * o + 2] : (FT)0;
    d.pot[s] = io.pot ? io.pot[o] : 0.0;
    d.vir[s] = io.vir ? io.vir[o] : 0.0;
}

// Three doubles per lane of a wave to out[3 (atom - a0)], atom = first + lane,
// for the atoms in [lo, hi): through LDS, so that consecutive lanes store
// consecutive words (the destination may be host memory, where every store that
// does not fill a line is a transfer of its own).
__device__ __forceinline__ void wave_store3(double* lds, double* out, int64_t a0, int64_t first, int64_t lo, int64_t hi,
                                            double x, double y, double z) {
    const int wl = threadIdx.x & 63;
    __builtin_amdgcn_wave_barrier();
    lds[3 * wl] = x;
    lds[3 * wl + 1] = y;
    lds[3 * wl + 2] = z;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        const int e = wl + 64 * q;
        const int64_t a = first + e / 3;
        if (a >= lo && a < hi) out[3 * (first - a0) + e] = lds[e];
    }
}

template <typename FT>
__global__ __launch_bounds__(256) void k_get_state(DevState d, int n_groups, StateIO io) {
    __shared__ double s_out[4][64 * 3];
    double* const lds = s_out[threadIdx.x >> 6];
    const int64_t s = (int64_t)blockIdx.x * 256 + threadIdx.x;
    // a wave's 64 slots belong to one group (groups are whole tiles of 64 slots or more)
    const int64_t s0 = s - (threadIdx.x & 63);
    if (s0 >= d.n_slots) return;
    const GroupInfo& G = group_of(d.groups, n_groups, s0);
    const int64_t first = G.first_atom + (s0 - G.start), a = first + (s - s0);
    const int64_t end = G.first_atom + G.count;
    const int64_t lo = io.a0, hi = end < io.a1 ? end : io.a1;
    if (first >= hi || first + 64 <= lo) return;
    if (io.x || io.v || io.f) {
        const Rec<FT> r = ((const Rec<FT>*)d.rec[ctrl_in(d, G.rep).cur & 1])[s];
        if (io.x) wave_store3(lds, io.x, io.a0, first, lo, hi, r.x, r.y, r.z);
        if (io.v) wave_store3(lds, io.v, io.a0, first, lo, hi, r.vx, r.vy, r.vz);
        if (io.f) wave_store3(lds, io.f, io.a0, first, lo, hi, (double)r.fx, (double)r.fy, (double)r.fz);
    }
    if (a < lo || a >= hi) return;
    if (io.pot) io.pot[a - io.a0] = d.pot[s];
    if (io.vir) io.vir[a - io.a0] = d.vir[s];
}

static inline unsigned blocks_for(int64_t n) { return (unsigned)((n + 255) / 256); }

#define MD_LAUNCH_IO(KERNEL)                                                                                  \
    if (d.n_slots <= 0) return hipSuccess;                                                                   \
    if (fp32) hipLaunchKernelGGL((KERNEL<float>), dim3(blocks_for(d.n_slots)), dim3(256), 0, st, d, n_groups, io); \
    else hipLaunchKernelGGL((KERNEL<double>), dim3(blocks_for(d.n_slots)), dim3(256), 0, st, d, n_groups, io);     \
    return hipGetLastError();
hipError_t launch_put_state(const DevState& d, bool fp32, int n_groups, const StateIO& io, hipStream_t st) {
    MD_LAUNCH_IO(k_put_state)
}
hipError_t launch_put_forces(const DevState& d, bool fp32, int n_groups, const StateIO& io, hipStream_t st) {
    MD_LAUNCH_IO(k_put_forces)
}
hipError_t launch_get_state(const DevState& d, bool fp32, int n_groups, const StateIO& io, hipStream_t st) {
    MD_LAUNCH_IO(k_get_state)
}
#undef MD_LAUNCH_IO

hipError_t launch_init_blank(const DevState& d, bool fp32, const GroupInfo* groups, int n_groups, int64_t n_slots,
                             hipStream_t st) {
    if (n_slots <= 0) return hipSuccess;
    if (fp32)
        hipLaunchKernelGGL(k_init_blank<float>, dim3(blocks_for(n_slots)), dim3(256), 0, st, (Rec<float>*)d.rec[0],
                           (Rec<float>*)d.rec[1], groups, n_groups, n_slots);
    else
        hipLaunchKernelGGL(k_init_blank<double>, dim3(blocks_for(n_slots)), dim3(256), 0, st, (Rec<double>*)d.rec[0],
                           (Rec<double>*)d.rec[1], groups, n_groups, n_slots);
    return hipGetLastError();
}

hipError_t launch_init_lattice(void* rec, bool fp32, int64_t slot0, int64_t sites, bool fcc, const double start[3],
                               const int64_t grid[3], double a, hipStream_t st) {
    if (sites <= 0) return hipSuccess;
    if (fp32)
        hipLaunchKernelGGL(k_init_lattice<float>, dim3(blocks_for(sites)), dim3(256), 0, st, (Rec<float>*)rec, slot0,
                           sites, fcc ? 1 : 0, start[0], start[1], start[2], grid[1], grid[2], a);
    else
        hipLaunchKernelGGL(k_init_lattice<double>, dim3(blocks_for(sites)), dim3(256), 0, st, (Rec<double>*)rec,
                           slot0, sites, fcc ? 1 : 0, start[0], start[1], start[2], grid[1], grid[2], a);
    return hipGetLastError();
}

hipError_t launch_init_mb(void* rec, bool fp32, int64_t slot0, int64_t n, double sigma, uint64_t seed,
                          hipStream_t st) {
    if (n / 2 <= 0) return hipSuccess;
    if (fp32)
        hipLaunchKernelGGL(k_init_mb<float>, dim3(blocks_for(n / 2)), dim3(256), 0, st, (Rec<float>*)rec, slot0, n,
                           sigma, seed);
    else
        hipLaunchKernelGGL(k_init_mb<double>, dim3(blocks_for(n / 2)), dim3(256), 0, st, (Rec<double>*)rec, slot0, n,
                           sigma, seed);
    return hipGetLastError();
}

}  // namespace md
