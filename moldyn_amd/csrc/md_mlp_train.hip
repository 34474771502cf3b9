// md_mlp_train.hip -- training kernels of the learned per-atom energy
// surrogate (FP32), on frames of one periodic system size.
//
// Pair lists (all pairs within the cutoff, ascending j) and features are
// built once per data set.  A minibatch of M atoms (whole frames, taken in any
// order through a frame list) goes through
//   features   G,
//   forward    A1 = X W1^T, H1 = silu(A1 + b1), A2 = H1 W2^T, H2 = silu(A2 + b2),
//              y = H2 w3 + b3, E = e_scale y + e_shift,
//   backward   D2 = w3 * silu'(A2), T = D2 W2, D1 = T * silu'(A1), dE/dG = e_scale inv_std (D1 W1),
//   forces     F_i = sum_j (c_i + c_j)(r_ij) d_ij / r_ij (pair lists),
//   loss       L = w_e mean (E - E_ref)^2 + w_f mean (F - F_ref)^2,
//   gradient   the energy term by back-propagation and the force term by the
//              double backward through dE/dG:
//              U = d L / d(dE/dG) (pair kernel), V1 = U~ W1^T, PP = V1 silu'(A1),
//              V2 = PP W2^T, G2 = V2 w3 silu''(A2) + dy D2, G1 = (G2 W2) silu'(A1)
//              + T V1 silu''(A1), dW2 = G2^T H1 + D2^T PP, dW1 = G1^T X + D1^T U~,
//              db2 = sum G2, db1 = sum G1, dw3 = sum (V2 silu'(A2) + dy H2), db3 = sum dy,
//   update     Adam.
// The network runs in two kernels on the FP32 matrix cores, k_tr_net (forward
// and force backward) and k_tr_net_grad (double backward and parameter
// gradients); between them only the pre-activations A1, A2 and T go through
// memory.  The blocks' gradients are added in a fixed order.
#include "md_common.h"
#include "md_train.h"

namespace md {

constexpr float kPiT = 3.14159265358979323846f;

// silu(a) and its first two derivatives
struct Silu3 {
    float h, d1, d2;
};
__device__ __forceinline__ Silu3 silu3(float a) {
    const float s = 1.0f / (1.0f + expf(-a));
    return {a * s, s * (1.0f + a * (1.0f - s)), s * (1.0f - s) * (2.0f + a * (1.0f - 2.0f * s))};
}

// ---------------------------------------------------------------- network (FP32 MFMA)
//
// A block of eight waves takes tiles of 32 rows (atoms); wave w owns columns
// 16 w .. 16 w + 15 of every 128-column matrix, and its slices of the weights
// stay in its registers as matrix operands over all tiles.  The rows' matrices
// pass from layer to layer through LDS.  Tiles of 64 rows spill registers in
// k_tr_net_grad (65,536 rows: 162 us, 128 us with 32) and leave CUs idle on
// small minibatches (6,655 rows: 44 and 25 us).
// What bounds them is the FP32 matrix rate with the SiLU evaluations between
// the products (two waves per SIMD: the products and the elementwise work
// overlap little): 65,536 rows take 76 us (82 kFLOP a row, 71 TFLOP/s) and 128 us
// (155 kFLOP, 79 TFLOP/s) of the 154 TFLOP/s a large FP32 product reaches here.
// Before, a tiled FP32 product on the vector units per layer with elementwise
// passes in between and the weight gradients in 128 splits: 1.93 ms per
// minibatch of 65,536 rows with the pair kernels, 0.31 ms now.
// v_mfma_f32_16x16x4_f32, lane l = 16 g + c: operand A holds row c, operand B
// column c, both at the k of lane group g; the result holds rows 4 g + i
// (i = 0..3) of column c.  The k of a product may come in any order that A and
// B share: four products in a row take k = 16 kk + 4 g + i, so that a lane reads
// its four A values as one 16-byte word of a row.
// LDS rows are 132 (36) words apart: the 16-byte reads of 16 rows, and the
// 4-byte accesses of rows 4 g + i, each fall on all 64 banks.
// A1, A2 and T are stored as the result fragments lie in the registers (16
// bytes a lane, consecutive lanes on consecutive words), for k_tr_net_grad to
// read in the same way.
typedef float f32x4 __attribute__((ext_vector_type(4)));
constexpr int kTrBS = 512, kTrW = kTrBS / 64;
constexpr int kLdH = kMlpH + 4, kLdX = kMlpK + 4;

// acc[t] += rows 16 t .. of `act` (LDS, stride LD, K = 16 KK columns) times the
// wave's weight slice
template <int KK, int LD, int TT>
__device__ __forceinline__ void tile_gemm(const float* act, const f32x4 (&wgt)[KK], f32x4 (&acc)[TT]) {
    const int c = threadIdx.x & 15, g = (threadIdx.x >> 4) & 3;
#pragma unroll
    for (int kk = 0; kk < KK; ++kk)
#pragma unroll
        for (int t = 0; t < TT; ++t) {
            const f32x4 a = *reinterpret_cast<const f32x4*>(act + (16 * t + c) * LD + 16 * kk + 4 * g);
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], wgt[kk][i], acc[t], 0, 0, 0);
        }
}

// acc[ct] += (columns m0 .. m0 + 15 of P)^T times columns 16 ct .. of Q, over
// the tile's TR rows (both in LDS)
template <int TR, int LDP, int LDQ, int CT>
__device__ __forceinline__ void tile_outer(const float* P, int m0, const float* Q, f32x4 (&acc)[CT]) {
    const int c = threadIdx.x & 15, g = (threadIdx.x >> 4) & 3;
#pragma unroll
    for (int kk = 0; kk < TR / 16; ++kk)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int r = 16 * kk + 4 * g + i;
            const float a = P[r * LDP + m0 + c];
#pragma unroll
            for (int ct = 0; ct < CT; ++ct)
                acc[ct] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, Q[r * LDQ + 16 * ct + c], acc[ct], 0, 0, 0);
        }
}

// a result fragment into rows 16 t + 4 g + i, column n of an LDS matrix
template <int LD>
__device__ __forceinline__ void frag_to_lds(float* m, int t, int n, const f32x4& v) {
    const int g = (threadIdx.x >> 4) & 3;
#pragma unroll
    for (int i = 0; i < 4; ++i) m[(16 * t + 4 * g + i) * LD + n] = v[i];
}

// the weight slice B[k][n] = W[n * ldn + k * ldk], k = 16 kk + 4 g + i
template <int KK>
__device__ __forceinline__ void load_slice(f32x4 (&wgt)[KK], const float* W, int n, int ldn, int ldk) {
    const int g = (threadIdx.x >> 4) & 3;
#pragma unroll
    for (int kk = 0; kk < KK; ++kk)
#pragma unroll
        for (int i = 0; i < 4; ++i) wgt[kk][i] = W[n * ldn + (16 * kk + 4 * g + i) * ldk];
}

// normalised features of the tile's rows (0 past the last)
__device__ __forceinline__ void stage_x(const TrainState& t, int64_t row0, int64_t M, float* sx) {
    for (int e = threadIdx.x; e < kTrRows * (kMlpK / 4); e += kTrBS) {
        const int r = e / (kMlpK / 4), k = 4 * (e % (kMlpK / 4));
        f32x4 x = {0.0f, 0.0f, 0.0f, 0.0f};
        const int64_t row = row0 + r;
        if (row < M) {
            const int64_t b = row / t.n_atoms, i = row - b * t.n_atoms;
            x = *reinterpret_cast<const f32x4*>(t.G + ((int64_t)t.bf[b] * t.n_atoms + i) * kMlpK + k);
#pragma unroll
            for (int q = 0; q < 4; ++q) x[q] = (x[q] - t.g_mean[k + q]) * t.g_inv_std[k + q];
        }
        *reinterpret_cast<f32x4*>(sx + r * kLdX + k) = x;
    }
}

// Forward, and the backward to dE/dG: E and Gam of the M rows; `keep` stores
// A1, A2 and T for k_tr_net_grad.
__global__ __launch_bounds__(kTrBS) void k_tr_net(TrainState t, int64_t M, int64_t n_tiles, int keep) {
    constexpr int TR = kTrRows, TT = TR / 16;
    __shared__ __align__(16) float sx[TR * kLdX], sh[TR * kLdH], sd[TR * kLdH];
    __shared__ float sy[kTrW][TR];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, c = lane & 15, g = lane >> 4;
    const int n = 16 * w + c;
    const float* th = t.theta;
    f32x4 w1t[2], w2t[8], w2[8], w1[8];
    load_slice(w1t, th + kMlpOffW1, n, kMlpK, 1);
    load_slice(w2t, th + kMlpOffW2, n, kMlpH, 1);
    load_slice(w2, th + kMlpOffW2, n, 1, kMlpH);
    load_slice(w1, th + kMlpOffW1, 16 * (w & 1) + c, 1, kMlpK);
    const float b1 = th[kMlpOffB1 + n], b2 = th[kMlpOffB2 + n], w3 = th[kMlpOffW3 + n];
    const float gsc = t.e_scale * t.g_inv_std[16 * (w & 1) + c];
    for (int64_t tile = blockIdx.x; tile < n_tiles; tile += gridDim.x) {
        const int64_t row0 = tile * TR;
        const int64_t fo = (tile * kTrW + w) * TT * 64 + lane;  // this lane's words of the tile's fragments
        stage_x(t, row0, M, sx);
        __syncthreads();
        f32x4 s1[TT];
        {
            f32x4 a[TT];
#pragma unroll
            for (int q = 0; q < TT; ++q) a[q] = f32x4{b1, b1, b1, b1};
            tile_gemm<2, kLdX, TT>(sx, w1t, a);
#pragma unroll
            for (int q = 0; q < TT; ++q) {
                if (keep) reinterpret_cast<f32x4*>(t.A1)[fo + q * 64] = a[q];
                f32x4 h;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const Silu3 f = silu3(a[q][i]);
                    h[i] = f.h;
                    s1[q][i] = f.d1;
                }
                frag_to_lds<kLdH>(sh, q, n, h);
            }
        }
        __syncthreads();
        {
            f32x4 a[TT];
#pragma unroll
            for (int q = 0; q < TT; ++q) a[q] = f32x4{b2, b2, b2, b2};
            tile_gemm<8, kLdH, TT>(sh, w2t, a);
#pragma unroll
            for (int q = 0; q < TT; ++q) {
                if (keep) reinterpret_cast<f32x4*>(t.A2)[fo + q * 64] = a[q];
                f32x4 d, y;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const Silu3 f = silu3(a[q][i]);
                    d[i] = w3 * f.d1;
                    y[i] = w3 * f.h;
                }
                frag_to_lds<kLdH>(sd, q, n, d);
                // the wave's 16 columns of each row's y
#pragma unroll
                for (int o = 1; o < 16; o <<= 1)
#pragma unroll
                    for (int i = 0; i < 4; ++i) y[i] += __shfl_xor(y[i], o, 16);
                if (c == 0)
#pragma unroll
                    for (int i = 0; i < 4; ++i) sy[w][16 * q + 4 * g + i] = y[i];
            }
        }
        __syncthreads();
        if (threadIdx.x < TR && row0 + threadIdx.x < M) {
            float y = th[kMlpOffB3];
#pragma unroll
            for (int q = 0; q < kTrW; ++q) y += sy[q][threadIdx.x];
            t.E[row0 + threadIdx.x] = t.e_scale * y + t.e_shift;
        }
        {
            f32x4 a[TT];
#pragma unroll
            for (int q = 0; q < TT; ++q) a[q] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            tile_gemm<8, kLdH, TT>(sd, w2, a);
#pragma unroll
            for (int q = 0; q < TT; ++q) {
                if (keep) reinterpret_cast<f32x4*>(t.T)[fo + q * 64] = a[q];
                frag_to_lds<kLdH>(sh, q, n, a[q] * s1[q]);
            }
        }
        __syncthreads();
        // 2 TT tiles of 16 x 16: wave w takes column half w % 2 of row tiles
        // w / 2, w / 2 + 4, ...
        for (int q = w >> 1; q < TT; q += kTrW / 2) {
            f32x4 a[1] = {f32x4{0.0f, 0.0f, 0.0f, 0.0f}};
            tile_gemm<8, kLdH, 1>(sh + 16 * q * kLdH, w1, a);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int64_t row = row0 + 16 * q + 4 * g + i;
                if (row < M) t.Gam[row * kMlpK + 16 * (w & 1) + c] = gsc * a[0][i];
            }
        }
    }
}

// Gradient of the loss through E (dy) and through dE/dG (U, the adjoint of
// Gam), summed over the block's rows: parameters in theta's order at
// gpart[block][kMlpNP].  Rows past M add nothing: their U, X and dy are 0.
__global__ __launch_bounds__(kTrBS) void k_tr_net_grad(TrainState t, int64_t M, int64_t n_tiles) {
    constexpr int TR = kTrRows, TT = TR / 16;
    __shared__ __align__(16) float su[TR * kLdX], sx[TR * kLdX];
    __shared__ __align__(16) float sp[TR * kLdH], sh[TR * kLdH], sg[TR * kLdH], sd[TR * kLdH];
    __shared__ float sdy[TR];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, c = lane & 15, g = lane >> 4;
    const int n = 16 * w + c;
    const float* th = t.theta;
    f32x4 w1t[2], w2t[8], w2[8];
    load_slice(w1t, th + kMlpOffW1, n, kMlpK, 1);
    load_slice(w2t, th + kMlpOffW2, n, kMlpH, 1);
    load_slice(w2, th + kMlpOffW2, n, 1, kMlpH);
    const float w3 = th[kMlpOffW3 + n];
    const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    f32x4 gw2[8], gw1[2];
#pragma unroll
    for (int q = 0; q < 8; ++q) gw2[q] = zero;
    gw1[0] = gw1[1] = zero;
    float gw3 = 0.0f, gb2 = 0.0f, gb1 = 0.0f, gb3 = 0.0f;
    for (int64_t tile = blockIdx.x; tile < n_tiles; tile += gridDim.x) {
        const int64_t row0 = tile * TR;
        const int64_t fo = (tile * kTrW + w) * TT * 64 + lane;
        __syncthreads();  // the last tile's reads of su, sx, sg and sh
        stage_x(t, row0, M, sx);
        for (int e = threadIdx.x; e < TR * (kMlpK / 4); e += kTrBS) {
            const int r = e / (kMlpK / 4), k = 4 * (e % (kMlpK / 4));
            f32x4 u = zero;
            if (row0 + r < M) {
                u = *reinterpret_cast<const f32x4*>(t.U + (row0 + r) * kMlpK + k);
#pragma unroll
                for (int q = 0; q < 4; ++q) u[q] *= t.e_scale * t.g_inv_std[k + q];
            }
            *reinterpret_cast<f32x4*>(su + r * kLdX + k) = u;
        }
        if (threadIdx.x < TR) {
            const float dy = row0 + threadIdx.x < M ? t.dy[row0 + threadIdx.x] : 0.0f;
            sdy[threadIdx.x] = dy;
            gb3 += dy;
        }
        __syncthreads();
        f32x4 s1[TT], q1[TT], d1[TT];  // silu'(A1), T V1 silu''(A1), D1
        {
            f32x4 v[TT];
#pragma unroll
            for (int q = 0; q < TT; ++q) v[q] = zero;
            tile_gemm<2, kLdX, TT>(su, w1t, v);  // V1 = Ut W1^T
#pragma unroll
            for (int q = 0; q < TT; ++q) {
                const f32x4 a = reinterpret_cast<const f32x4*>(t.A1)[fo + q * 64];
                const f32x4 tt = reinterpret_cast<const f32x4*>(t.T)[fo + q * 64];
                f32x4 h;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const Silu3 f = silu3(a[i]);
                    h[i] = f.h;
                    s1[q][i] = f.d1;
                    q1[q][i] = tt[i] * v[q][i] * f.d2;
                    d1[q][i] = tt[i] * s1[q][i];
                }
                frag_to_lds<kLdH>(sh, q, n, h);
                frag_to_lds<kLdH>(sp, q, n, v[q] * s1[q]);  // PP
            }
        }
        __syncthreads();
        {
            f32x4 v[TT];
#pragma unroll
            for (int q = 0; q < TT; ++q) v[q] = zero;
            tile_gemm<8, kLdH, TT>(sp, w2t, v);  // V2 = PP W2^T
#pragma unroll
            for (int q = 0; q < TT; ++q) {
                const f32x4 a = reinterpret_cast<const f32x4*>(t.A2)[fo + q * 64];
                f32x4 g2, d2;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const Silu3 f = silu3(a[i]);
                    const float dy = sdy[16 * q + 4 * g + i];
                    d2[i] = w3 * f.d1;
                    g2[i] = v[q][i] * w3 * f.d2 + dy * d2[i];
                    gw3 += v[q][i] * f.d1 + dy * f.h;
                    gb2 += g2[i];
                }
                frag_to_lds<kLdH>(sg, q, n, g2);
                frag_to_lds<kLdH>(sd, q, n, d2);
            }
        }
        __syncthreads();
        // dW2 += G2^T H1 + D2^T PP
        tile_outer<TR, kLdH, kLdH, 8>(sg, 16 * w, sh, gw2);
        tile_outer<TR, kLdH, kLdH, 8>(sd, 16 * w, sp, gw2);
        {
            f32x4 v[TT];
#pragma unroll
            for (int q = 0; q < TT; ++q) v[q] = zero;
            tile_gemm<8, kLdH, TT>(sg, w2, v);  // G2 W2
            __syncthreads();                    // sg and sh are read: G1 and D1 take their place
#pragma unroll
            for (int q = 0; q < TT; ++q) {
                f32x4 g1;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    g1[i] = v[q][i] * s1[q][i] + q1[q][i];
                    gb1 += g1[i];
                }
                frag_to_lds<kLdH>(sg, q, n, g1);
                frag_to_lds<kLdH>(sh, q, n, d1[q]);
            }
        }
        __syncthreads();
        // dW1 += G1^T X + D1^T Ut
        tile_outer<TR, kLdH, kLdX, 2>(sg, 16 * w, sx, gw1);
        tile_outer<TR, kLdH, kLdX, 2>(sh, 16 * w, su, gw1);
    }
    float* out = t.gpart + (int64_t)blockIdx.x * kMlpNP;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int m = 16 * w + 4 * g + i;
#pragma unroll
        for (int ct = 0; ct < 8; ++ct) out[kMlpOffW2 + m * kMlpH + 16 * ct + c] = gw2[ct][i];
#pragma unroll
        for (int ct = 0; ct < 2; ++ct) out[kMlpOffW1 + m * kMlpK + 16 * ct + c] = gw1[ct][i];
    }
    // column sums over the four lane groups
#pragma unroll
    for (int o = 16; o < 64; o <<= 1) {
        gw3 += __shfl_xor(gw3, o, 64);
        gb2 += __shfl_xor(gb2, o, 64);
        gb1 += __shfl_xor(gb1, o, 64);
    }
    if (g == 0) {
        out[kMlpOffW3 + n] = gw3;
        out[kMlpOffB2 + n] = gb2;
        out[kMlpOffB1 + n] = gb1;
    }
    if (w == 0) {  // threads < TR took the rows' dy
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) gb3 += __shfl_xor(gb3, o, 64);
        if (lane == 0) out[kMlpOffB3] = gb3;
    }
}

// The blocks' gradients added in block order, four interleaved FP64 sums per
// parameter, then what the caller asked for: stored (accumulate 0) or added
// (accumulate 1) to t.grad, or one Adam step on theta (adam).
struct AdamArgs {
    float lr, b1, b2, eps, c1, c2;  // c1 = 1 - b1^step, c2 = 1 - b2^step
};
template <bool ADAM>
__global__ __launch_bounds__(256) void k_tr_grad_sum(TrainState t, int nb, int accumulate, AdamArgs a) {
    __shared__ double s[4][64];
    const int q = threadIdx.x >> 6, p = blockIdx.x * 64 + (threadIdx.x & 63);
    double v = 0.0;
    if (p < kMlpNP)
#pragma unroll 8
        for (int b = q; b < nb; b += 4) v += (double)t.gpart[(int64_t)b * kMlpNP + p];
    s[q][threadIdx.x & 63] = v;
    __syncthreads();
    if (q != 0 || p >= kMlpNP) return;
    const float gi = (float)((s[0][threadIdx.x] + s[1][threadIdx.x]) + (s[2][threadIdx.x] + s[3][threadIdx.x]));
    if (!ADAM) {
        t.grad[p] = accumulate ? t.grad[p] + gi : gi;
        return;
    }
    const float mi = a.b1 * t.adam_m[p] + (1.0f - a.b1) * gi;
    const float vi = a.b2 * t.adam_v[p] + (1.0f - a.b2) * gi * gi;
    t.adam_m[p] = mi;
    t.adam_v[p] = vi;
    t.theta[p] -= a.lr * (mi / a.c1) / (sqrtf(vi / a.c2) + a.eps);
}

// ---------------------------------------------------------------- pairs, features

// Positions of frame f staged in LDS 256 at a time; atom i visits every
// j != i of its frame in ascending order and calls visit(j) for the pairs with
// r^2 < rc^2 (the reference minimum image).
template <class Visit>
__device__ __forceinline__ void tr_all_pairs(const TrainState& t, int f, int i, Visit visit) {
    __shared__ double sx[256], sy[256], sz[256];
    const int n = t.n_atoms;
    const double* P = t.pos + (int64_t)f * n * 3;
    const double bx = t.box[3 * f], by = t.box[3 * f + 1], bz = t.box[3 * f + 2];
    double xi = 0, yi = 0, zi = 0;
    if (i < n) {
        xi = P[3 * i];
        yi = P[3 * i + 1];
        zi = P[3 * i + 2];
    }
    const double rc2 = (double)t.rc * t.rc;
    for (int j0 = 0; j0 < n; j0 += 256) {
        __syncthreads();
        const int jl = j0 + threadIdx.x;
        if (jl < n) {
            sx[threadIdx.x] = P[3 * jl];
            sy[threadIdx.x] = P[3 * jl + 1];
            sz[threadIdx.x] = P[3 * jl + 2];
        }
        __syncthreads();
        const int cnt = min(256, n - j0);
        if (i < n)
            for (int q = 0; q < cnt; ++q) {
                if (j0 + q == i) continue;
                const double dx = min_image(sx[q] - xi, bx), dy = min_image(sy[q] - yi, by),
                             dz = min_image(sz[q] - zi, bz);
                const double r2 = (dx * dx + dy * dy) + dz * dz;
                if (r2 < rc2) visit(j0 + q);
            }
    }
}

// neighbour counts of every atom of frames [f0, f0 + nf), and their maximum
__global__ __launch_bounds__(256) void k_tr_count(TrainState t, int f0, int nf, int32_t* max_cnt) {
    const int f = f0 + blockIdx.y;
    const int i = blockIdx.x * 256 + threadIdx.x;
    int c = 0;
    tr_all_pairs(t, f, i, [&](int) { ++c; });
    if (i < t.n_atoms) {
        t.ncnt[(int64_t)f * t.n_atoms + i] = c;
        atomicMax(max_cnt, c);
    }
}

// neighbour indices (ascending) of every atom of frames [f0, f0 + nf)
__global__ __launch_bounds__(256) void k_tr_fill(TrainState t, int f0, int nf) {
    const int f = f0 + blockIdx.y;
    const int i = blockIdx.x * 256 + threadIdx.x;
    int32_t* out = t.nbr + ((int64_t)f * t.n_atoms + (i < t.n_atoms ? i : 0)) * t.cap;
    int c = 0;
    tr_all_pairs(t, f, i, [&](int j) {
        if (c < t.cap) out[c] = j;
        ++c;
    });
}

// displacement x_j - x_i (minimum image) and distance of a listed pair
struct TrPair {
    double dx, dy, dz;
    float r;
};
__device__ __forceinline__ TrPair tr_pair(const double* P, double xi, double yi, double zi, double bx, double by,
                                          double bz, int j) {
    TrPair p;
    p.dx = min_image(P[3 * j] - xi, bx);
    p.dy = min_image(P[3 * j + 1] - yi, by);
    p.dz = min_image(P[3 * j + 2] - zi, bz);
    p.r = (float)sqrt((p.dx * p.dx + p.dy * p.dy) + p.dz * p.dz);
    return p;
}

// G of every atom of frames [f0, f0 + nf) from the pair lists
__global__ __launch_bounds__(256) void k_tr_features(TrainState t, int f0, int nf) {
    const int f = f0 + blockIdx.y;
    const int n = t.n_atoms;
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const int64_t row = (int64_t)f * n + i;
    const double* P = t.pos + (int64_t)f * n * 3;
    const double bx = t.box[3 * f], by = t.box[3 * f + 1], bz = t.box[3 * f + 2];
    const double xi = P[3 * i], yi = P[3 * i + 1], zi = P[3 * i + 2];
    float g[kMlpK];
#pragma unroll
    for (int k = 0; k < kMlpK; ++k) g[k] = 0.0f;
    const int cnt = t.ncnt[row];
    const int32_t* nb = t.nbr + row * t.cap;
    for (int q = 0; q < cnt; ++q) {
        const TrPair p = tr_pair(P, xi, yi, zi, bx, by, bz, nb[q]);
        const float fc = 0.5f * (cosf(kPiT * p.r / t.rc) + 1.0f);
#pragma unroll
        for (int k = 0; k < kMlpK; ++k) {
            const float u = p.r - t.mu[k];
            g[k] = fmaf(expf(-u * u * t.inv_2w2), fc, g[k]);
        }
    }
    float* out = t.G + row * kMlpK;
#pragma unroll
    for (int k = 0; k < kMlpK; ++k) out[k] = g[k];
}

// per-feature sum, sum of squares, min, max over all atoms (block partials)
__global__ __launch_bounds__(256) void k_tr_feature_stats(TrainState t, int64_t n_rows, double* part) {
    const int k = threadIdx.x % kMlpK, lane_row = threadIdx.x / kMlpK;  // 8 rows at a time
    double s = 0, s2 = 0, mn = 1e300, mx = -1e300;
    for (int64_t r = (int64_t)blockIdx.x * 8 + lane_row; r < n_rows; r += (int64_t)gridDim.x * 8) {
        const double v = t.G[r * kMlpK + k];
        s += v;
        s2 += v * v;
        mn = fmin(mn, v);
        mx = fmax(mx, v);
    }
    __shared__ double sh[4][256];
    sh[0][threadIdx.x] = s;
    sh[1][threadIdx.x] = s2;
    sh[2][threadIdx.x] = mn;
    sh[3][threadIdx.x] = mx;
    __syncthreads();
    if (threadIdx.x < kMlpK) {
        for (int q = 1; q < 8; ++q) {
            const int o = q * kMlpK + threadIdx.x;
            s += sh[0][o];
            s2 += sh[1][o];
            mn = fmin(mn, sh[2][o]);
            mx = fmax(mx, sh[3][o]);
        }
        double* p = part + (int64_t)blockIdx.x * 4 * kMlpK;
        p[threadIdx.x] = s;
        p[kMlpK + threadIdx.x] = s2;
        p[2 * kMlpK + threadIdx.x] = mn;
        p[3 * kMlpK + threadIdx.x] = mx;
    }
}

// ---------------------------------------------------------------- pair kernels
//
// L lanes per atom share its pairs (pair q goes to lane q % L) and add their
// sums at the end: a lane per atom leaves 65,536 atoms one wave per SIMD, with
// nothing to run while a neighbour's row is on its way.  The 32 basis values of
// a pair are bound by the exponentials: one base-2 hardware exponential each,
// with the factor log2(e) / (2 w^2) rounded once (the argument carries the same
// two roundings as before).  L = 8 below four waves per SIMD at L = 4.
// Minibatch of 65,536 atoms of about 33 pairs: forces 88 -> 47 us, adjoint 76 ->
// 48 us; of 6,655 atoms: 66 -> 12 and 56 -> 17 us.
struct TrBasis {
    float r, fcw, dfc;  // distance, cutoff / w^2, derivative of the cutoff
};
__device__ __forceinline__ TrBasis tr_basis(const TrainState& t, float r) {
    float sn, cs;
    sincospif(r / t.rc, &sn, &cs);
    return {r, 0.5f * (cs + 1.0f) * t.inv_w2, -0.5f * kPiT / t.rc * sn};
}
// d/dr of basis function k: exp(-u^2 / 2 w^2) (f_c' - u f_c / w^2), u = r - mu_k
__device__ __forceinline__ float tr_dg(const TrainState& t, const TrBasis& b, int k) {
    const float u = b.r - t.mu[k];
    return __builtin_amdgcn_exp2f(-(u * u) * t.exp2_2w2) * fmaf(-u, b.fcw, b.dfc);
}

// sum over the L lanes of an atom (every lane gets it)
template <int L>
__device__ __forceinline__ float lanes_sum(float v) {
#pragma unroll
    for (int o = 1; o < L; o <<= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// Forces of the minibatch frames from Gam (rows r = b n + i), the loss terms
// and their derivatives phi = dL/dF, dy = dL/dy.
template <int L>
__global__ __launch_bounds__(256) void k_tr_forces(TrainState t, double* loss_part) {
    const int b = blockIdx.y, f = t.bf[b];
    const int n = t.n_atoms;
    const int i = blockIdx.x * (256 / L) + threadIdx.x / L, sub = threadIdx.x % L;
    double le = 0.0, lf = 0.0;
    if (i < n) {
        const int64_t ri = (int64_t)b * n + i;  // row in the minibatch
        const int64_t di = (int64_t)f * n + i;  // row in the data set
        const double* P = t.pos + (int64_t)f * n * 3;
        const double bx = t.box[3 * f], by = t.box[3 * f + 1], bz = t.box[3 * f + 2];
        const double xi = P[3 * i], yi = P[3 * i + 1], zi = P[3 * i + 2];
        f32x4 gi[kMlpK / 4];
#pragma unroll
        for (int k = 0; k < kMlpK / 4; ++k) gi[k] = reinterpret_cast<const f32x4*>(t.Gam + ri * kMlpK)[k];
        float fx = 0.f, fy = 0.f, fz = 0.f;
        const int cnt = t.ncnt[di];
        const int32_t* nb = t.nbr + di * t.cap;
        for (int q = sub; q < cnt; q += L) {
            const int j = nb[q];
            const f32x4* gj = reinterpret_cast<const f32x4*>(t.Gam + ((int64_t)b * n + j) * kMlpK);
            f32x4 gs[kMlpK / 4];
#pragma unroll
            for (int k = 0; k < kMlpK / 4; ++k) gs[k] = gj[k];
            const TrPair p = tr_pair(P, xi, yi, zi, bx, by, bz, j);
            const TrBasis bs = tr_basis(t, p.r);
            float c = 0.f;
#pragma unroll
            for (int k = 0; k < kMlpK; ++k) c = fmaf(gi[k / 4][k % 4] + gs[k / 4][k % 4], tr_dg(t, bs, k), c);
            const float s = c / p.r;
            fx = fmaf(s, (float)p.dx, fx);
            fy = fmaf(s, (float)p.dy, fy);
            fz = fmaf(s, (float)p.dz, fz);
        }
        fx = lanes_sum<L>(fx);
        fy = lanes_sum<L>(fy);
        fz = lanes_sum<L>(fz);
        if (sub == 0) {
            const float ex = fx - t.Fref[3 * di], ey = fy - t.Fref[3 * di + 1], ez = fz - t.Fref[3 * di + 2];
            const float ee = t.E[ri] - t.Eref[di];
            t.F[3 * ri] = fx;
            t.F[3 * ri + 1] = fy;
            t.F[3 * ri + 2] = fz;
            const float cf = 2.0f * t.w_f / (3.0f * (float)t.n_total);
            t.phi[3 * ri] = cf * ex;
            t.phi[3 * ri + 1] = cf * ey;
            t.phi[3 * ri + 2] = cf * ez;
            t.dy[ri] = 2.0f * t.w_e / (float)t.n_total * ee * t.e_scale;
            le = (double)ee * ee;
            lf = ((double)ex * ex + (double)ey * ey) + (double)ez * ez;
        }
    }
    // block sums of the squared errors (fixed order)
    __shared__ double sl[2][4];
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
        le += __shfl_xor(le, o, 64);
        lf += __shfl_xor(lf, o, 64);
    }
    if ((threadIdx.x & 63) == 0) {
        sl[0][threadIdx.x >> 6] = le;
        sl[1][threadIdx.x >> 6] = lf;
    }
    __syncthreads();
    if (threadIdx.x < 2) {
        const int64_t blk = (int64_t)blockIdx.y * gridDim.x + blockIdx.x;
        const double* v = sl[threadIdx.x];
        loss_part[2 * blk + threadIdx.x] = (v[0] + v[1]) + (v[2] + v[3]);
    }
}

// out[0..1] = block partials of the squared errors, summed in a fixed order
__global__ __launch_bounds__(256) void k_tr_loss_sum(const double* __restrict__ part, int64_t blocks,
                                                    double* __restrict__ out) {
    __shared__ double s[256];
    const int col = threadIdx.x & 1, row = threadIdx.x >> 1;
    double v = 0.0;
    for (int64_t q = row; q < blocks; q += 128) v += part[2 * q + col];
    s[threadIdx.x] = v;
    for (int o = 128; o >= 2; o >>= 1) {
        __syncthreads();
        if ((int)threadIdx.x < o) s[threadIdx.x] += s[threadIdx.x + o];
    }
    if (threadIdx.x < 2) out[threadIdx.x] = s[threadIdx.x];
}

// U_i = sum_j ((phi_i - phi_j) . d_ij / r_ij) dg(r_ij)
template <int L>
__global__ __launch_bounds__(256) void k_tr_u(TrainState t) {
    const int b = blockIdx.y, f = t.bf[b];
    const int n = t.n_atoms;
    const int i = blockIdx.x * (256 / L) + threadIdx.x / L, sub = threadIdx.x % L;
    if (i >= n) return;
    const int64_t ri = (int64_t)b * n + i;
    const int64_t di = (int64_t)f * n + i;
    const double* P = t.pos + (int64_t)f * n * 3;
    const double bx = t.box[3 * f], by = t.box[3 * f + 1], bz = t.box[3 * f + 2];
    const double xi = P[3 * i], yi = P[3 * i + 1], zi = P[3 * i + 2];
    const float px = t.phi[3 * ri], py = t.phi[3 * ri + 1], pz = t.phi[3 * ri + 2];
    float u[kMlpK];
#pragma unroll
    for (int k = 0; k < kMlpK; ++k) u[k] = 0.0f;
    const int cnt = t.ncnt[di];
    const int32_t* nb = t.nbr + di * t.cap;
    for (int q = sub; q < cnt; q += L) {
        const int j = nb[q];
        const float* pj = t.phi + 3 * ((int64_t)b * n + j);
        const float qx = px - pj[0], qy = py - pj[1], qz = pz - pj[2];
        const TrPair p = tr_pair(P, xi, yi, zi, bx, by, bz, j);
        const float proj = (qx * (float)p.dx + qy * (float)p.dy + qz * (float)p.dz) / p.r;
        const TrBasis bs = tr_basis(t, p.r);
#pragma unroll
        for (int k = 0; k < kMlpK; ++k) u[k] = fmaf(proj, tr_dg(t, bs, k), u[k]);
    }
    // the lanes' sums: each halving leaves a lane half of the values to add up
    // (lane group o keeps the upper half), L lanes then hold 32 / L values each
#pragma unroll
    for (int o = 1, w = kMlpK / 2; o < L; o <<= 1, w >>= 1) {
        const bool up = sub & o;
#pragma unroll
        for (int k = 0; k < kMlpK / 2; ++k) {
            if (k >= w) break;
            const float keep = up ? u[k + w] : u[k], give = up ? u[k] : u[k + w];
            u[k] = keep + __shfl_xor(give, o, 64);
        }
    }
    int k0 = 0;
#pragma unroll
    for (int o = 1, w = kMlpK / 2; o < L; o <<= 1, w >>= 1) k0 += (sub & o) ? w : 0;
    f32x4* out = reinterpret_cast<f32x4*>(t.U + ri * kMlpK + k0);
#pragma unroll
    for (int k = 0; k < kMlpK / L / 4; ++k) out[k] = f32x4{u[4 * k], u[4 * k + 1], u[4 * k + 2], u[4 * k + 3]};
}

// ---------------------------------------------------------------- launchers

static inline unsigned nblk(int64_t n) { return (unsigned)((n + 255) / 256); }

hipError_t tr_count_pairs(const TrainState& t, int f0, int nf, int32_t* max_cnt, hipStream_t st) {
    hipLaunchKernelGGL(k_tr_count, dim3(nblk(t.n_atoms), nf), dim3(256), 0, st, t, f0, nf, max_cnt);
    return hipGetLastError();
}

hipError_t tr_fill_pairs(const TrainState& t, int f0, int nf, hipStream_t st) {
    hipLaunchKernelGGL(k_tr_fill, dim3(nblk(t.n_atoms), nf), dim3(256), 0, st, t, f0, nf);
    return hipGetLastError();
}

hipError_t tr_features(const TrainState& t, int f0, int nf, hipStream_t st) {
    hipLaunchKernelGGL(k_tr_features, dim3(nblk(t.n_atoms), nf), dim3(256), 0, st, t, f0, nf);
    return hipGetLastError();
}

hipError_t tr_feature_stats(const TrainState& t, int64_t rows, double* part, int blocks, hipStream_t st) {
    hipLaunchKernelGGL(k_tr_feature_stats, dim3(blocks), dim3(256), 0, st, t, rows, part);
    return hipGetLastError();
}

hipError_t tr_forward_backward(const TrainState& t, int nf, bool keep, hipStream_t st) {
    const int64_t M = (int64_t)nf * t.n_atoms, tiles = (M + kTrRows - 1) / kTrRows;
    hipLaunchKernelGGL(k_tr_net, dim3((unsigned)(tiles < t.n_cu ? tiles : t.n_cu)), dim3(kTrBS), 0, st, t, M, tiles,
                       keep ? 1 : 0);
    return hipGetLastError();
}

// lanes per atom of the pair kernels
static inline int pair_lanes(const TrainState& t, int nf) {
    return (int64_t)nf * t.n_atoms * 4 >= (int64_t)t.n_cu * 16 * 64 ? 4 : 8;
}

int64_t tr_loss_blocks(const TrainState& t, int nf) {
    const int a = 256 / pair_lanes(t, nf);  // atoms per block
    return (int64_t)((t.n_atoms + a - 1) / a) * nf;
}

hipError_t tr_forces(const TrainState& t, int nf, double* loss_part, hipStream_t st) {
    const int l = pair_lanes(t, nf), a = 256 / l;
    const dim3 grid((unsigned)((t.n_atoms + a - 1) / a), nf);
    if (l == 4) hipLaunchKernelGGL(k_tr_forces<4>, grid, dim3(256), 0, st, t, loss_part);
    else hipLaunchKernelGGL(k_tr_forces<8>, grid, dim3(256), 0, st, t, loss_part);
    return hipGetLastError();
}

hipError_t tr_loss_sum(const TrainState& t, int nf, const double* loss_part, double* out, hipStream_t st) {
    hipLaunchKernelGGL(k_tr_loss_sum, dim3(1), dim3(256), 0, st, loss_part, tr_loss_blocks(t, nf), out);
    return hipGetLastError();
}

// Gradient of the minibatch loss: the blocks' sums at t.gpart, their number in *parts.
hipError_t tr_gradient(const TrainState& t, int nf, int* parts, hipStream_t st) {
    const int64_t M = (int64_t)nf * t.n_atoms;
    const int l = pair_lanes(t, nf), a = 256 / l;
    const dim3 grid((unsigned)((t.n_atoms + a - 1) / a), nf);
    if (l == 4) hipLaunchKernelGGL(k_tr_u<4>, grid, dim3(256), 0, st, t);
    else hipLaunchKernelGGL(k_tr_u<8>, grid, dim3(256), 0, st, t);
    const int64_t tiles = (M + kTrRows - 1) / kTrRows;
    *parts = (int)(tiles < t.n_cu ? tiles : t.n_cu);
    hipLaunchKernelGGL(k_tr_net_grad, dim3(*parts), dim3(kTrBS), 0, st, t, M, tiles);
    return hipGetLastError();
}

hipError_t tr_grad_sum(const TrainState& t, int parts, bool accumulate, hipStream_t st) {
    hipLaunchKernelGGL(k_tr_grad_sum<false>, dim3((kMlpNP + 63) / 64), dim3(256), 0, st, t, parts, accumulate ? 1 : 0,
                       AdamArgs{});
    return hipGetLastError();
}

hipError_t tr_adam(const TrainState& t, int parts, float lr, int step, hipStream_t st) {
    const AdamArgs a{lr, 0.9f, 0.999f, 1e-8f, 1.0f - powf(0.9f, (float)step), 1.0f - powf(0.999f, (float)step)};
    hipLaunchKernelGGL(k_tr_grad_sum<true>, dim3((kMlpNP + 63) / 64), dim3(256), 0, st, t, parts, 0, a);
    return hipGetLastError();
}

}  // namespace md
