// mlp.hip -- a small fully connected network trained and evaluated by hand-written kernels (learned
// warm start of steady runs; no reference counterpart).
//
// Network: n_in -> width (tanh) -> ... -> width (tanh) -> n_out (linear), FP32.  Parameters are one
// flat array: for each layer l the weights W_l [out x in] (row-major) then the biases b_l [out].
// Features are normalised as (f - in_shift) * in_scale and outputs de-normalised as
// y * out_scale + out_shift inside the kernels.
//
// Kernels: for networks of width <= 128 the whole-network kernels below (k_net, k_wgrad, k_adam_net).  For wider
// ones an LDS-tiled FP32 GEMM on the matrix cores (64x64 block tile, one 32x32 v_mfma_f32_32x32x2_f32
// accumulator per wave) with strided operands and fused
// epilogues (bias, tanh, tanh-derivative), split along K with a fixed-order second pass for the
// weight gradients (deterministic); column sums for the bias gradients; the squared-error gradient;
// Adam.  There a training step (batch gather by a counter-based hash, forward, backward, Adam, step
// counter) reads its step number from device memory, so it is captured once into a hipGraph and
// replayed.
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <random>
#include <string>
#include <vector>

#include "mlp.hpp"
#include "mstcfd.h"

namespace {

#define HIPCHK(expr)                                                                                     \
    do {                                                                                                 \
        hipError_t _e = (expr);                                                                          \
        if (_e != hipSuccess)                                                                            \
            return mst::fail(MST_E_HIP, std::string(#expr) + ": " + hipGetErrorString(_e));              \
    } while (0)

constexpr int TM = 64, TN = 64, TK = 16, GT = 256;
typedef float floatx16 __attribute__((ext_vector_type(16)));
enum { EPI_NONE = 0, EPI_BIAS = 1, EPI_BIAS_TANH = 2, EPI_DTANH = 3 };

struct GemmArgs {
    const float *A, *B;  // A(m,k) = A[m*sam + k*sak], B(k,n) = B[k*sbk + n*sbn]
    float *C;            // C(m,n) = C[m*ldc + n] (+ z * cz for split K)
    int64_t M, N, K;
    int64_t sam, sak, sbk, sbn, ldc;
    const float *bias;   // EPI_BIAS*: bias[n]
    const float *P;      // EPI_DTANH: C *= 1 - P(m,n)^2, P(m,n) = P[m*ldc + n]
    int64_t kchunk, cz;  // split K: block z covers k in [z*kchunk, (z+1)*kchunk)
};

template <int EPI>
__global__ __launch_bounds__(GT) void k_gemm(const GemmArgs g) {
    __shared__ float As[TK][TM + 4];
    __shared__ float Bs[TK][TN + 4];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int wm = (wv >> 1) * 32, wn = (wv & 1) * 32;  // the wave's 32 x 32 quarter of the 64 x 64 tile
    const int64_t m0 = (int64_t)blockIdx.y * TM, n0 = (int64_t)blockIdx.x * TN;
    const int64_t k0 = (int64_t)blockIdx.z * g.kchunk;
    const int64_t k1 = k0 + g.kchunk < g.K ? k0 + g.kchunk : g.K;
    floatx16 acc;
#pragma unroll
    for (int r = 0; r < 16; r++) acc[r] = 0.f;
    for (int64_t kt = k0; kt < k1; kt += TK) {
        // 1024 elements per tile, 4 per lane, zero outside the matrices
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int e = tid + r * GT;
            const int am = e % TM, ak = e / TM;  // A tile: TK x TM, m fastest
            const int64_t gm = m0 + am, gk = kt + ak;
            As[ak][am] = (gm < g.M && gk < k1) ? g.A[gm * g.sam + gk * g.sak] : 0.f;
            const int bn = e % TN, bk = e / TN;
            const int64_t gn = n0 + bn, gk2 = kt + bk;
            Bs[bk][bn] = (gn < g.N && gk2 < k1) ? g.B[gk2 * g.sbk + gn * g.sbn] : 0.f;
        }
        __syncthreads();
        // v_mfma_f32_32x32x2_f32: A(i, k) from lane i + 32k, B(k, j) from lane j + 32k
#pragma unroll
        for (int k = 0; k < TK; k += 2) {
            const float av = As[k + (lane >> 5)][wm + (lane & 31)];
            const float bv = Bs[k + (lane >> 5)][wn + (lane & 31)];
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(av, bv, acc, 0, 0, 0);
        }
        __syncthreads();
    }
    float *C = g.C + (int64_t)blockIdx.z * g.cz;
    // D(i, j) in lane j + 32 ((i / 4) % 2), register (i % 4) + 4 (i / 8)
    const int64_t n = n0 + wn + (lane & 31);
#pragma unroll
    for (int r = 0; r < 16; r++) {
        const int64_t m = m0 + wm + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
        if (m >= g.M || n >= g.N) continue;
        float v = acc[r];
        if constexpr (EPI == EPI_BIAS || EPI == EPI_BIAS_TANH) v += g.bias[n];
        if constexpr (EPI == EPI_BIAS_TANH) v = tanhf(v);
        if constexpr (EPI == EPI_DTANH) {
            const float p = g.P[m * g.ldc + n];
            v *= 1.f - p * p;
        }
        C[m * g.ldc + n] = v;
    }
}

// out[i] = sum_z part[z*n + i] in z order (second pass of a split-K product)
__global__ __launch_bounds__(GT) void k_sum_splits(int64_t n, int nz, const float *__restrict__ part,
                                                  float *__restrict__ out) {
    const int64_t i = (int64_t)blockIdx.x * GT + threadIdx.x;
    if (i >= n) return;
    float s = 0.f;
    for (int z = 0; z < nz; z++) s += part[(int64_t)z * n + i];
    out[i] = s;
}

// column sums of X [rows x cols] (bias gradients): one block per column, fixed-order tree
__global__ __launch_bounds__(GT) void k_colsum(int64_t rows, int64_t cols, const float *__restrict__ X,
                                              float *__restrict__ out) {
    __shared__ float s[GT];
    const int64_t c = blockIdx.x;
    float a = 0.f;
    for (int64_t r = threadIdx.x; r < rows; r += GT) a += X[r * cols + c];
    s[threadIdx.x] = a;
    __syncthreads();
    for (int w = GT / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) s[threadIdx.x] += s[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[c] = s[0];
}

// counter-based hash (splitmix64 finaliser) for the batch sample indices
__device__ __forceinline__ uint64_t mix64(uint64_t z) {
    z += 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

// sample of batch row i at a step (all samples in order when the batch covers the data set)
__device__ __forceinline__ int64_t batch_sample(int64_t B, int64_t n, uint64_t seed, int64_t step, int64_t i) {
    return B >= n ? i : (int64_t)(mix64(seed ^ mix64((uint64_t)step * 0x100000001B3ull + i)) % (uint64_t)n);
}

// gradient of the loss by one normalised output y (target t); d: the de-normalised difference
__device__ __forceinline__ float loss_grad(float y, float t, float shift, float scale, float inv, float &d) {
    d = y * scale + shift - t;
    return 2.f * d * scale * inv;
}

// one parameter's Adam step (Kingma & Ba); c1, c2 = 1 - b^t as floats
__device__ __forceinline__ float adam_param(float p, float g, float &m, float &v, float c1, float c2, float lr, float b1,
                                            float b2, float eps) {
    m = b1 * m + (1.f - b1) * g;
    v = b2 * v + (1.f - b2) * g * g;
    const float mh = m / c1, vh = v / c2;
    return p - lr * mh / (sqrtf(vh) + eps);
}

// batch rows: normalised features and targets of sample batch_sample(step, i)
__global__ __launch_bounds__(GT) void k_gather(int64_t B, int64_t n, int n_in, int n_out, const float *__restrict__ X,
                                              const float *__restrict__ T, const float *__restrict__ in_shift,
                                              const float *__restrict__ in_scale, const int64_t *__restrict__ step,
                                              uint64_t seed, float *__restrict__ Xb, float *__restrict__ Tb) {
    const int64_t i = (int64_t)blockIdx.x * GT + threadIdx.x;
    if (i >= B) return;
    const int64_t idx = batch_sample(B, n, seed, step[0], i);
    for (int k = 0; k < n_in; k++) Xb[i * n_in + k] = (X[idx * n_in + k] - in_shift[k]) * in_scale[k];
    for (int k = 0; k < n_out; k++) Tb[i * n_out + k] = T[idx * n_out + k];
}

// dY = 2 (Y*out_scale + out_shift - T) * out_scale / (B n_out), sq = (Y' - T)^2 per element
__global__ __launch_bounds__(GT) void k_loss_grad(int64_t n, int n_out, const float *__restrict__ Y,
                                                 const float *__restrict__ T, const float *__restrict__ out_shift,
                                                 const float *__restrict__ out_scale, float inv, float *__restrict__ dY,
                                                 float *__restrict__ sq) {
    const int64_t i = (int64_t)blockIdx.x * GT + threadIdx.x;
    if (i >= n) return;
    const int k = (int)(i % n_out);
    float d;
    dY[i] = loss_grad(Y[i], T[i], out_shift[k], out_scale[k], inv, d);
    if (sq) sq[i] = d * d;
}

// Adam: the step number comes from the device counter
__global__ __launch_bounds__(GT) void k_adam(int64_t n, float *__restrict__ p, const float *__restrict__ g,
                                            float *__restrict__ m, float *__restrict__ v, int64_t *__restrict__ step,
                                            float lr, float b1, float b2, float eps) {
    const int64_t i = (int64_t)blockIdx.x * GT + threadIdx.x;
    const double t = (double)(step[0] + 1);
    if (i < n) {
        float mi = m[i], vi = v[i];
        p[i] = adam_param(p[i], g[i], mi, vi, (float)(1.0 - pow((double)b1, t)), (float)(1.0 - pow((double)b2, t)), lr, b1,
                          b2, eps);
        m[i] = mi;
        v[i] = vi;
    }
}

__global__ void k_step_advance(int64_t *step) {
    if (blockIdx.x == 0 && threadIdx.x == 0) step[0] += 1;
}

// de-normalised outputs
__global__ __launch_bounds__(GT) void k_denorm(int64_t n, int n_out, const float *__restrict__ Y,
                                              const float *__restrict__ shift, const float *__restrict__ scale,
                                              float *__restrict__ out) {
    const int64_t i = (int64_t)blockIdx.x * GT + threadIdx.x;
    if (i >= n) return;
    const int k = (int)(i % n_out);
    out[i] = Y[i] * scale[k] + shift[k];
}

__global__ __launch_bounds__(GT) void k_normalise(int64_t n, int n_in, const float *__restrict__ X,
                                                 const float *__restrict__ shift, const float *__restrict__ scale,
                                                 float *__restrict__ out) {
    const int64_t i = (int64_t)blockIdx.x * GT + threadIdx.x;
    if (i >= n) return;
    const int k = (int)(i % n_in);
    out[i] = (X[i] - shift[k]) * scale[k];
}

// ------------------------------------------------------------------------------------ whole-network kernels
// v where the mask is all ones, 0 where it is zero (a select that stays a select)
__device__ __forceinline__ float keep(float v, unsigned mask) { return __uint_as_float(__float_as_uint(v) & mask); }

// Networks whose width and n_out fit one block's columns (NET_W, NET_OUT) run a training step in three
// launches and a forward pass in one, in place of one launch per layer and operation (28 for 4 x 128):
//   k_net     a block takes 32 MT rows through every layer; a wave owns 32 columns of each layer.  TRAIN: it
//             draws its batch rows, stores every layer's activations, forms the loss gradient and takes
//             the rows back through the layers, storing each layer's dZ.
//   k_wgrad   every layer's weight-gradient products (64 x 64 tiles, split over the rows as k_gemm's grid.z
//             is) and, in further blocks of the same grid, the partial column sums of the bias gradients
//   k_adam_net  sums the splits, steps Adam and repacks the weights
// What bounds them: v_mfma_f32_32x32x2_f32 takes 64 cycles of a SIMD, and most of the VALU's time (tanh) adds to it.
// One matrix and 16 vector FP32 instructions, 27 and 28 ns each alone: 60 ns together in the only wave of a SIMD, 62 in
// two waves with one kind each, 42 per wave where two or four waves have both; k_net has one wave per SIMD in training
// (256 blocks of 32 rows) and two in inference.  So the operands
// come in the order in which lanes consume them: weights from packed copies in matrix-fragment order (one
// coalesced 16-byte load per lane feeds four instructions; the next layer's loads are issued before this
// layer's products), activations from LDS in the same order.  (A branch-free tanh of 28 instructions was no
// faster than tanhf: 0.43 against 0.41 ms for 300,000 rows.)
// 4 x 128, batch 8192: 67 us per step (k_net 36, k_wgrad 23, k_adam_net 6) against 480 us launch by launch;
// 300,000 rows forward: 0.41 ms (half of it matrix instructions) against 1.25 ms.
// Every sum runs in k_gemm's, k_sum_splits' and k_colsum's order (k ascending in pairs; splits ascending), so
// both forms give the same bits: the launch-per-layer form stays for wider networks and for per-class timing.
constexpr int NET_W = 128, NET_OUT = 32, NET_IN = 64, NET_L = 17, NET_J = NET_W / 8;

struct NetArgs {
    int L, n_in, width, n_out;
    int64_t rows;
    const float *p;                  // parameters (biases are read from here)
    const float *pack;               // packed weights
    int64_t boff[NET_L];             // bias offsets in p
    int fo[NET_L], bo[NET_L];        // packed weights of layer l, forward and (l >= 1) backward, in float4s
    const float *X;                  // rows (TRAIN: the training set)
    const float *in_shift, *in_scale, *out_shift, *out_scale;
    float *Y;                        // out: de-normalised outputs (not TRAIN)
    // TRAIN
    const float *T;
    int64_t n_data;
    const int64_t *step;             // null: rows in order
    uint64_t seed;
    float inv;
    float *H[NET_L], *D[NET_L + 1];  // H[l]: input of layer l; D[l]: dZ of layer l - 1
    float *sq;
};

// groups of 8 values of k: of the inputs and outputs, and of a hidden layer (whole 32-column slices, the
// columns past its width zero, so that the products' loops have constant lengths)
__host__ __device__ inline int net_k8(int k) { return (k + 7) >> 3; }
__host__ __device__ inline int net_kw(int width) { return 4 * ((width + 31) >> 5); }

// LDS position of activation (row m, column k): lane (m, k & 1) of the products reads k = 8 j + 2 q + (k & 1),
// q = 0..3, as one float4.  S: floats per (j, k & 1) group, 4 more than its rows hold, so that the 32
// columns a wave writes for one row fall into 32 banks.
__device__ __forceinline__ int net_at(int k, int m, int S) { return (((k >> 3) << 1) | (k & 1)) * S + m * 4 + ((k >> 1) & 3); }

// the wave's weights of one layer, k8 <= KMAX groups (FIXED: KMAX of them)
template <int KMAX, bool FIXED>
__device__ __forceinline__ void net_weights(const float *pack, int off, int slice, int k8, float4 (&w)[NET_J]) {
    const float4 *b = reinterpret_cast<const float4 *>(pack) + off + (int64_t)slice * k8 * 64 + (threadIdx.x & 63);
#pragma unroll
    for (int j = 0; j < KMAX; j++)
        if (FIXED || j < k8) w[j] = b[j * 64];
}

// acc[t] = A(rows of tile t0 + t, :) B(:, the wave's 32 columns), k ascending; k8 <= KMAX.  FIXED (k8 = KMAX, a
// multiple of 4): the activations of the next four groups are read during the products of these four.
// beside(j) runs after group j's products are issued: other work between them.
template <int MT, int NT, int KMAX, bool FIXED, typename F>
__device__ __forceinline__ void net_mm(const float *lds, int t0, int k8, const float4 (&w)[NET_J], floatx16 (&acc)[NT],
                                       F beside) {
    constexpr int S = MT * 128 + 4, P = FIXED ? 4 : 1;
    const int lane = threadIdx.x & 63;
    const float *at = &lds[(lane >> 5) * S + (t0 * 32 + (lane & 31)) * 4];
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[t][r] = 0.f;
    float4 a[2][P][NT];
    auto read = [&](int j, float4 (&x)[P][NT]) {
#pragma unroll
        for (int q = 0; q < P; q++)
#pragma unroll
            for (int t = 0; t < NT; t++) x[q][t] = *reinterpret_cast<const float4 *>(&at[2 * (j + q) * S + t * 128]);
    };
    read(0, a[0]);
#pragma unroll
    for (int j = 0; j < KMAX; j += P) {
        if (FIXED || j < k8) {
            if (j + P < KMAX) read(j + P, a[((j / P) + 1) & 1]);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int q = 0; q < P; q++) {
                const float4(&x)[NT] = a[(j / P) & 1][q];
#pragma unroll
                for (int t = 0; t < NT; t++) acc[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(x[t].x, w[j + q].x, acc[t], 0, 0, 0);
#pragma unroll
                for (int t = 0; t < NT; t++) acc[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(x[t].y, w[j + q].y, acc[t], 0, 0, 0);
#pragma unroll
                for (int t = 0; t < NT; t++) acc[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(x[t].z, w[j + q].z, acc[t], 0, 0, 0);
#pragma unroll
                for (int t = 0; t < NT; t++) acc[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(x[t].w, w[j + q].w, acc[t], 0, 0, 0);
                beside(j + q);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
}

// KW: net_kw(width).  Hidden activations and their gradients are stored with rows of 8 KW floats (zero past
// the width) in buffers of whole tiles, so no store is guarded.  A block's output layer (at most 32
// columns) is one wave's work per row tile; the waves take turns over the blocks, since blocks that share a
// CU would otherwise load one SIMD.
template <int MT, int KW, bool TRAIN>
__global__ __launch_bounds__(GT, 2) void k_net(const NetArgs a) {
    constexpr int S = MT * 128 + 4, R = 32 * MT, LD = 8 * KW;
    __shared__ __align__(16) float buf[2][2 * NET_J * S];
    __shared__ int64_t sample[R];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, n = wv * 32 + (lane & 31), h = lane >> 5;
    const int64_t r0 = (int64_t)blockIdx.x * R;
    const int W = a.width, kin = net_k8(a.n_in), kout = net_k8(a.n_out);
    const bool mine = wv * 8 < 2 * KW;  // the wave has columns in the hidden layers
    const unsigned in_w = n < W ? ~0u : 0u;
    const unsigned lo = 4 * h * LD + n;  // the lane's part of an element's place in a [row][LD] array
    float4 w[NET_J] = {}, wn[NET_J] = {};
    if (mine) net_weights<NET_IN / 8, false>(a.pack, a.fo[0], wv, kin, w);
    if (tid < R) {  // rows past the last one take a row that is there
        const int64_t row = r0 + tid < a.rows ? r0 + tid : a.rows - 1;
        sample[tid] = TRAIN && a.step ? batch_sample(a.rows, a.n_data, a.seed, a.step[0], row) : row;
    }
    __syncthreads();
    for (int e = tid; e < R * kin * 8; e += GT) {  // inputs, zero beyond n_in
        const int m = e / (kin * 8), k = e % (kin * 8);
        float v = 0.f;
        if (k < a.n_in) {
            v = (a.X[sample[m] * a.n_in + k] - a.in_shift[k]) * a.in_scale[k];
            if constexpr (TRAIN) a.H[0][(r0 + m) * a.n_in + k] = v;
        }
        buf[0][net_at(k, m, S)] = v;
    }
    __syncthreads();
    int cur = 0;
    auto nothing = [](int) {};
    floatx16 acc[MT];
    // row m of the block held by register r of tile t in this lane: row_of(t, r) + 4 h
    auto row_of = [](int t, int r) { return t * 32 + 8 * (r >> 2) + (r & 3); };
    const int ot = (wv - (int)blockIdx.x * MT) & 3;  // the output layer's row tile of this wave (if < MT)
    for (int l = 0; l + 1 < a.L; l++) {
        const bool last = l + 2 == a.L;
        if (last ? ot < MT : mine) net_weights<KW, true>(a.pack, a.fo[l + 1], last ? 0 : wv, KW, wn);
        if (mine) {
            const float b = keep(a.p[a.boff[l] + (n < W ? n : 0)], in_w);
            auto finish = [&](int t, int r) {
                acc[t][r] = keep(tanhf(acc[t][r] + b), in_w);
                buf[cur ^ 1][net_at(n, row_of(t, r) + 4 * h, S)] = acc[t][r];
            };
            if (l == 0) {
                net_mm<MT, MT, NET_IN / 8, false>(buf[cur], 0, kin, w, acc, nothing);
            } else {
                // the tiles after each other, the tanh of one between the products of the next: one tile's
                // accumulators at a time, 108 registers against 128.  300,000 rows of 4 x 128: 407 us against 421
                // with all products first; warm starts by networks of 2 x 16 to 8 x 128: 1 to 4 % shorter.
#pragma unroll
                for (int t = 0; t < MT; t++) {
                    floatx16 one[1];
                    net_mm<MT, 1, KW, true>(buf[cur], t, KW, w, one, [&](int j) {
                        if (t == 0) return;
#pragma unroll
                        for (int r = 16 * j / KW; r < 16 * (j + 1) / KW; r++) finish(t - 1, r);
                    });
                    acc[t] = one[0];
                }
            }
#pragma unroll
            for (int t = 0; t < MT; t++)
                if (l == 0 || t == MT - 1)
#pragma unroll
                    for (int r = 0; r < 16; r++) finish(t, r);
            if constexpr (TRAIN) {
                float *Hl = a.H[l + 1] + r0 * LD;
#pragma unroll
                for (int t = 0; t < MT; t++)
#pragma unroll
                    for (int r = 0; r < 16; r++) (Hl + row_of(t, r) * LD)[lo] = acc[t][r];
            }
        }
        __syncthreads();
        cur ^= 1;
#pragma unroll
        for (int j = 0; j < NET_J; j++) w[j] = wn[j];
    }
    if constexpr (TRAIN)
        if (mine) net_weights<NET_OUT / 8, false>(a.pack, a.bo[a.L - 1], wv, kout, wn);
    if (ot < MT) {
        floatx16 oc[1];
        const int no = lane & 31, ns = no < a.n_out ? no : 0;
        const unsigned in_o = no < a.n_out ? ~0u : 0u;
        float t[TRAIN ? 16 : 1];
        if constexpr (TRAIN)
#pragma unroll
            for (int r = 0; r < 16; r++) t[r] = a.T[sample[row_of(ot, r) + 4 * h] * a.n_out + ns];
        const float b = a.p[a.boff[a.L - 1] + ns], sc = a.out_scale[ns], sh = a.out_shift[ns];
        net_mm<MT, 1, KW, true>(buf[cur], ot, KW, w, oc, nothing);
        if constexpr (TRAIN) {
            float d[16];
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int m = row_of(ot, r) + 4 * h;
                const float g = loss_grad(oc[0][r] + b, t[r], sh, sc, a.inv, d[r]);
                oc[0][r] = r0 + m < a.rows ? keep(g, in_o) : 0.f;
                if (no < kout * 8) buf[cur ^ 1][net_at(no, m, S)] = oc[0][r];
            }
            if (no < a.n_out) {
                const int64_t at = (r0 + 4 * h) * a.n_out + no;
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    a.D[a.L][at + row_of(ot, r) * a.n_out] = oc[0][r];
                    a.sq[at + row_of(ot, r) * a.n_out] = d[r] * d[r];
                }
            }
        } else if (no < a.n_out) {
            const int64_t at = (r0 + 4 * h) * a.n_out + no;
#pragma unroll
            for (int r = 0; r < 16; r++)
                if (r0 + row_of(ot, r) + 4 * h < a.rows) a.Y[at + row_of(ot, r) * a.n_out] = (oc[0][r] + b) * sc + sh;
        }
    }
    if constexpr (TRAIN) {
        __syncthreads();
        cur ^= 1;
        for (int l = a.L - 1; l >= 1; l--) {  // D[l] = (D[l + 1] W_l) (1 - H[l]^2)
#pragma unroll
            for (int j = 0; j < NET_J; j++) w[j] = wn[j];
            if (mine) {
                floatx16 hp[MT];  // this lane's own stores
                const float *Hl = a.H[l] + r0 * LD;
#pragma unroll
                for (int t = 0; t < MT; t++)
#pragma unroll
                    for (int r = 0; r < 16; r++) hp[t][r] = (Hl + row_of(t, r) * LD)[lo];
                if (l > 1) net_weights<KW, true>(a.pack, a.bo[l - 1], wv, KW, wn);
                if (l == a.L - 1)
                    net_mm<MT, MT, NET_OUT / 8, false>(buf[cur], 0, kout, w, acc, nothing);
                else
                    net_mm<MT, MT, KW, true>(buf[cur], 0, KW, w, acc, nothing);
                float *Dl = a.D[l] + r0 * LD;
#pragma unroll
                for (int t = 0; t < MT; t++)
#pragma unroll
                    for (int r = 0; r < 16; r++) {
                        float v = acc[t][r];
                        v *= 1.f - hp[t][r] * hp[t][r];
                        acc[t][r] = keep(v, in_w);
                        buf[cur ^ 1][net_at(n, row_of(t, r) + 4 * h, S)] = acc[t][r];
                    }
#pragma unroll
                for (int t = 0; t < MT; t++)
#pragma unroll
                    for (int r = 0; r < 16; r++) (Dl + row_of(t, r) * LD)[lo] = acc[t][r];
            }
            __syncthreads();
            cur ^= 1;
        }
    }
}

// LDS asked for (and not used) by a k_wgrad block: at most two blocks per CU, so that equal blocks spread evenly over the
// CUs.  Microseconds per training step, up to four on a CU / two: 4 x 128 53.4 / 53.2 (4,096 rows), 66.0 / 63.6 (8,192),
// 108.6 / 99.6 (16,384), 368 / 347 (65,536); 8 x 128 92.4 / 91.2, 124.9 / 113.5, 203 / 181, 725 / 673; 3 x 96 51.0 /
// 50.8 (8,192), 226 / 218 (65,536); 16 to 64 columns, and below 4,096 rows, the same within 1 %.
constexpr int WGRAD_LDS = 56000;

struct WgradArgs {
    int L;
    int64_t rows, kchunk;
    int nz;
    const float *dZ[NET_L], *H[NET_L];  // [row][ldm], [row][ldn]
    int M[NET_L], N[NET_L], ldm[NET_L], ldn[NET_L];
    int64_t so[NET_L];           // the layer's splits in `split` (nz x M x N)
    int first[NET_L + 1];        // first block of each layer's products
    int64_t co[NET_L];           // the layer's partial column sums in `split` (256 x ldm)
    int cfirst[NET_L + 1];       // first block of each layer's column sums
    float *split;
    int64_t *step;               // advanced here (nothing of this launch reads it); null: not a training step
};

// Column sums in k_colsum's order (the rows t, t + 256, ... for each t < 256, then a tree over t), first part:
// the sums of CS consecutive t, whose rows lie together in memory, into part[t][ld].
constexpr int CS = 16;
__device__ __forceinline__ void wgrad_colsum(const float *__restrict__ X, int64_t rows, int ld, int t0, float *part) {
    if ((ld & 3) == 0) {
        for (int e = threadIdx.x; e < CS * (ld >> 2); e += GT) {
            const int t = t0 + e / (ld >> 2), c = 4 * (e % (ld >> 2));
            float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll 16
            for (int64_t r = t; r < rows; r += GT) {
                const float4 x = *reinterpret_cast<const float4 *>(&X[r * ld + c]);
                v.x += x.x;
                v.y += x.y;
                v.z += x.z;
                v.w += x.w;
            }
            *reinterpret_cast<float4 *>(&part[t * ld + c]) = v;
        }
    } else {
        for (int e = threadIdx.x; e < CS * ld; e += GT) {
            const int t = t0 + e / ld, c = e % ld;
            float v = 0.f;
            for (int64_t r = t; r < rows; r += GT) v += X[r * ld + c];
            part[t * ld + c] = v;
        }
    }
}

__global__ __launch_bounds__(GT) void k_wgrad(const WgradArgs a) {
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    if (blockIdx.x == 0 && tid == 0 && a.step) a.step[0] += 1;
    int b = blockIdx.x, l = 0;
    if (b < a.cfirst[a.L]) {
        while (b >= a.cfirst[l + 1]) l++;
        wgrad_colsum(a.dZ[l], a.rows, a.ldm[l], CS * (b - a.cfirst[l]), a.split + a.co[l]);
        return;
    }
    while (b >= a.first[l + 1]) l++;
    b -= a.first[l];
    const int M = a.M[l], N = a.N[l], nt = (N + 63) / 64, mt = (M + 63) / 64;
    const int tn = b % nt, tm = (b / nt) % mt, z = b / (nt * mt);
    const int m0 = tm * 64 + (wv >> 1) * 32, n0 = tn * 64 + (wv & 1) * 32;
    if (m0 >= M || n0 >= N) return;
    const int64_t k0 = (int64_t)z * a.kchunk, k1 = k0 + a.kchunk < a.rows ? k0 + a.kchunk : a.rows;
    // A(m, k) = dZ[k][m], B(k, n) = H[k][n]; lanes past M or N read the last column (their results are
    // not stored).  Groups of 2 U rows, the next group's loads in flight during this group's products;
    // the row's part of an address is the same for all lanes, the lane's part constant.
    constexpr int U = 8;
    const int h = lane >> 5, lm = a.ldm[l], ln = a.ldn[l];
    const int mc = m0 + (lane & 31) < M ? m0 + (lane & 31) : M - 1, nc = n0 + (lane & 31) < N ? n0 + (lane & 31) : N - 1;
    const unsigned oa = h * lm + mc, ob = h * ln + nc;
    const float *pa = a.dZ[l] + k0 * lm, *pb = a.H[l] + k0 * ln;
    floatx16 acc;
#pragma unroll
    for (int r = 0; r < 16; r++) acc[r] = 0.f;
    // (the operands come from memory that the previous kernel wrote: about 2 us away, four groups of products)
    constexpr int NB = 5;
    float av[NB][U], bv[NB][U];
    const int groups = (int)((k1 - k0) / (2 * U)), rest = (int)((k1 - k0) % (2 * U));
    auto fetch = [&](int g, float (&x)[U], float (&y)[U]) {
#pragma unroll
        for (int u = 0; u < U; u++) {
            x[u] = (pa + (int64_t)(g * 2 * U + 2 * u) * lm)[oa];
            y[u] = (pb + (int64_t)(g * 2 * U + 2 * u) * ln)[ob];
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    auto products = [&](const float (&x)[U], const float (&y)[U]) {
#pragma unroll
        for (int u = 0; u < U; u++) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(x[u], y[u], acc, 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
    };
#pragma unroll
    for (int q = 0; q < NB - 1; q++)
        if (q < groups) fetch(q, av[q], bv[q]);
    for (int g = 0; g < groups; g += NB) {
#pragma unroll
        for (int q = 0; q < NB; q++) {
            if (g + q + NB - 1 < groups) fetch(g + q + NB - 1, av[(q + NB - 1) % NB], bv[(q + NB - 1) % NB]);
            if (g + q < groups) products(av[q], bv[q]);
        }
    }
    if (rest > 0) {  // rows past the last one read it and count as zero
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int k = groups * 2 * U + 2 * u, q = 2 * u + h < rest ? k : (int)(k1 - k0) - 1 - h;
            const unsigned in = 2 * u + h < rest ? ~0u : 0u;
            av[0][u] = keep(pa[(int64_t)q * lm + oa], in);
            bv[0][u] = keep(pb[(int64_t)q * ln + ob], in);
        }
        products(av[0], bv[0]);
    }
    float *C = a.split + a.so[l] + (int64_t)z * M * N;
    const int n = n0 + (lane & 31);
    if (n >= N) return;
#pragma unroll
    for (int r = 0; r < 16; r++) {
        const int m = m0 + 8 * (r >> 2) + 4 * h + (r & 3);
        if (m < M) C[(int64_t)m * N + n] = acc[r];
    }
}

// Layout of the packed weights: layer l forward, B(k, n) = W[n][k]; backward (l >= 1), B(k, n) = W[k][n].
// Per 32-column slice and 8-value group of k: lane (n & 31) + 32 (k & 1) holds k = 8 j + 2 q + (k & 1) as a float4.
struct PackArgs {
    int L;
    int64_t np;
    int64_t woff[NET_L], boff[NET_L];
    int din[NET_L], dout[NET_L], fo[NET_L], bo[NET_L];
    int kf[NET_L], kb[NET_L];  // groups of k of the forward and backward copies
    float *pack;
};

__device__ __forceinline__ int64_t net_packed(int off, int k8, int k, int n) {
    return 4 * ((int64_t)off + ((n >> 5) * k8 + (k >> 3)) * 64 + (k & 1) * 32 + (n & 31)) + ((k >> 1) & 3);
}

__device__ __forceinline__ int net_layer(const PackArgs &a, int64_t i) {
    int l = 0;
    while (l + 1 < a.L && i >= a.woff[l + 1]) l++;
    return l;
}

__device__ __forceinline__ void net_pack(const PackArgs &a, int l, int64_t w, float v) {  // weight w of layer l
    const int o = (int)(w / a.din[l]), i = (int)(w % a.din[l]);
    a.pack[net_packed(a.fo[l], a.kf[l], i, o)] = v;
    if (l >= 1) a.pack[net_packed(a.bo[l], a.kb[l], o, i)] = v;
}

__global__ __launch_bounds__(GT) void k_pack(const PackArgs a, const float *__restrict__ p) {
    const int64_t i = (int64_t)blockIdx.x * GT + threadIdx.x;
    if (i >= a.np) return;
    const int l = net_layer(a, i);
    if (i < a.boff[l]) net_pack(a, l, i - a.woff[l], p[i]);
}

// Sum of the splits of each weight gradient in order, and (the blocks from wblocks on, a wave per bias) the tree over
// the partial column sums; ADAM: the parameter's step (t = the advanced step counter) and its packed copies,
// else the gradient into g.
struct AdamArgs {
    PackArgs k;
    const float *split;
    int nz, wblocks;
    int64_t co;   // partial column sums of the first layer in split; the others follow
    int ldm[NET_L];
    float *p, *g, *m, *v;
    const int64_t *step;
    float lr, b1, b2, eps;
};

template <bool ADAM>
__global__ __launch_bounds__(GT) void k_adam_net(const AdamArgs a) {
    __shared__ float c[2];
    if constexpr (ADAM) {
        if (threadIdx.x < 2) c[threadIdx.x] = (float)(1.0 - pow((double)(threadIdx.x ? a.b2 : a.b1), (double)a.step[0]));
        __syncthreads();
    }
    int l;
    int64_t i;
    float s = 0.f;
    const bool weight = (int)blockIdx.x < a.wblocks;
    if (weight) {
        i = (int64_t)blockIdx.x * GT + threadIdx.x;
        if (i >= a.k.np) return;
        l = net_layer(a.k, i);
        if (i >= a.k.boff[l]) return;
        const int64_t nw = (int64_t)a.k.din[l] * a.k.dout[l];
        int64_t so = 0;
        for (int q = 0; q < l; q++) so += (int64_t)a.nz * a.k.din[q] * a.k.dout[q];
        const float *q = a.split + so + (i - a.k.woff[l]);
        int z = 0;
        for (; z + 16 <= a.nz; z += 16) {
            float x[16];
#pragma unroll
            for (int u = 0; u < 16; u++) x[u] = q[(int64_t)(z + u) * nw];
#pragma unroll
            for (int u = 0; u < 16; u++) s += x[u];
        }
        for (; z < a.nz; z++) s += q[(int64_t)z * nw];
    } else {
        int b = ((int)blockIdx.x - a.wblocks) * (GT / 64) + (threadIdx.x >> 6);  // the wave's bias
        int64_t co = a.co;
        for (l = 0; l < a.k.L && b >= a.k.dout[l]; l++) {
            b -= a.k.dout[l];
            co += (int64_t)GT * a.ldm[l];
        }
        if (l >= a.k.L) return;
        const int lane = threadIdx.x & 63, ld = a.ldm[l];
        const float *q = a.split + co + b + (int64_t)lane * ld;
        const float x0 = q[0], x1 = q[64 * ld], x2 = q[128 * ld], x3 = q[192 * ld];
        s = (x0 + x2) + (x1 + x3);
        for (int w = 32; w > 0; w >>= 1) s += __shfl_down(s, w, 64);
        if (lane) return;
        i = a.k.boff[l] + b;
    }
    if constexpr (ADAM) {
        float mi = a.m[i], vi = a.v[i];
        const float pn = adam_param(a.p[i], s, mi, vi, c[0], c[1], a.lr, a.b1, a.b2, a.eps);
        a.m[i] = mi;
        a.v[i] = vi;
        a.p[i] = pn;
        if (weight) net_pack(a.k, l, i - a.k.woff[l], pn);
    } else {
        a.g[i] = s;
    }
}

inline unsigned nblk(int64_t n) { return (unsigned)((n + GT - 1) / GT); }

}  // namespace

struct mst_mlp {
    int n_in = 0, width = 0, hidden = 0, n_out = 0, L = 0;
    std::vector<int> din, dout;        // per layer
    std::vector<int64_t> woff, boff;   // offsets into the parameter array
    int64_t np = 0;
    hipStream_t stream = nullptr;
    float *p = nullptr, *g = nullptr, *m = nullptr, *v = nullptr;  // params, gradient, Adam moments
    float *scal = nullptr;  // in_shift[n_in], in_scale[n_in], out_shift[n_out], out_scale[n_out]
    int64_t *step = nullptr;
    // training set
    float *X = nullptr, *T = nullptr;
    int64_t n_data = 0;
    uint64_t seed = 0;
    // work buffers for batches of up to cap rows
    int64_t cap = 0;
    std::vector<float *> H;  // H[0] = normalised input, H[l] = activations after layer l-1, H[L] = output
    std::vector<float *> D;  // gradients w.r.t. H[l]
    float *Tb = nullptr, *sq = nullptr, *split = nullptr;
    int64_t split_cap = 0;
    // whole-network kernels: packed weights (offsets in float4s per layer), current while pack_ok
    bool net_ok = false, pack_ok = false;
    float *pack = nullptr;
    int fo[NET_L] = {}, bo[NET_L] = {};
    // graph of one training step
    hipGraphExec_t gexec = nullptr;
    int g_batch = 0;
    float g_lr = 0;
    // per-dispatch timing (mst_mlp_timing_*): start/stop events carried by each launch of a class,
    // and the class's floating-point operations per launch (GEMMs: 2 M N K)
    bool timing = false;
    std::vector<std::pair<hipEvent_t, hipEvent_t>> ev[MST_MLP_K_COUNT];
    std::vector<double> flops[MST_MLP_K_COUNT];
    std::vector<hipEvent_t> pool;
};

namespace {

float *fptr(float *base, int64_t off) { return base + off; }

hipEvent_t take_event(mst_mlp *q) {
    if (!q->pool.empty()) {
        hipEvent_t e = q->pool.back();
        q->pool.pop_back();
        return e;
    }
    hipEvent_t e = nullptr;
    return hipEventCreate(&e) == hipSuccess ? e : nullptr;
}

// one launch on the network's stream; with timing on, the dispatch carries start/stop events of
// class kclass (no marker packets between the kernels)
template <typename K, typename... Args>
int mlp_launch(mst_mlp *q, int kclass, double flop, K kernel, dim3 grid, dim3 block, Args... args) {
    if (q->timing) {
        hipEvent_t e0 = take_event(q), e1 = take_event(q);
        if (!e0 || !e1) return mst::fail(MST_E_HIP, "hipEventCreate failed");
        hipExtLaunchKernelGGL(kernel, grid, block, 0, q->stream, e0, e1, 0, args...);
        HIPCHK(hipGetLastError());
        q->ev[kclass].push_back({e0, e1});
        q->flops[kclass].push_back(flop);
        return MST_OK;
    }
    hipLaunchKernelGGL(kernel, grid, block, 0, q->stream, args...);
    HIPCHK(hipGetLastError());
    return MST_OK;
}

// The captured training step holds raw pointers to the training set (X, T), the split buffer and
// the work buffers, and the row count by value: whatever frees or replaces one of them drops it.
void drop_graph(mst_mlp *q) {
    if (q->gexec) (void)hipGraphExecDestroy(q->gexec);
    q->gexec = nullptr;
}

// Whether a rocprofiler-sdk tool is loaded into this process.  Under rocprofv3 --kernel-trace the
// first capture/instantiate/replay of the training step ended in a host segmentation fault inside
// the HIP runtime, before any kernel ran (cause not found); while a tool is present the training
// steps are launched directly instead (same kernels, same results).
bool profiler_tool_loaded() {
    FILE *f = fopen("/proc/self/maps", "r");
    if (!f) return false;
    char line[4096];
    bool found = false;
    while (!found && fgets(line, sizeof(line), f)) found = strstr(line, "librocprofiler-sdk.so") != nullptr;
    fclose(f);
    return found;
}

void free_work(mst_mlp *q) {
    for (auto *p : q->H)
        if (p) (void)hipFree(p);
    for (auto *p : q->D)
        if (p) (void)hipFree(p);
    q->H.assign(q->L + 1, nullptr);
    q->D.assign(q->L + 1, nullptr);
    if (q->Tb) (void)hipFree(q->Tb);
    if (q->sq) (void)hipFree(q->sq);
    q->Tb = q->sq = nullptr;
    q->cap = 0;
    drop_graph(q);
}

int ensure_work(mst_mlp *q, int64_t rows) {
    if (rows <= q->cap) return MST_OK;
    free_work(q);
    if (q->net_ok) rows = (rows + 31) / 32 * 32;  // k_net stores whole tiles
    for (int l = 0; l <= q->L; l++) {
        const int w = l == 0 ? q->n_in : (l == q->L ? q->n_out : (q->net_ok ? 8 * net_kw(q->width) : q->width));
        HIPCHK(hipMalloc((void **)&q->H[l], sizeof(float) * rows * w));
        HIPCHK(hipMalloc((void **)&q->D[l], sizeof(float) * rows * w));
    }
    HIPCHK(hipMalloc((void **)&q->Tb, sizeof(float) * rows * q->n_out));
    HIPCHK(hipMalloc((void **)&q->sq, sizeof(float) * rows * q->n_out));
    q->cap = rows;
    return MST_OK;
}

// C = A B (+ epilogue); with kchunk < K the K range is split over gridDim.z blocks writing
// C + z*cz (returned in *nz)
template <int EPI>
int gemm(mst_mlp *q, int kclass, GemmArgs a, int64_t kchunk = 0, int *nz = nullptr) {
    a.kchunk = kchunk > 0 ? kchunk : (a.K > 0 ? a.K : 1);
    const int64_t z = (a.K + a.kchunk - 1) / a.kchunk;
    dim3 grid((unsigned)((a.N + TN - 1) / TN), (unsigned)((a.M + TM - 1) / TM), (unsigned)(z > 0 ? z : 1));
    int rc = mlp_launch(q, kclass, 2.0 * (double)a.M * (double)a.N * (double)a.K, k_gemm<EPI>, grid, dim3(GT), a);
    if (rc) return rc;
    if (nz) *nz = (int)(z > 0 ? z : 1);
    return MST_OK;
}

// forward of rows already normalised in H[0]; H[L] = raw (normalised-space) output
int forward(mst_mlp *q, int64_t rows) {
    for (int l = 0; l < q->L; l++) {
        GemmArgs a;
        memset(&a, 0, sizeof(a));
        a.A = q->H[l];
        a.B = q->p + q->woff[l];
        a.C = q->H[l + 1];
        a.M = rows;
        a.N = q->dout[l];
        a.K = q->din[l];
        a.sam = q->din[l];
        a.sak = 1;
        a.sbk = 1;
        a.sbn = q->din[l];
        a.ldc = q->dout[l];
        a.bias = q->p + q->boff[l];
        int rc = l + 1 < q->L ? gemm<EPI_BIAS_TANH>(q, MST_MLP_K_GEMM_FWD, a) : gemm<EPI_BIAS>(q, MST_MLP_K_GEMM_FWD, a);
        if (rc) return rc;
    }
    return MST_OK;
}

// the batch dimension of the weight gradients is split into chunks of >= 256 rows (at most 64)
int64_t split_chunk(int64_t rows) { return std::max<int64_t>(256, ((rows + 63) / 64 + TK - 1) / TK * TK); }
int64_t split_need(const mst_mlp *q, int64_t rows) {
    const int64_t nsplit = (rows + split_chunk(rows) - 1) / split_chunk(rows);
    int64_t all = 0;  // the whole-network form keeps every layer's splits
    for (int l = 0; l < q->L; l++) all += (int64_t)q->din[l] * q->dout[l];
    const int64_t one = nsplit * q->width * std::max(q->width, std::max(q->n_in, q->n_out));
    return q->net_ok ? std::max(one, (nsplit * all + 3) / 4 * 4 + (int64_t)GT * ((q->L - 1) * 8 * net_kw(q->width) + q->n_out)) : one;
}
// (outside graph capture) the split buffer for batches of `rows`
int ensure_split(mst_mlp *q, int64_t rows) {
    const int64_t need = split_need(q, rows);
    if (need <= q->split_cap) return MST_OK;
    drop_graph(q);
    if (q->split) (void)hipFree(q->split);
    q->split = nullptr;
    q->split_cap = 0;
    HIPCHK(hipMalloc((void **)&q->split, sizeof(float) * need));
    q->split_cap = need;
    return MST_OK;
}

// gradient of the mean squared error over rows (targets in Tb) into q->g; per-element squares in sq
int backward(mst_mlp *q, int64_t rows) {
    const int64_t ny = rows * q->n_out;
    int rc0 = mlp_launch(q, MST_MLP_K_OTHER, 0.0, k_loss_grad, dim3(nblk(ny)), dim3(GT), ny, q->n_out,
                         (const float *)q->H[q->L], (const float *)q->Tb, (const float *)(q->scal + 2 * q->n_in),
                         (const float *)(q->scal + 2 * q->n_in + q->n_out), 1.f / (float)ny, q->D[q->L], q->sq);
    if (rc0) return rc0;
    const int64_t kchunk = split_chunk(rows);
    if (split_need(q, rows) > q->split_cap) return mst::fail(MST_E_ARG, "mlp: split buffer too small");
    for (int l = q->L - 1; l >= 0; l--) {
        // D[l+1] holds dZ_l (the output layer is linear; hidden layers got the tanh factor below)
        GemmArgs a;
        memset(&a, 0, sizeof(a));
        a.A = q->D[l + 1];  // dZ^T : A(m,k) = dZ[k*out + m]
        a.B = q->H[l];      // H[l] : B(k,n) = H[k*in + n]
        a.C = q->split;
        a.M = q->dout[l];
        a.N = q->din[l];
        a.K = rows;
        a.sam = 1;
        a.sak = q->dout[l];
        a.sbk = q->din[l];
        a.sbn = 1;
        a.ldc = q->din[l];
        a.cz = (int64_t)q->dout[l] * q->din[l];
        int nz = 1;
        int rc = gemm<EPI_NONE>(q, MST_MLP_K_GEMM_WGRAD, a, kchunk, &nz);
        if (rc) return rc;
        const int64_t nw = (int64_t)q->dout[l] * q->din[l];
        rc = mlp_launch(q, MST_MLP_K_OTHER, 0.0, k_sum_splits, dim3(nblk(nw)), dim3(GT), nw, nz,
                        (const float *)q->split, q->g + q->woff[l]);
        if (rc) return rc;
        rc = mlp_launch(q, MST_MLP_K_OTHER, 0.0, k_colsum, dim3(q->dout[l]), dim3(GT), rows, (int64_t)q->dout[l],
                        (const float *)q->D[l + 1], q->g + q->boff[l]);
        if (rc) return rc;
        if (l == 0) break;
        // dZ_{l-1} = (dZ_l W_l) * (1 - H[l]^2)
        GemmArgs b;
        memset(&b, 0, sizeof(b));
        b.A = q->D[l + 1];
        b.B = q->p + q->woff[l];  // W(k=out, n=in) = W[k*in + n]
        b.C = q->D[l];
        b.M = rows;
        b.N = q->din[l];
        b.K = q->dout[l];
        b.sam = q->dout[l];
        b.sak = 1;
        b.sbk = q->din[l];
        b.sbn = 1;
        b.ldc = q->din[l];
        b.P = q->H[l];
        rc = gemm<EPI_DTANH>(q, MST_MLP_K_GEMM_DGRAD, b);
        if (rc) return rc;
    }
    return MST_OK;
}

// ------------------------------------------------------------------------------------ whole-network launches
// Networks that the whole-network kernels take; per-class timing needs a launch per layer and operation.
bool use_net(const mst_mlp *q) { return q->net_ok && !q->timing; }

PackArgs pack_args(const mst_mlp *q) {
    PackArgs a;
    memset(&a, 0, sizeof(a));
    a.L = q->L;
    a.np = q->np;
    for (int l = 0; l < q->L; l++) {
        a.woff[l] = q->woff[l];
        a.boff[l] = q->boff[l];
        a.din[l] = q->din[l];
        a.dout[l] = q->dout[l];
        a.fo[l] = q->fo[l];
        a.bo[l] = q->bo[l];
        a.kf[l] = l == 0 ? net_k8(q->n_in) : net_kw(q->width);
        a.kb[l] = l + 1 == q->L ? net_k8(q->n_out) : net_kw(q->width);
    }
    a.pack = q->pack;
    return a;
}

int ensure_pack(mst_mlp *q) {
    if (q->pack_ok) return MST_OK;
    hipLaunchKernelGGL(k_pack, dim3(nblk(q->np)), dim3(GT), 0, q->stream, pack_args(q), (const float *)q->p);
    HIPCHK(hipGetLastError());
    q->pack_ok = true;
    return MST_OK;
}

NetArgs net_args(const mst_mlp *q, int64_t rows) {
    NetArgs a;
    memset(&a, 0, sizeof(a));
    a.L = q->L;
    a.n_in = q->n_in;
    a.width = q->width;
    a.n_out = q->n_out;
    a.rows = rows;
    a.p = q->p;
    a.pack = q->pack;
    for (int l = 0; l < q->L; l++) {
        a.boff[l] = q->boff[l];
        a.fo[l] = q->fo[l];
        a.bo[l] = q->bo[l];
    }
    a.in_shift = q->scal;
    a.in_scale = q->scal + q->n_in;
    a.out_shift = q->scal + 2 * q->n_in;
    a.out_scale = q->scal + 2 * q->n_in + q->n_out;
    return a;
}

template <int MT, bool TRAIN>
int launch_net(mst_mlp *q, const NetArgs &a) {
    const dim3 grid((unsigned)((a.rows + 32 * MT - 1) / (32 * MT)));
    switch (net_kw(q->width)) {
        case 4: hipLaunchKernelGGL((k_net<MT, 4, TRAIN>), grid, dim3(GT), 0, q->stream, a); break;
        case 8: hipLaunchKernelGGL((k_net<MT, 8, TRAIN>), grid, dim3(GT), 0, q->stream, a); break;
        case 12: hipLaunchKernelGGL((k_net<MT, 12, TRAIN>), grid, dim3(GT), 0, q->stream, a); break;
        default: hipLaunchKernelGGL((k_net<MT, 16, TRAIN>), grid, dim3(GT), 0, q->stream, a); break;
    }
    HIPCHK(hipGetLastError());
    return MST_OK;
}

// loss gradient of `rows` rows of (X, T) with respect to every weight (split sums) and bias (q->g); step
// set: batch rows drawn from the n_data rows at the device step counter, which is advanced
int net_backward(mst_mlp *q, const float *X, const float *T, int64_t n_data, int64_t rows, int64_t *step, AdamArgs *ad) {
    int rc = ensure_pack(q);
    if (rc) return rc;
    NetArgs a = net_args(q, rows);
    a.X = X;
    a.T = T;
    a.n_data = n_data;
    a.step = step;
    a.seed = q->seed;
    a.inv = 1.f / (float)(rows * q->n_out);
    for (int l = 0; l < q->L; l++) {
        a.H[l] = q->H[l];
        a.D[l + 1] = q->D[l + 1];
    }
    a.sq = q->sq;
    rc = launch_net<1, true>(q, a);
    if (rc) return rc;
    WgradArgs w;
    memset(&w, 0, sizeof(w));
    w.L = q->L;
    w.rows = rows;
    w.kchunk = split_chunk(rows);
    w.nz = (int)((rows + w.kchunk - 1) / w.kchunk);
    w.split = q->split;
    w.step = step;
    int64_t so = 0;
    int blocks = 0;
    for (int l = 0; l < q->L; l++) {  // the longest chains first
        w.cfirst[l] = blocks;
        blocks += GT / CS;
    }
    w.cfirst[q->L] = blocks;
    for (int l = 0; l < q->L; l++) {
        w.dZ[l] = q->D[l + 1];
        w.H[l] = q->H[l];
        w.M[l] = q->dout[l];
        w.N[l] = q->din[l];
        w.ldm[l] = l + 1 == q->L ? q->n_out : 8 * net_kw(q->width);
        w.ldn[l] = l == 0 ? q->n_in : 8 * net_kw(q->width);
        w.so[l] = so;
        so += (int64_t)w.nz * q->din[l] * q->dout[l];
        w.first[l] = blocks;
        blocks += ((q->dout[l] + 63) / 64) * ((q->din[l] + 63) / 64) * w.nz;
    }
    so = (so + 3) / 4 * 4;  // (16-byte stores)
    for (int l = 0; l < q->L; l++) {
        w.co[l] = so;
        so += (int64_t)GT * w.ldm[l];
    }
    w.first[q->L] = blocks;
    if (so > q->split_cap) return mst::fail(MST_E_ARG, "mlp: split buffer too small");
    hipLaunchKernelGGL(k_wgrad, dim3((unsigned)blocks), dim3(GT), WGRAD_LDS, q->stream, w);
    HIPCHK(hipGetLastError());
    memset(ad, 0, sizeof(*ad));
    ad->k = pack_args(q);
    ad->split = q->split;
    ad->nz = w.nz;
    ad->wblocks = (int)nblk(q->np);
    ad->co = w.co[0];
    for (int l = 0; l < q->L; l++) ad->ldm[l] = w.ldm[l];
    ad->p = q->p;
    ad->g = q->g;
    ad->m = q->m;
    ad->v = q->v;
    ad->step = step;
    return MST_OK;
}

// the sums of net_backward, into Adam's step or q->g
template <bool ADAM>
int launch_adam(mst_mlp *q, const AdamArgs &a) {
    const int biases = (q->L - 1) * q->width + q->n_out;
    hipLaunchKernelGGL(k_adam_net<ADAM>, dim3((unsigned)(a.wblocks + (biases + GT / 64 - 1) / (GT / 64))), dim3(GT), 0,
                       q->stream, a);
    HIPCHK(hipGetLastError());
    return MST_OK;
}

int net_train_step(mst_mlp *q, int batch, float lr) {
    AdamArgs a;
    int rc = net_backward(q, q->X, q->T, q->n_data, batch, q->step, &a);
    if (rc) return rc;
    a.lr = lr;
    a.b1 = 0.9f;
    a.b2 = 0.999f;
    a.eps = 1e-8f;
    return launch_adam<true>(q, a);
}

int train_step_enqueue(mst_mlp *q, int batch, float lr) {
    int rc = mlp_launch(q, MST_MLP_K_OTHER, 0.0, k_gather, dim3(nblk(batch)), dim3(GT), (int64_t)batch, q->n_data,
                        q->n_in, q->n_out, (const float *)q->X, (const float *)q->T, (const float *)q->scal,
                        (const float *)(q->scal + q->n_in), (const int64_t *)q->step, q->seed, q->H[0], q->Tb);
    if (!rc) rc = forward(q, batch);
    if (!rc) rc = backward(q, batch);
    if (rc) return rc;
    rc = mlp_launch(q, MST_MLP_K_OTHER, 0.0, k_adam, dim3(nblk(q->np)), dim3(GT), q->np, q->p, (const float *)q->g,
                    q->m, q->v, q->step, lr, 0.9f, 0.999f, 1e-8f);
    if (!rc) rc = mlp_launch(q, MST_MLP_K_OTHER, 0.0, k_step_advance, dim3(1), dim3(64), q->step);
    return rc;
}

double sum_host(const float *dptr, int64_t n) {
    std::vector<float> h(n);
    if (hipMemcpy(h.data(), dptr, sizeof(float) * n, hipMemcpyDeviceToHost) != hipSuccess) return NAN;
    double s = 0;
    for (float x : h) s += x;
    return s;
}

}  // namespace

namespace mst {

// later work of stream `after` waits for the earlier work of `before` (by an event of its own, which nothing keeps)
static int follow(hipStream_t after, hipStream_t before) {
    if (after == before) return MST_OK;
    hipEvent_t ev = nullptr;
    HIPCHK(hipEventCreateWithFlags(&ev, hipEventDisableTiming));
    hipError_t e = hipEventRecord(ev, before);
    if (e == hipSuccess) e = hipStreamWaitEvent(after, ev, 0);
    (void)hipEventDestroy(ev);
    HIPCHK(e);
    return MST_OK;
}

int mlp_forward_device(mst_mlp *q, const float *dX, int64_t rows, float *dY, hipStream_t stream) {
    if (use_net(q)) {
        int rc = ensure_pack(q);
        if (rc) return rc;
        // the network runs on its own stream, between the caller's earlier and later work
        rc = follow(q->stream, stream);
        if (rc) return rc;
        NetArgs a = net_args(q, rows);
        a.X = dX;
        a.Y = dY;
        rc = launch_net<2, false>(q, a);
        if (rc) return rc;
        return follow(stream, q->stream);
    }
    // rows in chunks of at most 1 << 20 through the work buffers
    const int64_t chunk = 1 << 20;
    int rc = ensure_work(q, std::min(rows, chunk));
    if (rc) return rc;
    (void)stream;  // the network runs on its own stream; the caller's stream is synchronised around it
    HIPCHK(hipStreamSynchronize(stream));
    for (int64_t r0 = 0; r0 < rows; r0 += chunk) {
        const int64_t nr = std::min(chunk, rows - r0);
        hipLaunchKernelGGL(k_normalise, dim3(nblk(nr * q->n_in)), dim3(GT), 0, q->stream, nr * q->n_in, q->n_in,
                           dX + r0 * q->n_in, (const float *)q->scal, (const float *)(q->scal + q->n_in), q->H[0]);
        HIPCHK(hipGetLastError());
        rc = forward(q, nr);
        if (rc) return rc;
        hipLaunchKernelGGL(k_denorm, dim3(nblk(nr * q->n_out)), dim3(GT), 0, q->stream, nr * q->n_out, q->n_out,
                           (const float *)q->H[q->L], (const float *)(q->scal + 2 * q->n_in),
                           (const float *)(q->scal + 2 * q->n_in + q->n_out), dY + r0 * q->n_out);
        HIPCHK(hipGetLastError());
    }
    HIPCHK(hipStreamSynchronize(q->stream));
    return MST_OK;
}

int mlp_dims(const mst_mlp *q, int *n_in, int *n_out) {
    *n_in = q->n_in;
    *n_out = q->n_out;
    return MST_OK;
}

}  // namespace mst

extern "C" {

int mst_mlp_create(int n_in, int width, int hidden_layers, int n_out, uint64_t seed, mst_mlp **out) {
    if (!out || n_in < 1 || n_in > 64 || width < 1 || width > 4096 || hidden_layers < 1 || hidden_layers > 16 ||
        n_out < 1 || n_out > 64)
        return mst::fail(MST_E_ARG, "mlp: bad sizes");
    *out = nullptr;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0) return mst::fail(MST_E_HIP, "no HIP device available");
    mst_mlp *q = new (std::nothrow) mst_mlp();
    if (!q) return mst::fail(MST_E_ARG, "out of host memory");
    q->n_in = n_in;
    q->width = width;
    q->hidden = hidden_layers;
    q->n_out = n_out;
    q->L = hidden_layers + 1;
    q->seed = seed;
    int64_t off = 0;
    for (int l = 0; l < q->L; l++) {
        const int di = l == 0 ? n_in : width, dd = l + 1 == q->L ? n_out : width;
        q->din.push_back(di);
        q->dout.push_back(dd);
        q->woff.push_back(off);
        off += (int64_t)di * dd;
        q->boff.push_back(off);
        off += dd;
    }
    q->np = off;
    q->H.assign(q->L + 1, nullptr);
    q->D.assign(q->L + 1, nullptr);
    // Glorot-uniform weights, zero biases, from a seeded mt19937_64
    std::vector<float> p(q->np, 0.f);
    std::mt19937_64 eng(seed);
    for (int l = 0; l < q->L; l++) {
        const double a = std::sqrt(6.0 / (q->din[l] + q->dout[l]));
        for (int64_t i = 0; i < (int64_t)q->din[l] * q->dout[l]; i++)
            p[q->woff[l] + i] = (float)(a * (2.0 * ((eng() >> 11) * (1.0 / 9007199254740992.0)) - 1.0));
    }
    // whole-network kernels: columns of a layer within one block (k_net)
    q->net_ok = width <= NET_W && n_out <= NET_OUT && n_in <= NET_IN && q->L <= NET_L;
    int64_t packed = 0;  // float4s
    for (int l = 0; q->net_ok && l < q->L; l++) {
        q->fo[l] = (int)packed;
        packed += (int64_t)((q->dout[l] + 31) / 32) * (l == 0 ? net_k8(n_in) : net_kw(width)) * 64;
        q->bo[l] = (int)packed;
        if (l >= 1) packed += (int64_t)((q->din[l] + 31) / 32) * (l + 1 == q->L ? net_k8(n_out) : net_kw(width)) * 64;
    }
    std::vector<float> sc(2 * n_in + 2 * n_out, 0.f);
    for (int k = 0; k < n_in; k++) sc[n_in + k] = 1.f;
    for (int k = 0; k < n_out; k++) sc[2 * n_in + n_out + k] = 1.f;
    bool ok = hipStreamCreate(&q->stream) == hipSuccess && hipMalloc((void **)&q->p, sizeof(float) * q->np) == hipSuccess &&
              hipMalloc((void **)&q->g, sizeof(float) * q->np) == hipSuccess &&
              hipMalloc((void **)&q->m, sizeof(float) * q->np) == hipSuccess &&
              hipMalloc((void **)&q->v, sizeof(float) * q->np) == hipSuccess &&
              hipMalloc((void **)&q->scal, sizeof(float) * sc.size()) == hipSuccess &&
              hipMalloc((void **)&q->step, sizeof(int64_t)) == hipSuccess &&
              (!q->net_ok || (hipMalloc((void **)&q->pack, 16 * packed) == hipSuccess &&
                              hipMemset(q->pack, 0, 16 * packed) == hipSuccess)) &&  // the padding stays zero
              hipMemcpy(q->p, p.data(), sizeof(float) * q->np, hipMemcpyHostToDevice) == hipSuccess &&
              hipMemset(q->m, 0, sizeof(float) * q->np) == hipSuccess &&
              hipMemset(q->v, 0, sizeof(float) * q->np) == hipSuccess &&
              hipMemset(q->g, 0, sizeof(float) * q->np) == hipSuccess &&
              hipMemset(q->step, 0, sizeof(int64_t)) == hipSuccess &&
              hipMemcpy(q->scal, sc.data(), sizeof(float) * sc.size(), hipMemcpyHostToDevice) == hipSuccess;
    if (!ok) {
        mst_mlp_destroy(q);
        return mst::fail(MST_E_HIP, "mlp: device allocation failed");
    }
    *out = q;
    return MST_OK;
}

int mst_mlp_destroy(mst_mlp *q) {
    if (!q) return MST_OK;
    if (q->stream) (void)hipStreamSynchronize(q->stream);
    free_work(q);
    for (auto &v : q->ev)
        for (auto &pr : v) {
            (void)hipEventDestroy(pr.first);
            (void)hipEventDestroy(pr.second);
        }
    for (auto e : q->pool) (void)hipEventDestroy(e);
    for (void *b : {(void *)q->p, (void *)q->g, (void *)q->m, (void *)q->v, (void *)q->scal, (void *)q->step,
                    (void *)q->X, (void *)q->T, (void *)q->split, (void *)q->pack})
        if (b) (void)hipFree(b);
    if (q->stream) (void)hipStreamDestroy(q->stream);
    delete q;
    return MST_OK;
}

int mst_mlp_num_params(const mst_mlp *q, int64_t *n) {
    if (!q || !n) return mst::fail(MST_E_ARG, "null argument");
    *n = q->np;
    return MST_OK;
}

int mst_mlp_get_params(mst_mlp *q, float *p, int64_t n) {
    if (!q || !p || n != q->np) return mst::fail(MST_E_ARG, "parameter count mismatch");
    HIPCHK(hipStreamSynchronize(q->stream));
    HIPCHK(hipMemcpy(p, q->p, sizeof(float) * n, hipMemcpyDeviceToHost));
    return MST_OK;
}

int mst_mlp_set_params(mst_mlp *q, const float *p, int64_t n) {
    if (!q || !p || n != q->np) return mst::fail(MST_E_ARG, "parameter count mismatch");
    HIPCHK(hipStreamSynchronize(q->stream));
    q->pack_ok = false;
    HIPCHK(hipMemcpy(q->p, p, sizeof(float) * n, hipMemcpyHostToDevice));
    return MST_OK;
}

int mst_mlp_set_scaling(mst_mlp *q, const float *in_shift, const float *in_scale, const float *out_shift,
                        const float *out_scale) {
    if (!q || !in_shift || !in_scale || !out_shift || !out_scale) return mst::fail(MST_E_ARG, "null argument");
    std::vector<float> sc;
    sc.insert(sc.end(), in_shift, in_shift + q->n_in);
    sc.insert(sc.end(), in_scale, in_scale + q->n_in);
    sc.insert(sc.end(), out_shift, out_shift + q->n_out);
    sc.insert(sc.end(), out_scale, out_scale + q->n_out);
    HIPCHK(hipStreamSynchronize(q->stream));
    HIPCHK(hipMemcpy(q->scal, sc.data(), sizeof(float) * sc.size(), hipMemcpyHostToDevice));
    return MST_OK;
}

int mst_mlp_set_data(mst_mlp *q, const float *X, const float *T, int64_t n) {
    if (!q || !X || !T || n < 1) return mst::fail(MST_E_ARG, "bad training set");
    HIPCHK(hipStreamSynchronize(q->stream));
    drop_graph(q);
    if (q->X) (void)hipFree(q->X);
    if (q->T) (void)hipFree(q->T);
    q->X = q->T = nullptr;
    HIPCHK(hipMalloc((void **)&q->X, sizeof(float) * n * q->n_in));
    HIPCHK(hipMalloc((void **)&q->T, sizeof(float) * n * q->n_out));
    HIPCHK(hipMemcpy(q->X, X, sizeof(float) * n * q->n_in, hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(q->T, T, sizeof(float) * n * q->n_out, hipMemcpyHostToDevice));
    q->n_data = n;
    return MST_OK;
}

int mst_mlp_reset_optimizer(mst_mlp *q) {
    if (!q) return mst::fail(MST_E_ARG, "null argument");
    HIPCHK(hipStreamSynchronize(q->stream));
    HIPCHK(hipMemset(q->m, 0, sizeof(float) * q->np));
    HIPCHK(hipMemset(q->v, 0, sizeof(float) * q->np));
    HIPCHK(hipMemset(q->step, 0, sizeof(int64_t)));
    return MST_OK;
}

int mst_mlp_train(mst_mlp *q, int steps, int batch, double lr, int use_graph, double *loss) {
    if (!q || steps < 0 || batch < 1 || !(lr > 0)) return mst::fail(MST_E_ARG, "bad arguments");
    if (!q->X) return mst::fail(MST_E_ARG, "mlp: no training set");
    if (batch > q->n_data) batch = (int)q->n_data;
    int rc = ensure_work(q, batch);
    if (!rc) rc = ensure_split(q, batch);
    if (rc) return rc;
    const bool net = use_net(q);  // three launches a step: nothing to gain from a graph
    if (!net) q->pack_ok = false;  // the launch-per-layer Adam leaves the packed copies behind
    if (net || (use_graph && (q->timing || profiler_tool_loaded()))) use_graph = 0;  // per-dispatch events need direct launches
    if (use_graph && (!q->gexec || q->g_batch != batch || q->g_lr != (float)lr)) {
        drop_graph(q);
        hipGraph_t g = nullptr;
        HIPCHK(hipStreamBeginCapture(q->stream, hipStreamCaptureModeThreadLocal));
        rc = train_step_enqueue(q, batch, (float)lr);
        hipError_t e = hipStreamEndCapture(q->stream, &g);
        if (rc) {
            if (g) (void)hipGraphDestroy(g);
            return rc;
        }
        if (e != hipSuccess) return mst::fail(MST_E_HIP, std::string("graph capture: ") + hipGetErrorString(e));
        e = hipGraphInstantiate(&q->gexec, g, nullptr, nullptr, 0);
        (void)hipGraphDestroy(g);
        if (e != hipSuccess) return mst::fail(MST_E_HIP, std::string("graph instantiate: ") + hipGetErrorString(e));
        q->g_batch = batch;
        q->g_lr = (float)lr;
    }
    for (int s = 0; s < steps; s++) {
        if (use_graph) {
            HIPCHK(hipGraphLaunch(q->gexec, q->stream));
        } else {
            rc = net ? net_train_step(q, batch, (float)lr) : train_step_enqueue(q, batch, (float)lr);
            if (rc) return rc;
        }
    }
    HIPCHK(hipStreamSynchronize(q->stream));
    if (loss) *loss = steps > 0 ? sum_host(q->sq, (int64_t)batch * q->n_out) / ((double)batch * q->n_out) : NAN;
    return MST_OK;
}

int mst_mlp_forward(mst_mlp *q, const float *X, int64_t n, float *Y) {
    if (!q || !X || !Y || n < 1) return mst::fail(MST_E_ARG, "bad arguments");
    float *dX = nullptr, *dY = nullptr;
    HIPCHK(hipMalloc((void **)&dX, sizeof(float) * n * q->n_in));
    HIPCHK(hipMalloc((void **)&dY, sizeof(float) * n * q->n_out));
    int rc = MST_OK;
    if (hipMemcpy(dX, X, sizeof(float) * n * q->n_in, hipMemcpyHostToDevice) != hipSuccess)
        rc = mst::fail(MST_E_HIP, "copy failed");
    if (!rc) rc = mst::mlp_forward_device(q, dX, n, dY, q->stream);
    if (!rc && hipStreamSynchronize(q->stream) != hipSuccess) rc = mst::fail(MST_E_HIP, "forward pass failed");
    if (!rc && hipMemcpy(Y, dY, sizeof(float) * n * q->n_out, hipMemcpyDeviceToHost) != hipSuccess)
        rc = mst::fail(MST_E_HIP, "copy failed");
    (void)hipFree(dX);
    (void)hipFree(dY);
    return rc;
}

// full-batch gradient of the mean squared error of (X, T) (de-normalised outputs against T)
int mst_mlp_gradient(mst_mlp *q, const float *X, const float *T, int64_t n, float *grad, double *loss) {
    if (!q || !X || !T || n < 1) return mst::fail(MST_E_ARG, "bad arguments");
    int rc = ensure_work(q, n);
    if (!rc) rc = ensure_split(q, n);
    if (rc) return rc;
    float *dX = nullptr;
    HIPCHK(hipMalloc((void **)&dX, sizeof(float) * n * q->n_in));
    if (hipMemcpy(dX, X, sizeof(float) * n * q->n_in, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(q->Tb, T, sizeof(float) * n * q->n_out, hipMemcpyHostToDevice) != hipSuccess) {
        (void)hipFree(dX);
        return mst::fail(MST_E_HIP, "copy failed");
    }
    if (use_net(q)) {
        AdamArgs a;
        rc = net_backward(q, dX, q->Tb, n, n, nullptr, &a);
        if (!rc) rc = launch_adam<false>(q, a);
    } else {
        hipLaunchKernelGGL(k_normalise, dim3(nblk(n * q->n_in)), dim3(GT), 0, q->stream, n * q->n_in, q->n_in,
                           (const float *)dX, (const float *)q->scal, (const float *)(q->scal + q->n_in), q->H[0]);
        rc = forward(q, n);
        if (!rc) rc = backward(q, n);
    }
    hipError_t e = hipStreamSynchronize(q->stream);
    (void)hipFree(dX);
    if (rc) return rc;
    if (e != hipSuccess) return mst::fail(MST_E_HIP, hipGetErrorString(e));
    if (grad) HIPCHK(hipMemcpy(grad, q->g, sizeof(float) * q->np, hipMemcpyDeviceToHost));
    if (loss) *loss = sum_host(q->sq, n * q->n_out) / ((double)n * q->n_out);
    return MST_OK;
}

int mst_mlp_timing_enable(mst_mlp *q, int on) {
    if (!q) return mst::fail(MST_E_ARG, "null argument");
    HIPCHK(hipStreamSynchronize(q->stream));
    q->timing = on != 0;
    return MST_OK;
}

int mst_mlp_timing_get(mst_mlp *q, int kclass, int64_t *count, double *total_ms, double *total_flop) {
    if (!q || kclass < 0 || kclass >= MST_MLP_K_COUNT || !count || !total_ms)
        return mst::fail(MST_E_ARG, "bad kernel class");
    HIPCHK(hipStreamSynchronize(q->stream));
    double tot = 0, fl = 0;
    for (size_t i = 0; i < q->ev[kclass].size(); i++) {
        float ms = 0;
        HIPCHK(hipEventElapsedTime(&ms, q->ev[kclass][i].first, q->ev[kclass][i].second));
        tot += ms;
        fl += q->flops[kclass][i];
    }
    *count = (int64_t)q->ev[kclass].size();
    *total_ms = tot;
    if (total_flop) *total_flop = fl;
    return MST_OK;
}

int mst_mlp_timing_reset(mst_mlp *q) {
    if (!q) return mst::fail(MST_E_ARG, "null argument");
    HIPCHK(hipStreamSynchronize(q->stream));
    for (int k = 0; k < MST_MLP_K_COUNT; k++) {
        for (auto &pr : q->ev[k]) {
            q->pool.push_back(pr.first);
            q->pool.push_back(pr.second);
        }
        q->ev[k].clear();
        q->flops[k].clear();
    }
    return MST_OK;
}

}  // extern "C"
