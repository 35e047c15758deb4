// The selector network: forward, softmax cross-entropy, backward and Adam,
// as hand-written HIP kernels (FP32).  A network whose weights fit one CU's
// LDS (the selector's 24 -> 128 -> 128 -> 22 does) takes two launches per
// step: mlp_pass_kernel, one workgroup per 16 samples from x to its share of
// every gradient, and mlp_update_kernel, which adds the shares and takes the
// Adam step.  Larger networks run layer by layer: an LDS-tiled GEMM kernel
// with transpose flags, bias / activation and reduction kernels.  Every sum
// has a fixed order: training is deterministic for a given seed.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <new>
#include <vector>

#include "clspmv.h"
#include "clspmv_mlp.h"
#include "host/internal.hpp"
#include "runtime.hpp"

using namespace clspmv;

namespace {

constexpr int kT = 16;  // GEMM tile

// C[M x N] = op(A) * op(B) (+ C when accumulate), op(A) is M x K, op(B) K x N.
// A is row-major M x K (lda = K) or, transposed, K x M (lda = M); likewise B.
__global__ __launch_bounds__(kT* kT) void gemm_kernel(int M, int N, int K, const float* __restrict__ A, int ta,
                                                      const float* __restrict__ B, int tb, float* __restrict__ C,
                                                      int accumulate) {
    __shared__ float As[kT][kT + 1];
    __shared__ float Bs[kT][kT + 1];
    const int tx = threadIdx.x % kT, ty = threadIdx.x / kT;
    const int row = blockIdx.y * kT + ty, col = blockIdx.x * kT + tx;
    float acc = 0.f;
    for (int k0 = 0; k0 < K; k0 += kT) {
        const int ka = k0 + tx, kb = k0 + ty;
        float a = 0.f, b = 0.f;
        if (row < M && ka < K) a = ta ? A[(size_t)ka * M + row] : A[(size_t)row * K + ka];
        if (col < N && kb < K) b = tb ? B[(size_t)col * K + kb] : B[(size_t)kb * N + col];
        As[ty][tx] = a;
        Bs[ty][tx] = b;
        __syncthreads();
#pragma unroll
        for (int k = 0; k < kT; ++k) acc += As[ty][k] * Bs[k][tx];
        __syncthreads();
    }
    if (row < M && col < N) {
        float* c = C + (size_t)row * N + col;
        *c = accumulate ? *c + acc : acc;
    }
}

__global__ void bias_act_kernel(float* __restrict__ Z, const float* __restrict__ b, int M, int N, int relu) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= M * N) return;
    float v = Z[i] + b[i % N];
    Z[i] = relu ? fmaxf(v, 0.f) : v;
}

// Per sample: softmax of the logits; dZ = (p - onehot) / n; loss_i.
__global__ void softmax_ce_kernel(const float* __restrict__ Z, const int* __restrict__ y, int n, int c,
                                  float* __restrict__ dZ, float* __restrict__ loss_i) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const float* z = Z + (size_t)i * c;
    float mx = z[0];
    for (int j = 1; j < c; ++j) mx = fmaxf(mx, z[j]);
    float s = 0.f;
    for (int j = 0; j < c; ++j) s += expf(z[j] - mx);
    const int t = y[i];
    for (int j = 0; j < c; ++j) {
        const float p = expf(z[j] - mx) / s;
        dZ[(size_t)i * c + j] = (p - (j == t ? 1.f : 0.f)) / (float)n;
    }
    loss_i[i] = -(z[t] - mx - logf(s));
}

__global__ void relu_back_kernel(float* __restrict__ dH, const float* __restrict__ H, int n) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n && H[i] <= 0.f) dH[i] = 0.f;
}

// out[j] = sum_i A[i][j] (x scale): one workgroup per 64 columns, its 16
// waves' row classes (i mod 16) added in order.  (One thread per column took
// 330 us for 1920 x 128.)
__global__ __launch_bounds__(1024) void colsum_kernel(const float* __restrict__ A, int M, int N, float scale,
                                                      float* __restrict__ out) {
    __shared__ float part[16][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int j = blockIdx.x * 64 + lane;
    float s = 0.f;
    if (j < N)
        for (int i = w; i < M; i += 16) s += A[(size_t)i * N + j];
    part[w][lane] = s;
    __syncthreads();
    if (w || j >= N) return;
    s = 0.f;
#pragma unroll
    for (int k = 0; k < 16; ++k) s += part[k][lane];
    out[j] = s * scale;
}

// ---------------------------------------------------------------- in one CU
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kPassThreads = 512, kPassWaves = kPassThreads / 64;
constexpr int kPassSamples = 16;   // the rows of one 16 x 16 matrix-core tile
constexpr int kPassGroups = 256;   // workgroups at most (one per CU); each takes every kPassGroups-th tile
constexpr int kPassHidden = 16 * kPassWaves;  // one 16-column tile of the hidden layers per wave
constexpr int kPassEnds = 4;       // 16-column tiles of the features and of the classes at most
constexpr int kPassLds = 40960;    // floats: all 160 KiB of a CU

__host__ __device__ constexpr int pad16(int n) { return (n + 15) / 16 * 16; }
// LDS row stride of a matrix of n columns (a multiple of 16).  A tile's
// operand is read as 4 consecutive columns of 16 rows or 16 consecutive
// columns of 4 rows: strides of 4 x odd mod 64 banks keep the first free of
// conflicts, and all of them but 4 and 60 the second to two lanes per bank.
__host__ __device__ constexpr int lds_stride(int n) { return n + (n % 64 ? 4 : 20); }

struct MlpShape {
    int in, hid, cls;
    __host__ __device__ int inp() const { return pad16(in); }
    __host__ __device__ int hp() const { return pad16(hid); }
    __host__ __device__ int cp() const { return pad16(cls); }
    __host__ __device__ int params() const { return in * hid + hid + hid * hid + hid + hid * cls + cls; }
    // LDS offsets (floats): the weights and biases, then a tile's x, hidden
    // activations and logits
    __host__ __device__ int w1() const { return 0; }
    __host__ __device__ int w2() const { return w1() + inp() * lds_stride(hp()); }
    __host__ __device__ int w3() const { return w2() + hp() * lds_stride(hp()); }
    __host__ __device__ int b1() const { return w3() + hp() * lds_stride(cp()); }
    __host__ __device__ int b2() const { return b1() + hp(); }
    __host__ __device__ int b3() const { return b2() + hp(); }
    __host__ __device__ int x() const { return b3() + cp(); }
    __host__ __device__ int h1() const { return x() + kPassSamples * lds_stride(inp()); }
    __host__ __device__ int h2() const { return h1() + kPassSamples * lds_stride(hp()); }
    __host__ __device__ int z() const { return h2() + kPassSamples * lds_stride(hp()); }
    __host__ __device__ int losses() const { return z() + kPassSamples * lds_stride(cp()); }
    __host__ __device__ int floats() const { return losses() + kPassSamples; }
    bool one_cu() const {
        return hid <= kPassHidden && in <= 16 * kPassEnds && cls <= 16 * kPassEnds && floats() <= kPassLds;
    }
};

// Rows wave, wave + 8, ... of a rows x cols matrix at src straight into LDS
// rows of `stride` (no registers, no wait between them: the caller waits
// with lds_loads_done).  The loads of a row are 64 lanes side by side.
__device__ __forceinline__ void load_rows(const float* __restrict__ src, int rows, int cols, float* dst, int stride,
                                          int wave, int lane) {
    for (int r = wave; r < rows; r += kPassWaves)
        for (int c = 0; c < cols; c += 64)
            if (lane < cols - c)
                __builtin_amdgcn_global_load_lds(
                    (const __attribute__((address_space(1))) void*)(src + (size_t)r * cols + c + lane),
                    (__attribute__((address_space(3))) void*)(dst + r * stride + c), 4, 0, 0);
}
__device__ __forceinline__ void lds_loads_done() { __builtin_amdgcn_s_waitcnt(0x0F70); }  // vmcnt(0)

// The reverse, for the gradients.
__device__ __forceinline__ void store_rows(const float* src, int stride, int rows, int cols, float* __restrict__ dst,
                                           int wave, int lane) {
    for (int r = wave; r < rows; r += kPassWaves)
        for (int c = lane; c < cols; c += 64) dst[(size_t)r * cols + c] = src[r * stride + c];
}

// v_mfma_f32_16x16x4f32: lane l gives A[l % 16][l / 16] and B[l / 16][l % 16]
// and holds rows 4 (l / 16) .. + 3 of column l % 16 of the result.
// acc += A B over K (a multiple of 16): A's element (m, k) at a[m * am + k *
// ak], B's (k, n) at b[k * bk + n * bn].
__device__ __forceinline__ f32x4 tile_product(const float* a, int am, int ak, const float* b, int bk, int bn, int K,
                                              int lane, f32x4 acc) {
    const int i = lane & 15, q = lane >> 4;
    a += i * am + q * ak;
    b += q * bk + i * bn;
    float av[4], bv[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        av[u] = a[4 * u * ak];
        bv[u] = b[4 * u * bk];
    }
    for (int k = 16; k < K; k += 16) {  // the next 16 load while these multiply
        float an[4], bn4[4];
        a += 16 * ak;
        b += 16 * bk;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            an[u] = a[4 * u * ak];
            bn4[u] = b[4 * u * bk];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(av[u], bv[u], acc, 0, 0, 0);
            av[u] = an[u];
            bv[u] = bn4[u];
        }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(av[u], bv[u], acc, 0, 0, 0);
    return acc;
}

// N tiles of a weight gradient side by side, acc[t] += A B_t with K = 16
// samples: B_t is B's columns 16 t .. + 15.  Tiles past `tiles` read whatever
// LDS holds there (inside the array) and are never stored: no branch between
// the loads.
template <int N>
__device__ __forceinline__ void tile_outer(const float* a, int ak, const float* b, int bk, int lane, f32x4 (&acc)[N]) {
    const int i = lane & 15, q = lane >> 4;
    float av[4], bv[N][4];
#pragma unroll
    for (int u = 0; u < 4; ++u) av[u] = a[i + (4 * u + q) * ak];
#pragma unroll
    for (int t = 0; t < N; ++t)
#pragma unroll
        for (int u = 0; u < 4; ++u) bv[t][u] = b[16 * t + i + (4 * u + q) * bk];
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int t = 0; t < N; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[u], bv[t][u], acc[t], 0, 0, 0);
}

__device__ __forceinline__ float sum16(float v) {
#pragma unroll
    for (int m = 1; m < 16; m <<= 1) v += __shfl_xor(v, m, 64);
    return v;
}

__device__ __forceinline__ float column_sum(const float* a, int stride) {
    float v[kPassSamples], s = 0.f;
#pragma unroll
    for (int m = 0; m < kPassSamples; ++m) v[m] = a[m * stride];
#pragma unroll
    for (int m = 0; m < kPassSamples; ++m) s += v[m];
    return s;
}

// Forward pass of 16 samples at a time and, TRAIN, loss and backward pass:
// the workgroup's weights stay in LDS, the activations of a tile too, the
// weight gradients of its tiles in the matrix cores' accumulators (wave w
// holds rows 16 w .. of W2's and W3's and columns 16 w .. of W1's).  TRAIN
// writes the workgroup's sums for every parameter and its loss to
// part[group][params + 1], else the logits to zout.
// Bound by what one CU can draw and by the chain of layers: 1920 samples of
// the 24-128-128-22 network are 120 workgroups of 1060 16x16x4 products each
// and take 27 us, of it 7 the 90 KB of weights coming in, 3 forward, 1
// softmax, 5 backward, 5 the 90 KB of gradients going out.  A training step
// is 35-39 us with the update kernel (7 us) against 1340 layer by layer with
// 20 launches (column sums by one thread per column 330 us, 16 x 16 tiles
// on the VALU 30 us each).
template <bool TRAIN>
__global__ __launch_bounds__(kPassThreads) void mlp_pass_kernel(MlpShape s, const float* __restrict__ p,
                                                                const float* __restrict__ x,
                                                                const int* __restrict__ label, int n,
                                                                float* __restrict__ part, float* __restrict__ zout) {
    __shared__ __align__(16) float lds[kPassLds];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 15, row4 = (lane >> 4) * 4;
    const int I = s.in, H = s.hid, C = s.cls, Ip = s.inp(), Hp = s.hp(), Cp = s.cp();
    const int is = lds_stride(Ip), hs = lds_stride(Hp), cs = lds_stride(Cp);
    float *W1 = lds + s.w1(), *W2 = lds + s.w2(), *W3 = lds + s.w3(), *B1 = lds + s.b1(), *B2 = lds + s.b2(),
          *B3 = lds + s.b3(), *X = lds + s.x(), *H1 = lds + s.h1(), *H2 = lds + s.h2(), *Z = lds + s.z();
    const float *g1 = p, *gb1 = g1 + I * H, *g2 = gb1 + H, *gb2 = g2 + H * H, *g3 = gb2 + H, *gb3 = g3 + H * C;
    // padding rows and columns are zero throughout (W2's are there only where
    // hid is no multiple of 16; the activations' are written with the rest)
    for (int i = tid * 4; i < s.h1(); i += kPassThreads * 4)
        if (H != Hp || i < s.w2() || i >= s.w3())
            *reinterpret_cast<float4*>(lds + i) = make_float4(0.f, 0.f, 0.f, 0.f);
    __syncthreads();
    load_rows(g1, I, H, W1, hs, wave, lane);
    load_rows(gb1, 1, H, B1, 0, wave, lane);
    load_rows(g2, H, H, W2, hs, wave, lane);
    load_rows(gb2, 1, H, B2, 0, wave, lane);
    load_rows(g3, H, C, W3, cs, wave, lane);
    load_rows(gb3, 1, C, B3, 0, wave, lane);

    const bool hidden = 16 * wave < Hp;  // this wave has a tile of the hidden layers
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    f32x4 d1[kPassEnds], d2[kPassWaves], d3[kPassEnds];
#pragma unroll
    for (int t = 0; t < kPassEnds; ++t) d1[t] = d3[t] = zero;
#pragma unroll
    for (int t = 0; t < kPassWaves; ++t) d2[t] = zero;
    float db1 = 0.f, db2 = 0.f, db3 = 0.f, loss = 0.f;  // column tid's bias gradients; sample tid / 16's losses

    for (int s0 = blockIdx.x * kPassSamples; s0 < n; s0 += gridDim.x * kPassSamples) {
        const int live = min(kPassSamples, n - s0);
        load_rows(x + (size_t)s0 * I, live, I, X, is, wave, lane);
        for (int m = wave; m < kPassSamples; m += kPassWaves)
            if (m >= live && lane < I) X[m * is + lane] = 0.f;
        int t = -1;  // label of sample tid / 16
        if constexpr (TRAIN)
            if (tid < 16 * kPassSamples && (tid >> 4) < live) t = label[s0 + (tid >> 4)];
        lds_loads_done();
        __syncthreads();
        // hidden layers: column tile `wave` of H1 and H2
        if (hidden) {
            const f32x4 v = tile_product(X, is, 1, W1 + 16 * wave, hs, 1, Ip, lane, zero);
#pragma unroll
            for (int r = 0; r < 4; ++r) H1[(row4 + r) * hs + 16 * wave + col] = fmaxf(v[r] + B1[16 * wave + col], 0.f);
        }
        __syncthreads();
        if (hidden) {
            const f32x4 v = tile_product(H1, hs, 1, W2 + 16 * wave, hs, 1, Hp, lane, zero);
#pragma unroll
            for (int r = 0; r < 4; ++r) H2[(row4 + r) * hs + 16 * wave + col] = fmaxf(v[r] + B2[16 * wave + col], 0.f);
        }
        __syncthreads();
        if (16 * wave < Cp) {
            const f32x4 v = tile_product(H2, hs, 1, W3 + 16 * wave, cs, 1, Hp, lane, zero);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int m = row4 + r, c = 16 * wave + col;
                const float z = v[r] + B3[c];
                if constexpr (TRAIN)
                    Z[m * cs + c] = z;
                else if (c < C && s0 + m < n)
                    zout[(size_t)(s0 + m) * C + c] = z;
            }
        }
        if constexpr (TRAIN) {
            __syncthreads();
            // softmax of the logits, sixteen lanes per sample:
            // dz = (p - onehot) / n, zero past the last sample and class
            if (tid < 16 * kPassSamples) {
                const int m = tid >> 4, j = tid & 15;
                const bool on = s0 + m < n;
                float* zr = Z + m * cs;
                float zv[kPassEnds], mx = zr[0];  // class 0: always there
#pragma unroll
                for (int k = 0; k < kPassEnds; ++k) {
                    zv[k] = 16 * k + j < C ? zr[16 * k + j] : mx;
                    mx = fmaxf(mx, zv[k]);
                }
#pragma unroll
                for (int d = 1; d < 16; d <<= 1) mx = fmaxf(mx, __shfl_xor(mx, d, 64));
                float ev[kPassEnds], sum = 0.f;
#pragma unroll
                for (int k = 0; k < kPassEnds; ++k) {
                    ev[k] = 16 * k + j < C ? expf(zv[k] - mx) : 0.f;
                    sum += ev[k];
                }
                sum = sum16(sum);
                float picked = 0.f;
#pragma unroll
                for (int k = 0; k < kPassEnds; ++k)
                    if (16 * k + j < C) {
                        const bool hit = 16 * k + j == t;
                        zr[16 * k + j] = on ? (ev[k] / sum - (hit ? 1.f : 0.f)) / (float)n : 0.f;
                        if (hit) picked = zv[k] - mx;
                    }
                picked = sum16(picked);
                if (on && j == 0) loss -= picked - logf(sum);
            }
            __syncthreads();
            // dW3 += H2^T dZ;  dH2 = dZ W3^T where H2 > 0, in H2's place
            f32x4 dh = zero;
            if (hidden) {
                tile_outer<kPassEnds>(H2 + 16 * wave, hs, Z, cs, lane, d3);
                dh = tile_product(Z, cs, 1, W3 + 16 * wave * cs, 1, cs, Cp, lane, zero);
            }
            if (tid < C)
                db3 += column_sum(Z + tid, cs);
            __syncthreads();
            if (hidden) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    float* h = H2 + (row4 + r) * hs + 16 * wave + col;
                    *h = *h <= 0.f ? 0.f : dh[r];
                }
            }
            __syncthreads();
            // dW2 += H1^T dH2;  dH1 = dH2 W2^T where H1 > 0, in H1's place
            if (hidden) {
                tile_outer<kPassWaves>(H1 + 16 * wave, hs, H2, hs, lane, d2);
                dh = tile_product(H2, hs, 1, W2 + 16 * wave * hs, 1, hs, Hp, lane, zero);
            }
            if (tid < H)
                db2 += column_sum(H2 + tid, hs);
            __syncthreads();
            if (hidden) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    float* h = H1 + (row4 + r) * hs + 16 * wave + col;
                    *h = *h <= 0.f ? 0.f : dh[r];
                }
            }
            __syncthreads();
            // dW1 += X^T dH1
            if (hidden) {
                tile_outer<kPassEnds>(H1 + 16 * wave, hs, X, is, lane, d1);
            }
            if (tid < H)
                db1 += column_sum(H1 + tid, hs);
        }
        __syncthreads();  // every wave is done with X, H1 and H2
    }
    if constexpr (TRAIN) {
        float* losses = lds + s.losses();
        if (tid < 16 * kPassSamples && (tid & 15) == 0) losses[tid >> 4] = loss;
        float* o = part + (size_t)blockIdx.x * (s.params() + 1);
        float *o1 = o, *ob1 = o1 + I * H, *o2 = ob1 + H, *ob2 = o2 + H * H, *o3 = ob2 + H, *ob3 = o3 + H * C;
        // through the weights' LDS, so that the stores are whole rows (the
        // tiles past a matrix' padding are dropped here)
        if (hidden) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int own = 16 * wave + row4 + r;
#pragma unroll
                for (int t = 0; t < kPassWaves; ++t)
                    if (16 * t < Hp) W2[own * hs + 16 * t + col] = d2[t][r];
#pragma unroll
                for (int t = 0; t < kPassEnds; ++t) {
                    if (16 * t < Cp) W3[own * cs + 16 * t + col] = d3[t][r];
                    if (16 * t < Ip) W1[(16 * t + col) * hs + own] = d1[t][r];
                }
            }
        }
        __syncthreads();
        store_rows(W1, hs, I, H, o1, wave, lane);
        store_rows(W2, hs, H, H, o2, wave, lane);
        store_rows(W3, cs, H, C, o3, wave, lane);
        if (tid < H) ob1[tid] = db1, ob2[tid] = db2;
        if (tid < C) ob3[tid] = db3;
        if (tid == 0) {
            float l = 0.f;
            for (int m = 0; m < kPassSamples; ++m) l += losses[m];
            o[s.params()] = l;
        }
    }
}

struct AdamStep {
    float lr, b1, b2, eps, c1, c2;  // c1 = 1 - b1^t, c2 = 1 - b2^t
};

struct AdamState {
    float p, m, v;
};
__device__ __forceinline__ AdamState adam(const AdamStep& a, float gi, AdamState o) {
    const float mi = a.b1 * o.m + (1.f - a.b1) * gi;
    const float vi = a.b2 * o.v + (1.f - a.b2) * gi * gi;
    return {o.p - a.lr * (mi / a.c1) / (sqrtf(vi / a.c2) + a.eps), mi, vi};
}

__global__ void adam_kernel(const float* __restrict__ g, long long n, AdamStep a, float* __restrict__ p,
                            float* __restrict__ m, float* __restrict__ v) {
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const AdamState q = adam(a, g[i], AdamState{p[i], m[i], v[i]});
    p[i] = q.p;
    m[i] = q.m;
    v[i] = q.v;
}

// Gradient i = the sum of the groups' shares (FP64, group class mod 8, then
// the classes in order), entry np the mean loss; with `update` the Adam step
// follows.  64 parameters per workgroup, each wave one class, its loads in
// flight together.
__global__ __launch_bounds__(kPassThreads) void mlp_update_kernel(const float* __restrict__ part, int groups, int np,
                                                                  int n, float* __restrict__ g,
                                                                  float* __restrict__ loss, int update, AdamStep a,
                                                                  float* __restrict__ p, float* __restrict__ m,
                                                                  float* __restrict__ v) {
    __shared__ double sums[kPassWaves][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int i = blockIdx.x * 64 + lane;
    AdamState state{0.f, 0.f, 0.f};
    if (update && w == 0 && i < np) state = AdamState{p[i], m[i], v[i]};  // loads with the shares
    double s = 0.0;
    if (i <= np)
        for (int k = w; k < groups; k += 16 * kPassWaves) {
            float t[16];
#pragma unroll
            for (int u = 0; u < 16; ++u) {
                const int q = k + u * kPassWaves;
                t[u] = q < groups ? part[(size_t)q * (np + 1) + i] : 0.f;
            }
#pragma unroll
            for (int u = 0; u < 16; ++u) s += (double)t[u];
        }
    sums[w][lane] = s;
    __syncthreads();
    if (w || i > np) return;
    s = 0.0;
#pragma unroll
    for (int k = 0; k < kPassWaves; ++k) s += sums[k][lane];
    if (i == np) {
        *loss = (float)(s / (double)n);
        return;
    }
    g[i] = (float)s;
    if (!update) return;
    state = adam(a, (float)s, state);
    p[i] = state.p;
    m[i] = state.m;
    v[i] = state.v;
}

__global__ void argmax_kernel(const float* __restrict__ Z, int n, int c, int* __restrict__ out) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    int best = 0;
    for (int j = 1; j < c; ++j)
        if (Z[(size_t)i * c + j] > Z[(size_t)i * c + best]) best = j;
    out[i] = best;
}

dim3 blocks(long long n) { return dim3((unsigned)((n + 255) / 256)); }

}  // namespace

struct clspmv_mlp_s {
    clspmv_ctx_t ctx = nullptr;
    int in = 0, hid = 0, cls = 0;
    long long np = 0;
    DevBuf p, g, m, v;          // parameters, gradients, Adam moments
    long long t = 0;            // Adam steps taken since creation or the last set_params
    DevBuf x, y, h1, h2, z;     // activations for the current n
    DevBuf d1, d2, dz, loss_i, loss;
    DevBuf part;                // one-CU networks: the workgroups' gradient shares
    int cap = 0;                // samples the activation buffers hold
    MlpShape shape{};
    bool one_cu = false;        // mlp_pass_kernel / mlp_update_kernel (else layer by layer)
    float *W1 = nullptr, *b1 = nullptr, *W2 = nullptr, *b2 = nullptr, *W3 = nullptr, *b3 = nullptr;
    float *gW1 = nullptr, *gb1 = nullptr, *gW2 = nullptr, *gb2 = nullptr, *gW3 = nullptr, *gb3 = nullptr;
    ~clspmv_mlp_s() {
        for (DevBuf* b : {&p, &g, &m, &v, &x, &y, &h1, &h2, &z, &d1, &d2, &dz, &loss_i, &loss, &part}) b->release();
    }
    void slice(float* base, float*& w1, float*& c1, float*& w2, float*& c2, float*& w3, float*& c3) const {
        w1 = base;
        c1 = w1 + (size_t)in * hid;
        w2 = c1 + hid;
        c2 = w2 + (size_t)hid * hid;
        w3 = c2 + hid;
        c3 = w3 + (size_t)hid * cls;
    }
    hipStream_t st() const { return ctx->stream(); }
    static int groups(int n) {
        return (int)std::min<long long>(((long long)n + kPassSamples - 1) / kPassSamples, kPassGroups);
    }
    // Loss and gradients of the n uploaded samples; with `update` the Adam
    // step too.
    void step(int n, bool update, const AdamStep& a) {
        if (!one_cu) {
            forward(n);
            backward(n);
            if (update)
                hipLaunchKernelGGL(adam_kernel, blocks(np), dim3(256), 0, st(), (const float*)g.ptr, np, a,
                                   (float*)p.ptr, (float*)m.ptr, (float*)v.ptr);
            return;
        }
        hipLaunchKernelGGL(mlp_pass_kernel<true>, dim3(groups(n)), dim3(kPassThreads), 0, st(), shape,
                           (const float*)p.ptr, (const float*)x.ptr, (const int*)y.ptr, n, (float*)part.ptr,
                           (float*)nullptr);
        hipLaunchKernelGGL(mlp_update_kernel, dim3((unsigned)(np / 64 + 1)), dim3(kPassThreads), 0, st(),
                           (const float*)part.ptr, groups(n), (int)np, n, (float*)g.ptr, (float*)loss.ptr, update, a,
                           (float*)p.ptr, (float*)m.ptr, (float*)v.ptr);
    }
    int ensure(int n) {
        if (n <= cap) return CLSPMV_OK;
        cap = 0;
        for (DevBuf* b : {&x, &y, &h1, &h2, &z, &d1, &d2, &dz, &loss_i, &part}) b->release();
        int rc = x.alloc((size_t)n * in * 4);
        if (!rc) rc = y.alloc((size_t)n * 4);
        if (!rc) rc = z.alloc((size_t)n * cls * 4);
        if (one_cu) {
            if (!rc) rc = part.alloc((size_t)groups(n) * (size_t)(np + 1) * 4);
            if (!rc) cap = n;
            return rc;
        }
        if (!rc) rc = h1.alloc((size_t)n * hid * 4);
        if (!rc) rc = h2.alloc((size_t)n * hid * 4);
        if (!rc) rc = d1.alloc((size_t)n * hid * 4);
        if (!rc) rc = d2.alloc((size_t)n * hid * 4);
        if (!rc) rc = dz.alloc((size_t)n * cls * 4);
        if (!rc) rc = loss_i.alloc((size_t)n * 4);
        if (!rc) cap = n;
        return rc;
    }
    void gemm(int M, int N, int K, const float* A, int ta, const float* B, int tb, float* C, int acc) {
        hipLaunchKernelGGL(gemm_kernel, dim3((N + kT - 1) / kT, (M + kT - 1) / kT), dim3(kT * kT), 0, st(), M, N,
                           K, A, ta, B, tb, C, acc);
    }
    void colsum(const float* A, int M, int N, float scale, float* out) {
        hipLaunchKernelGGL(colsum_kernel, dim3((unsigned)((N + 63) / 64)), dim3(1024), 0, st(), A, M, N, scale, out);
    }
    // Logits of the n uploaded samples (the layers' activations too where
    // the network runs layer by layer).
    void forward(int n) {
        if (one_cu) {
            hipLaunchKernelGGL(mlp_pass_kernel<false>, dim3(groups(n)), dim3(kPassThreads), 0, st(), shape,
                               (const float*)p.ptr, (const float*)x.ptr, (const int*)nullptr, n, (float*)nullptr,
                               (float*)z.ptr);
            return;
        }
        const float* X = (const float*)x.ptr;
        float *H1 = (float*)h1.ptr, *H2 = (float*)h2.ptr, *Z = (float*)z.ptr;
        gemm(n, hid, in, X, 0, W1, 0, H1, 0);
        hipLaunchKernelGGL(bias_act_kernel, blocks((long long)n * hid), dim3(256), 0, st(), H1, b1, n, hid, 1);
        gemm(n, hid, hid, H1, 0, W2, 0, H2, 0);
        hipLaunchKernelGGL(bias_act_kernel, blocks((long long)n * hid), dim3(256), 0, st(), H2, b2, n, hid, 1);
        gemm(n, cls, hid, H2, 0, W3, 0, Z, 0);
        hipLaunchKernelGGL(bias_act_kernel, blocks((long long)n * cls), dim3(256), 0, st(), Z, b3, n, cls, 0);
    }
    void backward(int n) {
        const float* X = (const float*)x.ptr;
        float *H1 = (float*)h1.ptr, *H2 = (float*)h2.ptr, *Z = (float*)z.ptr;
        float *D1 = (float*)d1.ptr, *D2 = (float*)d2.ptr, *DZ = (float*)dz.ptr;
        hipLaunchKernelGGL(softmax_ce_kernel, blocks(n), dim3(256), 0, st(), Z, (const int*)y.ptr, n, cls, DZ,
                           (float*)loss_i.ptr);
        colsum((const float*)loss_i.ptr, n, 1, 1.f / (float)n, (float*)loss.ptr);
        gemm(hid, cls, n, H2, 1, DZ, 0, gW3, 0);                       // dW3 = H2^T dZ
        colsum(DZ, n, cls, 1.f, gb3);
        gemm(n, hid, cls, DZ, 0, W3, 1, D2, 0);                        // dH2 = dZ W3^T
        hipLaunchKernelGGL(relu_back_kernel, blocks((long long)n * hid), dim3(256), 0, st(), D2, H2, n * hid);
        gemm(hid, hid, n, H1, 1, D2, 0, gW2, 0);                       // dW2 = H1^T dH2
        colsum(D2, n, hid, 1.f, gb2);
        gemm(n, hid, hid, D2, 0, W2, 1, D1, 0);                        // dH1 = dH2 W2^T
        hipLaunchKernelGGL(relu_back_kernel, blocks((long long)n * hid), dim3(256), 0, st(), D1, H1, n * hid);
        gemm(in, hid, n, X, 1, D1, 0, gW1, 0);                         // dW1 = X^T dH1
        colsum(D1, n, hid, 1.f, gb1);
    }
    int upload(const float* hx, const int* hy, int n) {
        int rc = ensure(n);
        if (!rc) rc = hip_status(hipMemcpyAsync(x.ptr, hx, (size_t)n * in * 4, hipMemcpyHostToDevice, st()), "h2d");
        if (!rc && hy) rc = hip_status(hipMemcpyAsync(y.ptr, hy, (size_t)n * 4, hipMemcpyHostToDevice, st()), "h2d");
        return rc;
    }
};

extern "C" {

int clspmv_mlp_create(clspmv_ctx_t ctx, int in, int hidden, int classes, uint64_t seed, clspmv_mlp_t* out) {
    if (!ctx || !out || in <= 0 || hidden <= 0 || classes <= 1 || hidden > 4096 || in > 4096) return CLSPMV_E_INVALID;
    auto* m = new (std::nothrow) clspmv_mlp_s();
    if (!m) return CLSPMV_E_NOMEM;
    m->ctx = ctx;
    m->in = in;
    m->hid = hidden;
    m->cls = classes;
    m->shape = MlpShape{in, hidden, classes};
    m->one_cu = m->shape.one_cu();
    m->np = (long long)in * hidden + hidden + (long long)hidden * hidden + hidden + (long long)hidden * classes + classes;
    // He-uniform weights from a SplitMix64 stream, zero biases
    std::vector<float> h((size_t)m->np, 0.f);
    uint64_t s = seed;
    auto next = [&]() {
        uint64_t z = (s += 0x9E3779B97F4A7C15ull);
        z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
        z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
        z ^= z >> 31;
        return (double)(z >> 11) * (1.0 / 9007199254740992.0);
    };
    auto fill = [&](size_t off, long long fan_in, long long count) {
        const double a = std::sqrt(6.0 / (double)fan_in);
        for (long long i = 0; i < count; ++i) h[off + (size_t)i] = (float)((2.0 * next() - 1.0) * a);
    };
    size_t off = 0;
    fill(off, in, (long long)in * hidden);
    off += (size_t)in * hidden + hidden;
    fill(off, hidden, (long long)hidden * hidden);
    off += (size_t)hidden * hidden + hidden;
    fill(off, hidden, (long long)hidden * classes);
    int rc = m->p.upload(ctx, h.data(), h.size() * 4);
    std::fill(h.begin(), h.end(), 0.f);
    if (!rc) rc = m->g.upload(ctx, h.data(), h.size() * 4);
    if (!rc) rc = m->m.upload(ctx, h.data(), h.size() * 4);
    if (!rc) rc = m->v.upload(ctx, h.data(), h.size() * 4);
    if (!rc) rc = m->loss.alloc(4);
    if (rc) {
        delete m;
        return rc;
    }
    m->slice((float*)m->p.ptr, m->W1, m->b1, m->W2, m->b2, m->W3, m->b3);
    m->slice((float*)m->g.ptr, m->gW1, m->gb1, m->gW2, m->gb2, m->gW3, m->gb3);
    *out = m;
    return CLSPMV_OK;
}

int clspmv_mlp_free(clspmv_mlp_t m) {
    if (!m) return CLSPMV_E_INVALID;
    (void)hipStreamSynchronize(m->st());
    delete m;
    return CLSPMV_OK;
}

long long clspmv_mlp_num_params(clspmv_mlp_t m) { return m ? m->np : 0; }

int clspmv_mlp_get_params(clspmv_mlp_t m, float* params) {
    if (!m || !params) return CLSPMV_E_INVALID;
    return clspmv_memcpy_d2h(m->ctx, params, m->p.ptr, (size_t)m->np * 4);
}
// New parameters start a new optimisation: the Adam moments and step count
// are reset with them.
int clspmv_mlp_set_params(clspmv_mlp_t m, const float* params) {
    if (!m || !params) return CLSPMV_E_INVALID;
    int rc = clspmv_memcpy_h2d(m->ctx, m->p.ptr, params, (size_t)m->np * 4);
    if (!rc) rc = hip_status(hipMemsetAsync(m->m.ptr, 0, (size_t)m->np * 4, m->st()), "hipMemset");
    if (!rc) rc = hip_status(hipMemsetAsync(m->v.ptr, 0, (size_t)m->np * 4, m->st()), "hipMemset");
    if (!rc) m->t = 0;
    return rc;
}

static int check_labels(const clspmv_mlp_s* m, const int* labels, int n) {
    for (int i = 0; i < n; ++i)
        if (labels[i] < 0 || labels[i] >= m->cls) {
            set_error("label %d of sample %d outside [0, %d)", labels[i], i, m->cls);
            return CLSPMV_E_INVALID;
        }
    return CLSPMV_OK;
}

int clspmv_mlp_loss_grad(clspmv_mlp_t m, const float* x, const int* labels, int n, float* loss, float* grads) {
    if (!m || !x || !labels || n <= 0) return CLSPMV_E_INVALID;
    int rc = check_labels(m, labels, n);
    if (!rc) rc = m->upload(x, labels, n);
    if (rc) return rc;
    m->step(n, false, AdamStep{});
    rc = hip_status(hipGetLastError(), "mlp kernels");
    if (!rc && loss) rc = clspmv_memcpy_d2h(m->ctx, loss, m->loss.ptr, 4);
    if (!rc && grads) rc = clspmv_memcpy_d2h(m->ctx, grads, m->g.ptr, (size_t)m->np * 4);
    return rc;
}

int clspmv_mlp_train(clspmv_mlp_t m, const float* x, const int* labels, int n, int steps, float lr, float beta1,
                     float beta2, float eps, float* loss) {
    if (!m || !x || !labels || n <= 0 || steps < 0) return CLSPMV_E_INVALID;
    int rc = check_labels(m, labels, n);
    if (!rc) rc = m->upload(x, labels, n);
    if (rc) return rc;
    // the step count continues across calls, as the moments do, so that a
    // run split over several calls takes the same steps as one call
    for (int s = 0; s < steps; ++s) {
        const long long t = ++m->t;
        m->step(n, true,
                AdamStep{lr, beta1, beta2, eps, (float)(1.0 - std::pow((double)beta1, (double)t)),
                         (float)(1.0 - std::pow((double)beta2, (double)t))});
    }
    m->step(n, false, AdamStep{});
    rc = hip_status(hipGetLastError(), "mlp train");
    if (!rc && loss) rc = clspmv_memcpy_d2h(m->ctx, loss, m->loss.ptr, 4);
    return rc;
}

int clspmv_mlp_predict(clspmv_mlp_t m, const float* x, int n, float* logits, int* classes) {
    if (!m || !x || n <= 0) return CLSPMV_E_INVALID;
    int rc = m->upload(x, nullptr, n);
    if (rc) return rc;
    m->forward(n);
    hipLaunchKernelGGL(argmax_kernel, blocks(n), dim3(256), 0, m->st(), (const float*)m->z.ptr, n, m->cls,
                       (int*)m->y.ptr);
    rc = hip_status(hipGetLastError(), "mlp predict");
    if (!rc && logits) rc = clspmv_memcpy_d2h(m->ctx, logits, m->z.ptr, (size_t)n * m->cls * 4);
    if (!rc && classes) rc = clspmv_memcpy_d2h(m->ctx, classes, m->y.ptr, (size_t)n * 4);
    return rc;
}

}  // extern "C"
