// The selector network: forward, softmax cross-entropy, backward and Adam,
// as hand-written HIP kernels (FP32).  A network whose weights fit one CU's
// LDS (the selector's 24 -> 128 -> 128 -> 22 does) takes two launches per
// step: mlp_pass_kernel, one workgroup per 16 samples from x to the gradient
// of every layer's input, and mlp_update_kernel, one wave per 16 x 16 tile of
// the weight gradients, which takes the Adam step too.  Larger networks run
// layer by layer: an LDS-tiled GEMM kernel with transpose flags, bias /
// activation and reduction kernels.  Every sum has a fixed order, the same in
// both: training is deterministic for a given seed.
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

// out[j] = (sum_i A[i][j], i ascending) / div: one workgroup per 64 columns,
// whose 16 waves load kColsumRows rows to LDS while the first adds up those
// before, in order: the chain of mlp_update_kernel's sums, the same bits.
constexpr int kColsumRows = 128;
__global__ __launch_bounds__(1024) void colsum_kernel(const float* __restrict__ A, int M, int N, float div,
                                                      float* __restrict__ out) {
    constexpr int U = kColsumRows / 16;
    __shared__ float part[2][kColsumRows][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int j = blockIdx.x * 64 + lane;
    const float* col = A + min(j, N - 1);
    float s = 0.f;
    for (int i0 = 0, b = 0; i0 < M + kColsumRows; i0 += kColsumRows, b ^= 1) {
        if (i0 < M) {
            float v[U];
#pragma unroll
            for (int u = 0; u < U; ++u) v[u] = col[(size_t)min(i0 + w + 16 * u, M - 1) * N];
#pragma unroll
            for (int u = 0; u < U; ++u) part[b][w + 16 * u][lane] = v[u];
        }
        if (w == 0 && i0 > 0) {
            const int n = min(kColsumRows, M - (i0 - kColsumRows));
#pragma unroll 16
            for (int i = 0; i < n; ++i) s += part[b ^ 1][i][lane];
        }
        __syncthreads();
    }
    if (w == 0 && j < N) out[j] = s / div;
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
    __host__ __device__ int floats() const { return z() + kPassSamples * lds_stride(cp()); }
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

// What the passes of a training step hand to mlp_update_kernel, a row per
// sample: the hidden activations, the gradients of the two hidden layers'
// and the logits' inputs, the losses.
struct MlpActs {
    float *h1, *h2, *d1, *d2, *dz, *loss_i;
};

// Forward pass of 16 samples at a time and, TRAIN, loss and the gradients of
// every layer's input: the workgroup's weights stay in LDS, the activations
// of a tile too.  TRAIN writes them to `acts`, else the logits to zout.  Each
// sum runs over its terms in ascending order in one chain of fused
// multiply-adds, as gemm_kernel's, softmax_ce_kernel's and colsum_kernel's do:
// the same bits.
// Bound by what one CU can draw (90 KB of weights per workgroup, 7 us) and by
// the chain of layers.  20 training steps of the 24-128-128-22 network on
// 1920 samples take 1.11 ms with the update kernel, 28.3 to 29.0 ms layer by
// layer with 20 launches a step (column sums by one thread per column 330 us,
// 16 x 16 tiles on the VALU 30 us each), bitwise the same.  Weight gradients
// kept per workgroup and added afterwards took 0.83 ms, but round differently,
// and a hidden unit that then changes sides of zero moves the parameters by
// 1e-5 within a few Adam steps.
template <bool TRAIN>
__global__ __launch_bounds__(kPassThreads) void mlp_pass_kernel(MlpShape s, const float* __restrict__ p,
                                                                const float* __restrict__ x,
                                                                const int* __restrict__ label, int n,
                                                                MlpActs acts, float* __restrict__ zout) {
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
    // rows row4 .. + 3 of column 16 wave + col of a tile to a samples x cols array
    auto keep = [&](float* dst, int cols, int s0, const float (&v)[4]) {
        if (TRAIN && 16 * wave + col < cols)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (s0 + row4 + r < n) dst[(size_t)(s0 + row4 + r) * cols + 16 * wave + col] = v[r];
    };
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
            float h[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                h[r] = fmaxf(v[r] + B1[16 * wave + col], 0.f);
                H1[(row4 + r) * hs + 16 * wave + col] = h[r];
            }
            keep(acts.h1, H, s0, h);
        }
        __syncthreads();
        if (hidden) {
            const f32x4 v = tile_product(H1, hs, 1, W2 + 16 * wave, hs, 1, Hp, lane, zero);
            float h[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                h[r] = fmaxf(v[r] + B2[16 * wave + col], 0.f);
                H2[(row4 + r) * hs + 16 * wave + col] = h[r];
            }
            keep(acts.h2, H, s0, h);
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
                for (int k = 0; k < kPassEnds; ++k) ev[k] = 16 * k + j < C ? expf(zv[k] - mx) : 0.f;
#pragma unroll
                for (int k = 0; k < kPassEnds; ++k)
                    for (int c = 0; c < min(16, C - 16 * k); ++c) sum += __shfl(ev[k], (lane & 48) + c, 64);
#pragma unroll
                for (int k = 0; k < kPassEnds; ++k)
                    if (16 * k + j < C) {
                        const bool hit = 16 * k + j == t;
                        const float dz = on ? (ev[k] / sum - (hit ? 1.f : 0.f)) / (float)n : 0.f;
                        zr[16 * k + j] = dz;
                        if (on) acts.dz[(size_t)(s0 + m) * C + 16 * k + j] = dz;
                        if (on && hit) acts.loss_i[s0 + m] = -(zv[k] - mx - logf(sum));
                    }
            }
            __syncthreads();
            // dH2 = dZ W3^T where H2 > 0, in H2's place (each lane its own)
            if (hidden) {
                const f32x4 v = tile_product(Z, cs, 1, W3 + 16 * wave * cs, 1, cs, Cp, lane, zero);
                float d[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    float* h = H2 + (row4 + r) * hs + 16 * wave + col;
                    d[r] = *h <= 0.f ? 0.f : v[r];
                    *h = d[r];
                }
                keep(acts.d2, H, s0, d);
            }
            __syncthreads();
            // dH1 = dH2 W2^T where H1 > 0
            if (hidden) {
                const f32x4 v = tile_product(H2, hs, 1, W2 + 16 * wave * hs, 1, hs, Hp, lane, zero);
                float d[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) d[r] = H1[(row4 + r) * hs + 16 * wave + col] <= 0.f ? 0.f : v[r];
                keep(acts.d1, H, s0, d);
            }
        }
        __syncthreads();  // every wave is done with X, H1 and H2
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

// Gradients, mean loss and, with `update`, the Adam step.  A workgroup is one
// wave with one 16 x 16 tile of a weight gradient, P^T Q over the n samples in
// ascending order in one chain of matrix-core products (the bits of
// gemm_kernel's chain of fused multiply-adds); a bias gradient and the loss
// are such tiles with P = 1.  kUpdRows samples' operands are loaded ahead of
// those that multiply: the chain (8 cycles per sample) then hides most of the
// loads (64 rows 9 % slower, 192 rows 7 %).
constexpr int kUpdRows = 128;
__global__ __launch_bounds__(64) void mlp_update_kernel(MlpShape s, const float* __restrict__ x, MlpActs acts, int n,
                                                        float* __restrict__ g, float* __restrict__ loss, int update,
                                                        AdamStep a, float* __restrict__ p, float* __restrict__ m,
                                                        float* __restrict__ v) {
    const int lane = threadIdx.x, i = lane & 15, q = lane >> 4;
    const int I = s.in, H = s.hid, C = s.cls, It = s.inp() / 16, Ht = s.hp() / 16, Ct = s.cp() / 16;
    // the tile: P (null: ones) and Q with their widths, the tile's position
    // and the offset of the gradient it belongs to
    const float *P = nullptr, *Q;
    int pw = 1, qw, ti = 0, tj, off;
    const int o1 = 0, ob1 = I * H, o2 = ob1 + H, ob2 = o2 + H * H, o3 = ob2 + H, ob3 = o3 + H * C;
    int b = blockIdx.x;
    if (b < Ht * Ht) P = acts.h1, pw = H, Q = acts.d2, qw = H, ti = b / Ht, tj = b % Ht, off = o2;
    else if ((b -= Ht * Ht) < It * Ht) P = x, pw = I, Q = acts.d1, qw = H, ti = b / Ht, tj = b % Ht, off = o1;
    else if ((b -= It * Ht) < Ht * Ct) P = acts.h2, pw = H, Q = acts.dz, qw = C, ti = b / Ct, tj = b % Ct, off = o3;
    else if ((b -= Ht * Ct) < Ht) Q = acts.d1, qw = H, tj = b, off = ob1;
    else if ((b -= Ht) < Ht) Q = acts.d2, qw = H, tj = b, off = ob2;
    else if ((b -= Ht) < Ct) Q = acts.dz, qw = C, tj = b, off = ob3;
    else Q = acts.loss_i, qw = 1, tj = 0, off = -1;
    const int pc = min(16 * ti + i, pw - 1), qc = min(16 * tj + i, qw - 1);  // columns past the edge: never stored
    constexpr int U = kUpdRows / 4;
    float pv[U], qv[U];
    auto load = [&](int k0, float (&pn)[U], float (&qn)[U]) {
        const bool whole = k0 + kUpdRows <= n;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = k0 + 4 * u + q, kc = whole ? k : min(k, n - 1);
            pn[u] = P ? P[(size_t)kc * pw + pc] : 1.f;
            qn[u] = Q[(size_t)kc * qw + qc];
            if (k >= n) pn[u] = qn[u] = 0.f;
        }
    };
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    load(0, pv, qv);
    for (int k0 = 0; k0 < n; k0 += kUpdRows) {
        float pn[U], qn[U];
        if (k0 + kUpdRows < n) load(k0 + kUpdRows, pn, qn);
#pragma unroll
        for (int u = 0; u < U; ++u) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(pv[u], qv[u], acc, 0, 0, 0);
#pragma unroll
        for (int u = 0; u < U; ++u) pv[u] = pn[u], qv[u] = qn[u];
    }
    if (off < 0) {
        if (lane == 0) *loss = acc[0] / (float)n;
        return;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int row = 16 * ti + 4 * q + r, c = 16 * tj + i;
        if (row >= pw || c >= qw) continue;
        const int at = off + row * qw + c;
        g[at] = acc[r];
        if (!update) continue;
        const AdamState w = adam(a, acc[r], AdamState{p[at], m[at], v[at]});
        p[at] = w.p;
        m[at] = w.m;
        v[at] = w.v;
    }
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
    int cap = 0;                // samples the activation buffers hold
    MlpShape shape{};
    bool one_cu = false;        // mlp_pass_kernel / mlp_update_kernel (else layer by layer)
    float *W1 = nullptr, *b1 = nullptr, *W2 = nullptr, *b2 = nullptr, *W3 = nullptr, *b3 = nullptr;
    float *gW1 = nullptr, *gb1 = nullptr, *gW2 = nullptr, *gb2 = nullptr, *gW3 = nullptr, *gb3 = nullptr;
    ~clspmv_mlp_s() {
        for (DevBuf* b : {&p, &g, &m, &v, &x, &y, &h1, &h2, &z, &d1, &d2, &dz, &loss_i, &loss}) b->release();
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
        const MlpActs acts{(float*)h1.ptr, (float*)h2.ptr, (float*)d1.ptr, (float*)d2.ptr, (float*)dz.ptr,
                           (float*)loss_i.ptr};
        hipLaunchKernelGGL(mlp_pass_kernel<true>, dim3(groups(n)), dim3(kPassThreads), 0, st(), shape,
                           (const float*)p.ptr, (const float*)x.ptr, (const int*)y.ptr, n, acts, (float*)nullptr);
        const int It = shape.inp() / 16, Ht = shape.hp() / 16, Ct = shape.cp() / 16;
        hipLaunchKernelGGL(mlp_update_kernel, dim3(Ht * Ht + It * Ht + Ht * Ct + 2 * Ht + Ct + 1), dim3(64), 0, st(),
                           shape, (const float*)x.ptr, acts, n, (float*)g.ptr, (float*)loss.ptr, update, a,
                           (float*)p.ptr, (float*)m.ptr, (float*)v.ptr);
    }
    int ensure(int n) {
        if (n <= cap) return CLSPMV_OK;
        cap = 0;
        for (DevBuf* b : {&x, &y, &h1, &h2, &z, &d1, &d2, &dz, &loss_i}) b->release();
        int rc = x.alloc((size_t)n * in * 4);
        if (!rc) rc = y.alloc((size_t)n * 4);
        if (!rc) rc = z.alloc((size_t)n * cls * 4);
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
    void colsum(const float* A, int M, int N, float div, float* out) {
        hipLaunchKernelGGL(colsum_kernel, dim3((unsigned)((N + 63) / 64)), dim3(1024), 0, st(), A, M, N, div, out);
    }
    // Logits of the n uploaded samples (the layers' activations too where
    // the network runs layer by layer).
    void forward(int n) {
        if (one_cu) {
            hipLaunchKernelGGL(mlp_pass_kernel<false>, dim3(groups(n)), dim3(kPassThreads), 0, st(), shape,
                               (const float*)p.ptr, (const float*)x.ptr, (const int*)nullptr, n, MlpActs{},
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
        colsum((const float*)loss_i.ptr, n, 1, (float)n, (float*)loss.ptr);
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
