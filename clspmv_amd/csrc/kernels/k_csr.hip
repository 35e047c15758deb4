// CSR SpMV kernels (y += A*x) for gfx950.
//
//  * csr_scalar: one lane per row (A/kernels/spmv_csr_scalar.cl:5-23 is the
//    same one-thread-per-row scheme); used by spmv_all method 1.
//  * csr_vector<L>: L lanes per row (L = 2..64 picked from the mean row
//    length), DPP/shuffle group reduction.  The reference's CSR-vector uses
//    a fixed 32-lane "warp" per row (A/kernels/spmv_csr_vector.cl:4-40).
//  * csr_adaptive: rows of at most 64 entries in row groups
//    (csr_adaptive_kernel: one to sixteen lanes per row, the entries of 64
//    lanes interleaved at upload), the others by host-planned blocks
//    (csr_block):
//      STREAM  rows of a group that the groups' layout would pad too much,
//              up to 64 of them with at most 512 nnz;
//      VECTOR  one row of 65..1024 nnz: the wave strides the row and
//              reduces across its 64 lanes;
//      LONG    one 1024-nnz chunk of a longer row: the wave's partial is
//              stored in FP64 and a second kernel adds the partials of each
//              long row in order (deterministic, no atomics).
#include "kcommon.hpp"
#include "launch.hpp"

#include <algorithm>
#include <type_traits>

namespace clspmv {
namespace dev {

__global__ __launch_bounds__(256) void csr_scalar_kernel(const int* __restrict__ rp, const int* __restrict__ col,
                                                         const float* __restrict__ val,
                                                         const float* __restrict__ x, float* __restrict__ y,
                                                         int rows) {
    const int row = blockIdx.x * 256 + threadIdx.x;
    if (row >= rows) return;
    const int s = rp[row], e = rp[row + 1];
    float acc = y[row];
    for (int k = s; k < e; ++k) acc = fmaf(val[k], x[col[k]], acc);
    y[row] = acc;
}

template <int L>
__global__ __launch_bounds__(256) void csr_vector_kernel(const int* __restrict__ rp, const int* __restrict__ col,
                                                         const float* __restrict__ val,
                                                         const float* __restrict__ x, float* __restrict__ y,
                                                         int rows) {
    const int gid = blockIdx.x * 256 + threadIdx.x;
    const int lane = threadIdx.x & (L - 1);
    const int row = gid / L;
    if (row >= rows) return;  // whole L-groups exit together (L divides 256)
    const int s = rp[row], e = rp[row + 1];
    float acc = 0.f;
    int k = s + lane;
    for (; k + 3 * L < e; k += 4 * L) {
        int c0 = ld_stream(col + k), c1 = ld_stream(col + k + L), c2 = ld_stream(col + k + 2 * L),
            c3 = ld_stream(col + k + 3 * L);
        float v0 = ld_stream(val + k), v1 = ld_stream(val + k + L), v2 = ld_stream(val + k + 2 * L),
              v3 = ld_stream(val + k + 3 * L);
        acc = fmaf(v0, x[c0], acc);
        acc = fmaf(v1, x[c1], acc);
        acc = fmaf(v2, x[c2], acc);
        acc = fmaf(v3, x[c3], acc);
    }
    for (; k < e; k += L) acc = fmaf(ld_stream(val + k), x[ld_stream(col + k)], acc);
    acc = group_sum<L>(acc);
    if (lane == 0 && e > s) y[row] += acc;
}

// U x 64 products of a STREAM block (n <= 64 U entries) to LDS, every load
// issued before the first use: past the block's end the last entry is read
// again, as a branch around each load would wait for it (with that, and sums
// reading eight products at a time, 3000 rows of 1 with a 64 in every 512 take
// 3.1 us instead of 4.6, 1M 7.0 instead of 10.4).
template <int U>
__device__ __forceinline__ void csr_products(const int* __restrict__ col, const float* __restrict__ val, int n,
                                             const float* __restrict__ x, float* sh, int lane) {
    int c[U];
    float v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int k = min(lane + 64 * u, n - 1);
        c[u] = ld_stream(col + k);
        v[u] = ld_stream(val + k);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] *= x[c[u]];
#pragma unroll
    for (int u = 0; u < U; ++u)
        if (lane + 64 * u < n) sh[lane + 64 * u] = v[u];
}

// One block of rows (csr_adaptive_kernel's and csr_blocks_kernel's), by one wave:
//   {row, -(slot + 1)}  LONG, one chunk of a row: its sum to carry[slot]
//   {row, row + 1}      VECTOR, one row
//   {r0, r1}            STREAM, up to 64 rows of together at most
//                       kCsrStreamMaxNnz entries: the products go to LDS (sh,
//                       the wave's own), lane j sums row r0 + j from there;
//                       counts holds the rows' entries, a byte each, and a
//                       scan over the wave gives their offsets.
// Entries blk.z .. blk.w - 1 of col / val.
__device__ __forceinline__ void csr_block(int4 blk, const unsigned char* __restrict__ counts,
                                          const int* __restrict__ col, const float* __restrict__ val,
                                          const float* __restrict__ x, float* __restrict__ y,
                                          double* __restrict__ carry, float* sh, int lane) {
    const int r0 = blk.x, tag = blk.y, n0 = blk.z, n1 = blk.w;
    if (tag < 0 || tag - r0 == 1) {
        float acc = 0.f;
        int k = n0 + lane;
        for (; k + 192 < n1; k += 256) {
            int c0 = ld_stream(col + k), c1 = ld_stream(col + k + 64), c2 = ld_stream(col + k + 128),
                c3 = ld_stream(col + k + 192);
            float v0 = ld_stream(val + k), v1 = ld_stream(val + k + 64), v2 = ld_stream(val + k + 128),
                  v3 = ld_stream(val + k + 192);
            acc = fmaf(v0, x[c0], acc);
            acc = fmaf(v1, x[c1], acc);
            acc = fmaf(v2, x[c2], acc);
            acc = fmaf(v3, x[c3], acc);
        }
        for (; k < n1; k += 64) acc = fmaf(ld_stream(val + k), x[ld_stream(col + k)], acc);
        acc = wave_sum(acc);
        if (lane == 0) {
            if (tag < 0)
                carry[-tag - 1] = (double)acc;
            else if (n1 > n0)
                y[r0] += acc;
        }
        return;
    }
    const int n = n1 - n0;
    if (n == 0) return;  // a slice without entries in these rows
    const int r = r0 + lane;
    const int cnt = r < tag ? (int)counts[r] : 0;
    const float yo = cnt > 0 ? y[r] : 0.f;
    if (n <= 128)
        csr_products<2>(col + n0, val + n0, n, x, sh, lane);
    else if (n <= 256)
        csr_products<4>(col + n0, val + n0, n, x, sh, lane);
    else
        csr_products<kCsrStreamPerLane>(col + n0, val + n0, n, x, sh, lane);
    int k = wave_scan(cnt) - cnt;
    const int e = k + cnt;
    wave_lds_sync();
    if (cnt > 0) {
        float acc = 0.f;
        for (; k + 8 <= e; k += 8) {
            float p[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) p[u] = sh[k + u];
#pragma unroll
            for (int u = 0; u < 8; ++u) acc += p[u];
        }
        for (; k < e; ++k) acc += sh[k];
        y[r] = yo + acc;
    }
}

typedef float f32x2 __attribute__((ext_vector_type(2)));

// kCsrPairs pairs of a wave from pair p on (those past the wave's last are
// skipped, wave-uniform): two values and two columns per lane and pair.
struct CsrPairs {
    f32x2 v[kCsrPairs];
    unsigned c[kCsrPairs];
    __device__ __forceinline__ void load(const f32x2* __restrict__ val, const unsigned* __restrict__ col, int p,
                                         int pairs, int lane) {
#pragma unroll
        for (int u = 0; u < kCsrPairs; ++u)
            if (p + u < pairs) {
                v[u] = __builtin_nontemporal_load(val + (size_t)(p + u) * 64 + lane);
                c[u] = __builtin_nontemporal_load(col + (size_t)(p + u) * 64 + lane);
            }
    }
};

// A wave's pairs times x (the first kCsrPairs of them loaded by the caller):
// the lane's row holds entries 2 L p + 2 t and + 1 of pair p; entries past the
// row's length are padding (column 0 of the range, value 0) and multiply 0,
// not x, so that an infinity or NaN of x they do not belong to stays out of
// the sum.
template <int L>
__device__ __forceinline__ float csr_group_sum(CsrPairs& cur, const f32x2* __restrict__ val,
                                               const unsigned* __restrict__ col, int pairs, int len, int t, int lane,
                                               const float* xg) {
    float acc = 0.f;
    int left = len - 2 * t;  // entries of the row from this lane's first on
    for (int p = 0; p < pairs; p += kCsrPairs) {
        if (p) cur.load(val, col, p, pairs, lane);
        float xa[kCsrPairs], xb[kCsrPairs];
#pragma unroll
        for (int u = 0; u < kCsrPairs; ++u)
            if (p + u < pairs) {
                xa[u] = xg[cur.c[u] & 0xffffu];
                xb[u] = xg[cur.c[u] >> 16];
            }
#pragma unroll
        for (int u = 0; u < kCsrPairs; ++u)
            if (p + u < pairs) {
                acc = fmaf(cur.v[u].x, left > 0 ? xa[u] : 0.f, acc);
                acc = fmaf(cur.v[u].y, left > 1 ? xb[u] : 0.f, acc);
                left -= 2 * L;
            }
    }
    return acc;
}

// L lanes per row.  A workgroup of kCsrThreads threads owns one row group:
// kCsrThreads / L rows of at most 64 entries, the longest first, so that the
// 64 / L rows of a wave have nearly equal lengths; the wave's entries are
// stored pair by pair, 64 lanes side by side (8 + 4 bytes per lane and pair).
// The x range of the group is staged in LDS when it fits (kCsrWindow).
// Bound by HBM on large matrices with columns near the diagonal: 1,000,003
// rows of 9..27 entries within ~2000 columns (159 MB by CSR's count, 126 MB
// stored) take 26.0 us, 6.1 TB/s of CSR bytes.  Waves that staged 512
// consecutive entries' products in LDS and summed each row from there took
// 80 us: one L1 line per gathered x (an LDS read of the staged range is
// several times cheaper) and a chain of block descriptor, columns, x, row
// pointer and row sum in every wave.  512 threads per workgroup measured
// level with 1024 and 3 % ahead of 256 (the same matrix and 57 others); 4
// pairs in flight 2 % ahead of 2 and level with 8.
template <int L>
__global__ __launch_bounds__(kCsrThreads) void csr_adaptive_kernel(DevCsrAdaptive m, int nblock_wg,
                                                                   int blocks_per_wg,
                                                                   const float* __restrict__ x,
                                                                   float* __restrict__ y) {
    extern __shared__ float xs[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    if ((int)blockIdx.x < nblock_wg) {
        // few blocks: spread over the CUs (blocks_per_wg of the waves take
        // one).  Many: all waves, as a workgroup holds the groups' LDS (four
        // of eight: 100,000 rows of 30 or 70 20.3 -> 24.8 us)
        const int b = blockIdx.x * blocks_per_wg + wave;
        if (wave < blocks_per_wg && b < m.nblocks)
            csr_block(m.blocks[b], m.counts, m.col, m.val, x, y, m.carry, xs + wave * kCsrStreamMaxNnz, lane);
        return;
    }
    const int g = xcd_tile(blockIdx.x - nblock_wg, m.ngroups);
    const CsrGroup d = m.groups[g];
    const int p0 = m.pair[g * kCsrWaves + wave], pairs = m.pair[g * kCsrWaves + wave + 1] - p0;
    const int t = threadIdx.x % L;
    const unsigned meta = m.lane[g * (kCsrThreads / L) + threadIdx.x / L];  // length << 16 | row in group
    const int len = (int)(meta >> 16);
    float* yp = y + d.row0 + (meta & 0xffffu);
    const bool out = t == 0 && len > 0;
    const float yo = out ? *yp : 0.f;
    const f32x2* val = reinterpret_cast<const f32x2*>(m.gval) + (size_t)p0 * 64;
    const unsigned* col = m.gcol + (size_t)p0 * 64;
    CsrPairs first;
    first.load(val, col, 0, pairs, lane);  // in flight while x is staged
    const float* src = x + d.x0;
    float acc;
    if (d.mode == kCsrStaged) {
        for (int i = threadIdx.x * 4; i < d.xn; i += kCsrThreads * 4) {
            if (i + 4 <= d.xn) {
                const f32x4a4 q = *reinterpret_cast<const f32x4a4*>(src + i);
                *reinterpret_cast<float4*>(xs + i) = make_float4(q.x, q.y, q.z, q.w);
            } else {
#pragma unroll
                for (int j = 0; j < 3; ++j)
                    if (i + j < d.xn) xs[i + j] = src[i + j];
            }
        }
        __syncthreads();
        acc = csr_group_sum<L>(first, val, col, pairs, len, t, lane, xs);
    } else {
        acc = csr_group_sum<L>(first, val, col, pairs, len, t, lane, src);
    }
    acc = group_sum<L>(acc);
    if (out) *yp = yo + acc;
}

// Blocks of rows by themselves: an adaptive layout without groups, or one
// column slice of the column-sliced CSR, where all x reads of a launch fall in
// one slice of columns, small enough to stay in L2 while the entry streams
// pass through with nontemporal loads.
__global__ __launch_bounds__(256) void csr_blocks_kernel(const unsigned char* __restrict__ counts,
                                                         const int* __restrict__ col, const float* __restrict__ val,
                                                         const int4* __restrict__ blocks, int nblocks,
                                                         const float* __restrict__ x, float* __restrict__ y,
                                                         double* __restrict__ carry) {
    __shared__ float lds[4][kCsrStreamMaxNnz];
    const int wid = threadIdx.x >> 6;
    const int b = blockIdx.x * 4 + wid;
    if (b >= nblocks) return;
    csr_block(blocks[b], counts, col, val, x, y, carry, lds[wid], threadIdx.x & 63);
}

__global__ __launch_bounds__(256) void csr_long_finalize_kernel(const int* __restrict__ long_rows,
                                                                const int* __restrict__ long_first,
                                                                const double* __restrict__ carry, int n_long,
                                                                float* __restrict__ y) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n_long) return;
    double s = 0.0;
    for (int k = long_first[i]; k < long_first[i + 1]; ++k) s += carry[k];
    const int r = long_rows[i];
    y[r] = (float)((double)y[r] + s);
}

}  // namespace dev

int launch_csr_scalar(const DevCsr& m, const float* x, float* y, hipStream_t st) {
    if (m.rows == 0) return 0;
    hipLaunchKernelGGL(dev::csr_scalar_kernel, dim3((m.rows + 255) / 256), dim3(256), 0, st, m.row_ptr, m.col, m.val,
                       x, y, m.rows);
    return (int)hipGetLastError();
}

int launch_csr_vector(const DevCsr& m, int lanes, const float* x, float* y, hipStream_t st) {
    if (m.rows == 0) return 0;
    const long long threads = (long long)m.rows * lanes;
    dim3 grid((unsigned)((threads + 255) / 256));
    switch (lanes) {
#define CASE(L)                                                                                                     \
    case L:                                                                                                         \
        hipLaunchKernelGGL(dev::csr_vector_kernel<L>, grid, dim3(256), 0, st, m.row_ptr, m.col, m.val, x, y, m.rows); \
        break;
        CASE(2) CASE(4) CASE(8) CASE(16) CASE(32) CASE(64)
#undef CASE
        default:
            return (int)hipErrorInvalidValue;
    }
    return (int)hipGetLastError();
}

template <int L>
static void csr_adaptive_launch(const DevCsrAdaptive& m, const float* x, float* y, hipStream_t st) {
    const int per_wg = std::min(kCsrWaves, std::max(1, m.nblocks / 256));
    const int nblock_wg = (m.nblocks + per_wg - 1) / per_wg;
    hipLaunchKernelGGL(dev::csr_adaptive_kernel<L>, dim3(nblock_wg + m.ngroups), dim3(kCsrThreads),
                       (size_t)m.lds_floats * 4, st, m, nblock_wg, per_wg, x, y);
}

int launch_csr_adaptive(const DevCsrAdaptive& m, const float* x, float* y, hipStream_t st) {
    if (m.ngroups == 0 && m.nblocks > 0) {
        hipLaunchKernelGGL(dev::csr_blocks_kernel, dim3((m.nblocks + 3) / 4), dim3(256), 0, st, m.counts, m.col, m.val,
                           m.blocks, m.nblocks, x, y, m.carry);
        int e = (int)hipGetLastError();
        if (e) return e;
    } else if (m.ngroups > 0) {
        switch (m.lanes) {
            case 1: csr_adaptive_launch<1>(m, x, y, st); break;
            case 2: csr_adaptive_launch<2>(m, x, y, st); break;
            case 4: csr_adaptive_launch<4>(m, x, y, st); break;
            case 8: csr_adaptive_launch<8>(m, x, y, st); break;
            case 16: csr_adaptive_launch<16>(m, x, y, st); break;
            default: return (int)hipErrorInvalidValue;
        }
        int e = (int)hipGetLastError();
        if (e) return e;
    }
    if (m.n_long > 0) {
        hipLaunchKernelGGL(dev::csr_long_finalize_kernel, dim3((m.n_long + 255) / 256), dim3(256), 0, st, m.long_rows,
                           m.long_first, m.carry, m.n_long, y);
    }
    return (int)hipGetLastError();
}

int launch_csr_sliced(const DevCsrSliced& m, const float* x, float* y, hipStream_t st) {
    for (int s = 0; s < m.nslices; ++s) {
        const int b0 = m.slice_block_begin[s], nb = m.slice_block_begin[s + 1] - b0;
        if (nb == 0) continue;
        hipLaunchKernelGGL(dev::csr_blocks_kernel, dim3((nb + 3) / 4), dim3(256), 0, st, m.counts + (size_t)s * m.rows,
                           m.col, m.val, m.blocks + b0, nb, x, y, m.carry);
        int e = (int)hipGetLastError();
        if (e) return e;
    }
    if (m.n_long > 0) {
        hipLaunchKernelGGL(dev::csr_long_finalize_kernel, dim3((m.n_long + 255) / 256), dim3(256), 0, st, m.long_rows,
                           m.long_first, m.carry, m.n_long, y);
    }
    return (int)hipGetLastError();
}

}  // namespace clspmv
