// COO SpMV (y += A*x) as a segmented reduction over the row-sorted entries.
//
// The reference splits the entries into per-workgroup ranges, runs an LDS
// segmented scan with a barrier per step and folds the per-group carries in a
// second one-workgroup kernel (A/kernels/spmv_coo.cl:4-200).  Here one
// wavefront owns a 512-entry chunk and each lane four consecutive entries of
// each half of it, one dwordx4 per array and half (a wave's load is 1 KiB side
// by side):
//   1. each lane sums its entries since its last row break, and a segmented
//      scan in DPP moves carries these tails into the next lanes;
//   2. every break ends a segment: its sum and row go to the wave's LDS at
//      the break's ordinal in the chunk (ballots count the breaks before a
//      lane), and the wave then adds them to y 64 at a time -- consecutive
//      rows, one read-modify-write round trip instead of one per break;
//   3. a row that continues into the next chunk for at most kCooReach
//      entries is finished here from those entries (loaded with the chunk's
//      own) and left out there; a longer one goes to the chunks' carry
//      slots in FP64, which coo_carry_kernel adds in order.  Where no row
//      reaches that far (known at upload), that kernel is not launched.
// No atomics; results are deterministic.  The last chunk is padded with
// (last row, last col, 0.0) as it is loaded, as the reference pads to 32.
#include "kcommon.hpp"
#include "launch.hpp"

namespace clspmv {
namespace dev {

// Bound by HBM (12 bytes per entry), and without the staging by one L1 line
// per gathered x.  A workgroup's chunks share one x range: when it spans at
// most coo_window columns it is staged in LDS (before the segments' sums,
// which reuse the space), else x is read from memory.
// Measured (us; before: eight consecutive entries per lane, so that each
// load touched half of every line twice, breaks written to y from inside the
// lanes, two carries per chunk always): 500,009 rows of 6..18 entries near
// the diagonal 26.8 -> 18.5 (3.9 TB/s); 1M rows of 9..27 68 -> 42; 40^3
// stencil 11.9 -> 6.0; 8000 rows 6.6 -> 4.5 (the second launch).  Plain
// loads: with the nontemporal hint the same kernel took 48 instead of 42.
template <int T>
__global__ __launch_bounds__(T) void coo_segment_kernel(
    const int* __restrict__ rowi, const int* __restrict__ coli, const float* __restrict__ vali, int nnz, int chunks,
    const float* __restrict__ x, float* __restrict__ y, int* __restrict__ carry_row, double* __restrict__ carry_val) {
    constexpr int kWaves = T / 64, kWindow = coo_window(T);
    __shared__ __align__(16) float shared[kWindow];  // the x range, then the segments' sums
    __shared__ int rows_of[kWaves][kCooChunk];
    __shared__ int range[2][kWaves];
    static_assert(T * kCooPerLane <= kWindow, "the sums fit the x range's space");
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    float* seg_sum = shared + wave * kCooChunk;
    int* seg_row = rows_of[wave];
    const int chunk = blockIdx.x * kWaves + wave;
    const bool live = chunk < chunks;  // the others only take part in the barriers
    // nnz is an int: first + kCooChunk + kCooReach may pass it, in 64 bits
    const int first = live ? chunk * kCooChunk : 0;
    const int last = nnz - 1;
    // lane's entries: half h of the chunk, four from h * 256 + 4 lane
    int r[8], c[8];
    float v[8];
    int lo = INT32_MAX, hi = 0;
    if (live) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const long long k = (long long)first + h * (kCooChunk / 2) + lane * 4;
            int4 rq, cq;
            float4 vq;
            if (k + 4 <= nnz) {
                cq = *reinterpret_cast<const int4*>(coli + k);
                rq = *reinterpret_cast<const int4*>(rowi + k);
                vq = *reinterpret_cast<const float4*>(vali + k);
            } else {
                // past the end: (last row, last col, 0.0)
                const int lr = rowi[last], lc = coli[last], left = (int)(nnz - k);
                rq = make_int4(left > 0 ? rowi[k] : lr, left > 1 ? rowi[k + 1] : lr, left > 2 ? rowi[k + 2] : lr, lr);
                cq = make_int4(left > 0 ? coli[k] : lc, left > 1 ? coli[k + 1] : lc, left > 2 ? coli[k + 2] : lc, lc);
                vq = make_float4(left > 0 ? vali[k] : 0.f, left > 1 ? vali[k + 1] : 0.f, left > 2 ? vali[k + 2] : 0.f,
                                 0.f);
            }
            r[4 * h] = rq.x; r[4 * h + 1] = rq.y; r[4 * h + 2] = rq.z; r[4 * h + 3] = rq.w;
            c[4 * h] = cq.x; c[4 * h + 1] = cq.y; c[4 * h + 2] = cq.z; c[4 * h + 3] = cq.w;
            v[4 * h] = vq.x; v[4 * h + 1] = vq.y; v[4 * h + 2] = vq.z; v[4 * h + 3] = vq.w;
        }
    }
    // the next chunk's first kCooReach entries, one per lane (past the end:
    // row -1), the row after them, and the rows around this chunk's start
    const long long next = (long long)first + kCooChunk + lane;
    const int wk = (int)min(next, (long long)last);
    const int wr = next <= last ? rowi[wk] : -1;
    const int wc = coli[wk];
    const float wv = vali[wk];
    auto row_at = [&](long long k) { return k <= last ? rowi[k] : -1; };  // wave-uniform
    const int after_next = row_at((long long)first + kCooChunk + kCooReach);
    const int after_first = row_at((long long)first + kCooReach);
    const int before = first > 0 ? rowi[first - 1] : -1;

    // the columns the workgroup's chunks span; and
    // 1. row breaks: entry i's row differs from the entry before it (the
    //    chunk's first entry is none).  Each ends a segment; the ballots
    //    give its ordinal in the chunk.
    bool brk[8] = {false, false, false, false, false, false, false, false};
    int ordinal[2] = {0, 0}, segs = 0, half_segs = 0;
    int row0 = -1;
    float y0 = 0.f, y_last = 0.f, wp = 0.f;
    if (live) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            lo = min(lo, c[i]);
            hi = max(hi, c[i]);
        }
        lo = wave_min(lo);
        hi = -wave_min(-hi);
        const int middle = __builtin_amdgcn_readlane(r[3], 63);
        const int prev0 = lane_up1(r[3]), up = lane_up1(r[7]);
        const int prev1 = lane > 0 ? up : middle;
        brk[0] = lane > 0 && prev0 != r[0];
        brk[4] = prev1 != r[4];
#pragma unroll
        for (int i = 1; i < 8; ++i)
            if (i != 4) brk[i] = r[i] != r[i - 1];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            half_segs = segs;
            ordinal[h] = segs;
#pragma unroll
            for (int i = 4 * h; i < 4 * h + 4; ++i) {
                const unsigned long long m = __ballot(brk[i]);
                ordinal[h] = __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32),
                                                       __builtin_amdgcn_mbcnt_lo((unsigned)m, ordinal[h]));
                segs += __popcll(m);
            }
            int at = ordinal[h];
#pragma unroll
            for (int i = 4 * h; i < 4 * h + 4; ++i)
                if (brk[i]) seg_row[at++] = i == 0 ? prev0 : i == 4 ? prev1 : r[i - 1];
        }
        wave_lds_sync();
        if (lane < segs) {
            row0 = seg_row[lane];
            y0 = y[row0];  // in flight while x is staged
        }
        const int last_row = __builtin_amdgcn_readlane(r[7], 63);
        y_last = y[last_row];
        if (wr == last_row) wp = wv * x[wc];
    }
    if (lane == 0) {
        range[0][wave] = lo;
        range[1][wave] = hi;
    }
    __syncthreads();
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
        lo = min(lo, range[0][w]);
        hi = max(hi, range[1][w]);
    }
    lo &= ~3;
    const int span = hi - lo + 1;
    float xv[8];
    if (span <= kWindow) {  // the same for the whole workgroup
        for (int i = threadIdx.x * 4; i < span; i += T * 4) {
            if (i + 4 <= span) {
                const f32x4a4 q = *reinterpret_cast<const f32x4a4*>(x + lo + i);
                *reinterpret_cast<float4*>(shared + i) = make_float4(q.x, q.y, q.z, q.w);
            } else {
#pragma unroll
                for (int j = 0; j < 3; ++j)
                    if (i + j < span) shared[i + j] = x[lo + i + j];
            }
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 8; ++i) xv[i] = live ? shared[c[i] - lo] : 0.f;
        __syncthreads();
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) xv[i] = live ? x[c[i]] : 0.f;
    }
    if (!live) return;

    // 2. lane tails (sums since the lane's last break in the half) and their
    //    segmented scans; the second half's leading run takes the first's
    //    last tail.
    float tail[2];
    int any[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        tail[h] = 0.f;
        any[h] = lane == 0;
#pragma unroll
        for (int i = 4 * h; i < 4 * h + 4; ++i) {
            tail[h] = fmaf(v[i], xv[i], brk[i] ? 0.f : tail[h]);
            any[h] |= brk[i];
        }
    }
    const int rl = lane & 15;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        float t = tail[h];
        int f = any[h];
        seg_step(rl >= 1, dpp_f<0x111, 0xf>(t), dpp_i<0x111, 0xf>(f), t, f);
        seg_step(rl >= 2, dpp_f<0x112, 0xf>(t), dpp_i<0x112, 0xf>(f), t, f);
        seg_step(rl >= 4, dpp_f<0x114, 0xf>(t), dpp_i<0x114, 0xf>(f), t, f);
        seg_step(rl >= 8, dpp_f<0x118, 0xf>(t), dpp_i<0x118, 0xf>(f), t, f);
        seg_step((lane & 16) != 0, dpp_f<0x142, 0xa>(t), dpp_i<0x142, 0xa>(f), t, f);
        seg_step(lane >= 32, dpp_f<0x143, 0xc>(t), dpp_i<0x143, 0xc>(f), t, f);
        tail[h] = t;
    }
    const float middle_sum = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(tail[0]), 63));
    // no break of the second half up to this lane's last entry
    const bool open = ordinal[1] + brk[4] + brk[5] + brk[6] + brk[7] == half_segs;
    if (open) tail[1] += middle_sum;
    const float carried0 = lane_up1(tail[0]), carried1 = lane_up1(tail[1]);
    // each segment: the lane's own entries summed first, then what is carried
    // into the lane's first one
    float acc = 0.f, in = lane > 0 ? carried0 : 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        if (i == 4) {
            acc = 0.f;
            in = lane > 0 ? carried1 : middle_sum;
        }
        if (brk[i]) seg_sum[ordinal[i / 4]++] = acc + in;
        in = brk[i] ? 0.f : in;
        acc = fmaf(v[i], xv[i], brk[i] ? 0.f : acc);
    }
    const int first_row = __builtin_amdgcn_readfirstlane(r[0]);
    const int last_row = __builtin_amdgcn_readlane(r[7], 63);
    const float last_sum = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(tail[1]), 63));
    // 3. the first row, when it comes from the previous chunk: finished there
    //    (drop) or a carry; the last row, when it goes on: finished here from
    //    the window or a carry.
    const bool from_prev = before == first_row;
    const bool drop = from_prev && after_first != first_row;
    const bool first_carry = from_prev && !drop;
    const bool goes_on = __builtin_amdgcn_readfirstlane(wr) == last_row;
    const bool reach = goes_on && after_next != last_row;
    double tail_sum = (double)last_sum;
    if (reach) tail_sum += (double)wave_total(wp);
    wave_lds_sync();
    if (row0 >= 0 && !(lane == 0 && from_prev)) y[row0] = y0 + seg_sum[lane];
    for (int k = lane + 64; k < segs; k += 64) y[seg_row[k]] += seg_sum[k];
    const bool one_row = segs == 0;
    const bool last_carry = (goes_on && !reach) || (one_row && first_carry);
    if (lane == 0) {
        if (!last_carry && !(one_row && drop)) {
            y[last_row] = reach ? (float)((double)y_last + tail_sum) : y_last + last_sum;
        }
        if (carry_row) {
            carry_row[2 * chunk] = first_carry ? first_row : -1;
            carry_row[2 * chunk + 1] = last_carry ? last_row : -1;
            if (first_carry) carry_val[2 * chunk] = one_row ? 0.0 : (double)seg_sum[0];
            if (last_carry) carry_val[2 * chunk + 1] = tail_sum;
        }
    }
}

// Each run of equal rows in the carry list (-1: no carry in the slot) is
// summed in FP64 by the lane that owns its first entry, eight slots per round
// of loads.
__global__ __launch_bounds__(256) void coo_carry_kernel(const int* __restrict__ carry_row,
                                                        const double* __restrict__ carry_val, int n,
                                                        float* __restrict__ y, int rows) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const int r = carry_row[i], before = i > 0 ? carry_row[i - 1] : -1;
    if (r < 0 || r >= rows || before == r) return;
    const float yo = y[r];
    double s = 0.0;
    bool more = true;
    for (int k = i; more; k += 8) {
        int rr[8];
        double v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int q = min(k + u, n - 1);
            rr[u] = carry_row[q];
            v[u] = carry_val[q];  // a slot without a carry holds an old sum: not used
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            more = more && k + u < n && rr[u] == r;
            s += more ? v[u] : 0.0;
        }
    }
    y[r] = (float)((double)yo + s);
}

}  // namespace dev

int launch_coo(const DevCoo& m, const float* x, float* y, hipStream_t st) {
    if (m.chunks == 0) return 0;
#define CLSPMV_COO(T)                                                                                              \
    hipLaunchKernelGGL(dev::coo_segment_kernel<T>, dim3((m.chunks + T / 64 - 1) / (T / 64)), dim3(T), 0, st, m.row, \
                       m.col, m.val, m.nnz, m.chunks, x, y, m.carry_row, m.carry_val)
    if (m.chunks <= kCooFewChunks)
        CLSPMV_COO(256);
    else
        CLSPMV_COO(512);
#undef CLSPMV_COO
    int e = (int)hipGetLastError();
    if (e || !m.carry_row) return e;
    const int n = 2 * m.chunks;
    hipLaunchKernelGGL(dev::coo_carry_kernel, dim3((n + 255) / 256), dim3(256), 0, st, m.carry_row, m.carry_val, n, y,
                       m.rows);
    return (int)hipGetLastError();
}

}  // namespace clspmv
