// Sliced ELL plans on the device: a wave per slice walks its 64 rows side by
// side.  Rows' columns ascend, so the distinct column offsets col - row of a
// slice come one after the other as the smallest that any lane has left: one
// walk tells whether the slice is a diagonal one, and how wide; a second one
// writes offsets, masks and sources.
//
// Planned by the host, the first solve on a newly bound mesh -- the first after
// every adapt -- took several times as long as the next.  First mixed CG solve
// to 1e-2, host's plan -> so: 642k rows of triangles 16.8 -> 3.7 ms, 1.37M of
// tetrahedra 71 -> 15 ms, 301k of an unstructured mesh 44 -> 4.9 ms.
#include <hip/hip_runtime.h>

#include <climits>
#include <vector>

#include "sell_plan.h"

namespace flgpu {

// The rows of each run by length, longest first, equal ones in order; -1 past
// the last row.  A block per kSellRun rows ranks them in their run.
__global__ void __launch_bounds__(kSellRun)
k_sell_sort(int n, int nrow, int run, const int32_t* __restrict__ rowptr, int32_t* __restrict__ rows) {
    __shared__ int len[kSellWindow];
    const int r = blockIdx.x * kSellRun + threadIdx.x, w0 = (int)blockIdx.x * kSellRun / run * run, m = min(run, n - w0);
    for (int q = threadIdx.x; q < m; q += kSellRun) len[q] = rowptr[w0 + q + 1] - rowptr[w0 + q];
    __syncthreads();
    if (r < n) {
        const int t = r - w0, l = len[t];
        int rank = 0;
        for (int q = 0; q < m; q++) rank += len[q] > l || (len[q] == l && q < t);
        rows[w0 + rank] = r;
    } else if (r < nrow) {
        rows[r] = -1;
    }
}

// A lane's row: the entry it is at, and that entry's offset (INT_MAX past the
// row's end).
struct SellLane {
    int row, e, end, cur;
    __device__ __forceinline__ SellLane(int n, int sl, int lane, const int32_t* rows, const int32_t* rowptr,
                                        const int32_t* col) {
        const int q = sl * kSlice + lane;
        row = rows ? rows[q] : q < n ? q : -1;
        e = row >= 0 ? rowptr[row] : 0;
        end = row >= 0 ? rowptr[row + 1] : 0;
        cur = e < end ? col[e] - row : INT_MAX;
    }
    __device__ __forceinline__ void next(const int32_t* col) {
        e++;
        cur = e < end ? col[e] - row : INT_MAX;
    }
};

__device__ __forceinline__ int sell_wave_min(int v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = min(v, __shfl_xor(v, off, 64));
    return v;
}

// The row that a slice's column indices count from.
__device__ __forceinline__ int sell_first(int sl, bool sorted) {
    return sorted ? sl / (kSellWindow / kSlice) * kSellWindow : sl * kSlice;
}

// width[sl] = 2 steps + 1 for a diagonal slice; *far becomes 1 when a column
// index of another slice (or its padding's, the row itself) is out of int16
// range.
__global__ void __launch_bounds__(256)
k_sell_widths(int n, int nsl, int diagonals, const int32_t* __restrict__ rows, const int32_t* __restrict__ rowptr,
              const int32_t* __restrict__ col, int32_t* __restrict__ width, int32_t* __restrict__ far) {
    const int sl = blockIdx.x * 4 + (int)(threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (sl >= nsl) return;
    SellLane t(n, sl, lane, rows, rowptr, col);
    const int e0 = t.e, w = -sell_wave_min(-(t.end - t.e)), most = w + w / 8;
    int steps = 0, m = INT_MAX;
    while (diagonals && (m = sell_wave_min(t.cur)) != INT_MAX && steps < most) {
        steps++;
        if (t.cur == m) t.next(col);
    }
    const bool dia = diagonals && m == INT_MAX;
    if (!dia) {
        const int r0 = sell_first(sl, rows != nullptr);
        bool out = t.row >= 0 && t.row - r0 > INT16_MAX;
        for (int e = e0; e < t.end; e++) out |= col[e] - r0 < INT16_MIN || col[e] - r0 > INT16_MAX;
        if (__ballot(out) && lane == 0) atomicOr(far, 1);
    }
    if (lane == 0) width[sl] = dia ? 2 * steps + 1 : 2 * w;
}

__global__ void __launch_bounds__(256)
k_sell_fill(int n, int nsl, const int32_t* __restrict__ rows, const int32_t* __restrict__ rowptr,
            const int32_t* __restrict__ col, const int32_t* __restrict__ vmap, const int32_t* __restrict__ sptr,
            int32_t* __restrict__ src, uint64_t* __restrict__ mask, int32_t* __restrict__ off,
            int16_t* __restrict__ col16, int32_t* __restrict__ col32) {
    const int sl = blockIdx.x * 4 + (int)(threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (sl >= nsl) return;
    const int b = sptr[sl], base = b & ~(kSlice - 1), w = (sptr[sl + 1] - base) / kSlice;
    const int r0 = sell_first(sl, rows != nullptr);
    SellLane t(n, sl, lane, rows, rowptr, col);
    for (int j = 0; j < w; j++) {
        const int slot = base + j * kSlice + lane;
        bool in = t.e < t.end;
        if (b & 1) {
            const int m = sell_wave_min(t.cur);
            in = in && t.cur == m;
            if (lane == 0) off[base / kSlice + j] = m;
        } else {
            const int cj = in ? t.cur + t.row : t.row >= 0 ? t.row : r0;
            if (col16) col16[slot] = (int16_t)(cj - r0);
            else col32[slot] = cj;
        }
        src[slot] = !in ? -1 : vmap ? vmap[t.e] : t.e;
        const uint64_t lanes = __ballot(in);
        if (lane == 0) mask[base / kSlice + j] = lanes;
        if (in) t.next(col);
    }
}

int sell_build(hipStream_t s, int n, int64_t nnz, const int32_t* rowptr, const int32_t* col, const int32_t* vmap,
               bool sorted, SellPlan& p) {
    p.release();
    const int nsl = (n + kSlice - 1) / kSlice;
    if (sorted) {
        FLGPU_TRY(p.rows.alloc((size_t)nsl * kSlice));
        hipLaunchKernelGGL(k_sell_sort, dim3((n + kSellRun - 1) / kSellRun), dim3(kSellRun), 0, s, n, nsl * kSlice,
                           sell_run(n), rowptr, p.rows.p);
    }
    DevBuf<int32_t> width;  // the slices', then the flag
    FLGPU_TRY(width.alloc((size_t)nsl + 1));
    FLGPU_HIP(hipMemsetAsync(width.p + nsl, 0, sizeof(int32_t), s));
    const dim3 grid((nsl + 3) / 4);
    // (the diagonal slices' extra steps keep within 32-bit slots)
    hipLaunchKernelGGL(k_sell_widths, grid, dim3(256), 0, s, n, nsl, nnz < 1 << 30 ? 1 : 0, p.rows.p, rowptr, col,
                       width.p, width.p + nsl);
    FLGPU_HIP(hipGetLastError());
    std::vector<int32_t> w((size_t)nsl + 1), sptr((size_t)nsl + 1);
    FLGPU_HIP(hipMemcpyAsync(w.data(), width.p, sizeof(int32_t) * w.size(), hipMemcpyDeviceToHost, s));
    FLGPU_HIP(hipStreamSynchronize(s));
    int64_t at = 0;
    bool dia = false, plain = false;
    for (int sl = 0; sl < nsl; sl++) {
        sptr[sl] = (int32_t)at | (w[sl] & 1);
        at += (int64_t)(w[sl] >> 1) * kSlice;
        (w[sl] & 1 ? dia : plain) = true;
        if (at > INT32_MAX - kSlice) {
            p.release();
            return FLGPU_OK;
        }
    }
    sptr[nsl] = (int32_t)at;
    p.use16 = !w[nsl];
    p.nslot = at;
    const size_t steps = (size_t)at / kSlice + kSellAhead;
    FLGPU_TRY(p.sptr.upload(sptr.data(), sptr.size(), s));
    FLGPU_TRY(p.src.alloc((size_t)at));
    FLGPU_TRY(p.mask.alloc(steps));
    if (dia) FLGPU_TRY(p.off.alloc(steps));
    if (plain && p.use16) FLGPU_TRY(p.col16.alloc((size_t)at));
    if (plain && !p.use16) FLGPU_TRY(p.col32.alloc((size_t)at));
    hipLaunchKernelGGL(k_sell_fill, grid, dim3(256), 0, s, n, nsl, p.rows.p, rowptr, col, vmap, p.sptr.p, p.src.p,
                       p.mask.p, p.off.p, p.col16.p, p.col32.p);
    FLGPU_HIP(hipGetLastError());
    FLGPU_HIP(hipStreamSynchronize(s));  // sptr is freed on return
    p.nsl = nsl;
    return FLGPU_OK;
}

}  // namespace flgpu
