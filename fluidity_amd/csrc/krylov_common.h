// Device helpers shared by the Krylov and learned-preconditioner kernels:
// deterministic block reductions and CSR products.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <cstdlib>
#include <vector>

namespace flgpu {

enum {
    KSP_CONVERGED_RTOL = 2,
    KSP_CONVERGED_ATOL = 3,
    KSP_DIVERGED_ITS = -3,
    KSP_DIVERGED_DTOL = -4,
    KSP_DIVERGED_INDEFINITE_PC = -8,
    KSP_DIVERGED_NANORINF = -9,
    KSP_DIVERGED_INDEFINITE_MAT = -10
};

// Solver scalars, device resident.
struct Scal {
    double rz, rz_old, pAp, alpha, beta;
    double rr, zz, zw;
    double rnorm0, last_norm, true_rr, bb;
    double pivot, dmin, dmax;
    int32_t its, reason, done, max_its;
    double rtol, atol;
    int32_t norm_type, flexible, pad0, pad1;
};

constexpr int kVecBlock = 1024;    // threads per block of the vector kernels (16 waves)
constexpr int kMaxVecGrid = 256;   // their fixed grid: one block per CU, so that a consumer has few
                                   // partial sums to add
constexpr int kRowBlock = 256;     // threads per block of the CSR row products
constexpr int kMaxRowGrid = 2048;  // their fixed grid
constexpr int kPartStride = 2048;  // partials[k * kPartStride + block], >= either grid

// Regions of the partial-sum buffer (in units of kPartStride).  A producer
// kernel writes one per-block value per component; the consumer sums them.
enum {
    PART_SPMV = 0,  // 2 components: x.y, y.y of the CSR product
    PART_VEC = 2,   // 4 components: r.z, r.r, z.z, z.w of the CG update
    PART_PC = 6,    // 3 components: r.z, z.z, z.w of the learned apply
    PART_MISC = 9,  // 2 components: b.b, diagonal min/max
    PART_VEC2 = 11, // 4 components: the single-reduction CG's update, alternating with PART_VEC
    PART_COMPONENTS = 15
};

// Sum over the wave by DPP moves (8-cycle steps instead of LDS shuffles, in
// a fixed order), in every lane.
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_add(double v) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, ROWS, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, ROWS, 0xf, true);
    return v + __hiloint2double(hi, lo);
}
__device__ __forceinline__ double wave_total(double v) {
    v = dpp_add<0x111, 0xf>(v);  // row_shr 1, 2, 4, 8: the last lane of each 16 has their sum
    v = dpp_add<0x112, 0xf>(v);
    v = dpp_add<0x114, 0xf>(v);
    v = dpp_add<0x118, 0xf>(v);
    v = dpp_add<0x142, 0xa>(v);  // row_bcast 15 into rows 1 and 3, row_bcast 31 into rows 2 and 3
    v = dpp_add<0x143, 0xc>(v);
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), 63),
                            __builtin_amdgcn_readlane(__double2loint(v), 63));
}

// Sum over a block in a fixed order; result valid in thread 0.
template <int NV>
__device__ __forceinline__ void block_sum(double (&v)[NV], double (*sh)[NV]) {
#pragma unroll
    for (int k = 0; k < NV; k++) v[k] = wave_total(v[k]);
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (lane == 0)
#pragma unroll
        for (int k = 0; k < NV; k++) sh[wave][k] = v[k];
    __syncthreads();
    if (threadIdx.x == 0) {
        const int nw = blockDim.x >> 6;
#pragma unroll
        for (int k = 0; k < NV; k++) {
            double s = sh[0][k];
            for (int q = 1; q < nw; q++) s += sh[q][k];
            v[k] = s;
        }
    }
    __syncthreads();
}

// Per-block sums of NV values: thread 0 of each block stores them at
// partials[k * kPartStride + blockIdx.x].
template <int NV>
__device__ __forceinline__ void block_partials(double (&v)[NV], double* __restrict__ partials) {
    __shared__ double sh[kVecBlock / 64][NV];
    block_sum<NV>(v, sh);
    if (threadIdx.x == 0)
#pragma unroll
        for (int k = 0; k < NV; k++) partials[(size_t)k * kPartStride + blockIdx.x] = v[k];
}

// Totals of the nparts per-block sums of NV components, in every thread of a
// kVecBlock block: each wave takes 64 of a component's sums at a time, so up
// to kVecBlock / NV sums are one load, and the waves' totals are added in
// order.  The same sums in every block.
template <int NV>
__device__ __forceinline__ void part_totals(const double* __restrict__ partials, int nparts, double (&out)[NV]) {
    constexpr int G = kVecBlock / 64 / NV;  // waves per component
    __shared__ double sh[NV][G];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (wave < G * NV) {
        const int c = wave / G, g = wave % G;
        double t = 0.0;
#pragma unroll 4
        for (int b = g * 64 + lane; b < nparts; b += 64 * G) t += partials[(size_t)c * kPartStride + b];
        t = wave_total(t);
        if (lane == 0) sh[c][g] = t;
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < NV; c++) {
        out[c] = sh[c][0];
#pragma unroll
        for (int g = 1; g < G; g++) out[c] += sh[c][g];
    }
}

// Total of the nparts per-block sums a previous kernel wrote.  Every block
// that calls it forms the same sum in the same order (thread t adds parts
// t, t + blockDim, ..., then the fixed block order), so all blocks agree
// bit for bit and no grid-wide atomics or last-block election are needed.
// Result valid in thread 0.
template <int NV>
__device__ __forceinline__ void sum_partials(const double* __restrict__ partials, int nparts,
                                             double (&out)[NV]) {
    __shared__ double sh[kVecBlock / 64][NV];
#pragma unroll
    for (int k = 0; k < NV; k++) out[k] = 0.0;
    for (int b = threadIdx.x; b < nparts; b += blockDim.x)
#pragma unroll
        for (int k = 0; k < NV; k++) out[k] += partials[(size_t)k * kPartStride + b];
    block_sum<NV>(out, sh);
}

// ---------------------------------------------------------------------
// Streamed CSR products
// ---------------------------------------------------------------------
constexpr int kStreamPerThread = 8;
constexpr int kStreamNnz = kRowBlock * kStreamPerThread;  // entries staged per row block

// Row blocks for k_csr_stream: runs of consecutive rows holding at most
// kStreamNnz entries and at most kRowBlock rows; a longer row is a block of
// its own.  rb has nblocks + 1 entries, rbk the matching first entries.
inline void stream_row_blocks(const int32_t* rowptr, int n, std::vector<int32_t>& rb,
                              std::vector<int32_t>& rbk) {
    rb.clear();
    rb.push_back(0);
    int r = 0;
    while (r < n) {
        const int k0 = rowptr[r];
        int r1 = r;
        while (r1 < n && r1 - r < kRowBlock && rowptr[r1 + 1] - k0 <= kStreamNnz) r1++;
        if (r1 == r) r1 = r + 1;
        rb.push_back(r1);
        r = r1;
    }
    rbk.resize(rb.size());
    for (size_t q = 0; q < rb.size(); q++) rbk[q] = rowptr[rb[q]];
}

enum { DOT_NONE = 0, DOT_XY = 1, DOT_PC = 2 };

// Row blocks handled by this workgroup: with a grid that is a multiple of 8
// each XCD (the hardware hands consecutive workgroups to the 8 XCDs in
// turn) takes a contiguous share of the row blocks, so the vector entries
// and nodes that neighbouring rows gather stay in one L2.
struct RowBlocks {
    int b, hi, step;
    __device__ __forceinline__ explicit RowBlocks(int nrb) : RowBlocks(nrb, blockIdx.x, gridDim.x) {}
    // as workgroup `wg` of the first `n` of the grid
    __device__ __forceinline__ RowBlocks(int nrb, int wg, int n) {
        b = wg;
        hi = nrb;
        step = n;
        if ((n & 7) == 0) {
            const int xcd = wg & 7;
            b = (int)((int64_t)nrb * xcd / 8) + (wg >> 3);
            hi = (int)((int64_t)nrb * (xcd + 1) / 8);
            step = n >> 3;
        }
    }
};

// A CSR operand of k_csr_stream.  Column indices are either int32 or, when
// every entry of a row block lies within int16 range of the block's first
// row, int16 offsets from that row (half the index bytes).  Optional
// scales: y_i = rs_i * sum_k val_k (cs_j x_j) -- a diagonally scaled matrix
// stored unscaled (low-precision values of order one).
template <typename AV, typename CT>
struct CsrOp {
    int nrb;
    const int32_t* rb;     // nrb+1 first rows of the row blocks
    const int32_t* rbk;    // nrb+1 first entries of the row blocks (rowptr[rb[b]])
    const int32_t* rowptr;
    const CT* col;
    const AV* val;
    const float* cs;
    const float* rs;
};

template <typename CT>
__device__ __forceinline__ int csr_col(const CT* __restrict__ col, int k, int r0) {
    if constexpr (sizeof(CT) == 2)
        return r0 + (int)col[k];
    else
        return (int)col[k];
}

// y = A x (or y = bsub - A x) over row blocks.  A block reads its entries
// once, coalesced, stages the products val*x[col] in LDS and one thread per
// row adds them in entry order: the sequential row sum of a plain CSR
// product, with the product rounded before the addition.  A fixed grid
// walks the row blocks (RowBlocks).
// Per-block dot products into partials: DOT_XY: x_i y_i, y_i^2;
// DOT_PC: r_i y_i, y_i^2, y_i w_i.
template <typename V, typename AV, typename CT, typename XV, typename YV, int DOTS>
__global__ void __launch_bounds__(kRowBlock)
k_csr_stream(CsrOp<AV, CT> m, const XV* __restrict__ x, YV* __restrict__ y, const double* __restrict__ bsub,
             const V* __restrict__ dr, const V* __restrict__ dw, double* __restrict__ partials,
             const int* __restrict__ done_flag) {
    if (done_flag && *done_flag) return;
    __shared__ V prod[kStreamNnz];
    double d0 = 0.0, d1 = 0.0, d2 = 0.0;
    const int32_t* __restrict__ rowptr = m.rowptr;
    const CT* __restrict__ col = m.col;
    const AV* __restrict__ val = m.val;
    const float* __restrict__ cs = m.cs;
    const RowBlocks it(m.nrb);
    // The bounds and column indices of the next row block are loaded while
    // the current block's values and x entries are gathered, so a row block
    // costs one round trip to memory instead of three.
    int r0 = 0, r1 = 0, k0 = 0, k1 = 0, c[kStreamPerThread];
    auto fetch = [&](int bb, int& a0, int& a1, int& e0, int& e1, int (&cc)[kStreamPerThread]) {
        a0 = m.rb[bb];
        a1 = m.rb[bb + 1];
        e0 = m.rbk[bb];
        e1 = m.rbk[bb + 1];
#pragma unroll
        for (int j = 0; j < kStreamPerThread; j++) {
            const int k = e0 + (int)threadIdx.x + j * kRowBlock;
            cc[j] = (k < e1 && e1 - e0 <= kStreamNnz) ? csr_col(col, k, a0) : 0;
        }
    };
    if (it.b < it.hi) fetch(it.b, r0, r1, k0, k1, c);
    for (int b = it.b; b < it.hi; b += it.step) {
        int n0 = 0, n1 = 0, e0 = 0, e1 = 0, nc[kStreamPerThread];
        if (b + it.step < it.hi) fetch(b + it.step, n0, n1, e0, e1, nc);
        const int row = r0 + threadIdx.x;
        V acc = (V)0;
        if (k1 - k0 <= kStreamNnz) {
            int kb = 0, ke = 0;
            if (row < r1) {
                kb = rowptr[row] - k0;
                ke = rowptr[row + 1] - k0;
            }
            V pv[kStreamPerThread];
#pragma unroll
            for (int j = 0; j < kStreamPerThread; j++) {
                const int k = k0 + (int)threadIdx.x + j * kRowBlock;
                pv[j] = (V)0;
                if (k < k1) {
                    V xv = (V)x[c[j]];
                    if (cs) xv = xv * (V)cs[c[j]];
                    pv[j] = (V)val[k] * xv;
                }
            }
#pragma unroll
            for (int j = 0; j < kStreamPerThread; j++) {
                const int k = k0 + (int)threadIdx.x + j * kRowBlock;
                if (k < k1) prod[k - k0] = pv[j];
            }
            __syncthreads();
            for (int k = kb; k < ke; k++) acc += prod[k];
            __syncthreads();
        } else {  // one row longer than the staging buffer: in order, chunk by chunk
            for (int c0 = k0; c0 < k1; c0 += kStreamNnz) {
                const int c1 = min(k1, c0 + kStreamNnz);
                for (int k = c0 + threadIdx.x; k < c1; k += kRowBlock) {
                    const int cj = csr_col(col, k, r0);
                    V xv = (V)x[cj];
                    if (cs) xv = xv * (V)cs[cj];
                    prod[k - c0] = (V)val[k] * xv;
                }
                __syncthreads();
                if (threadIdx.x == 0)
                    for (int k = 0; k < c1 - c0; k++) acc += prod[k];
                __syncthreads();
            }
        }
        if (row < r1) {
            if (m.rs) acc = acc * (V)m.rs[row];
            double yv = (double)acc;
            if (bsub) yv = bsub[row] - yv;
            const YV yo = (YV)yv;
            y[row] = yo;
            if (DOTS == DOT_XY) {
                d0 += (double)x[row] * yv;
                d1 += yv * yv;
            } else if (DOTS == DOT_PC) {
                const double z = (double)yo;
                d0 += (double)dr[row] * z;
                d1 += z * z;
                d2 += z * (double)dw[row];
            }
        }
        r0 = n0;
        r1 = n1;
        k0 = e0;
        k1 = e1;
#pragma unroll
        for (int j = 0; j < kStreamPerThread; j++) c[j] = nc[j];
    }
    if (DOTS == DOT_XY) {
        double v[2] = {d0, d1};
        block_partials<2>(v, partials);
    } else if (DOTS == DOT_PC) {
        double v[3] = {d0, d1, d2};
        block_partials<3>(v, partials);
    }
}

// ---------------------------------------------------------------------
// Sliced ELL products
// ---------------------------------------------------------------------
// A slice is 64 consecutive rows, one wave: entry j of the slice's rows
// sits at slots sptr[s] + 64 j + lane, so every load of values and column
// offsets is one contiguous line per wave, with no row bounds, no LDS and
// no barrier.  A slice is as wide as its longest row; the slots past a
// row's end are padding (value 0, column the row itself) and are skipped.
// Meshes numbered in space-filling order give slices of near-equal rows, so
// the padding is small.  Where rows of different length alternate (quadratic
// elements, unstructured meshes) the rows are first sorted by length within
// runs (sell_run), equal ones in order: the slice then lists its rows, and
// column indices count from the first row of its window of kSellWindow rows.
// sell_order says which form a matrix takes, if any.
//
// A slice keeps a 64-bit lane mask per step, the rows that have an entry
// there.
//
// Diagonal slices.  Where nodes are numbered regularly (structured and
// extruded meshes) the rows of a slice share their column offsets col - row.
// A slice whose rows have at most 1/8 more distinct offsets than its longest
// row has entries keeps one offset per step instead of 64 column indices: 98
// of 100 slices of linear lattices, 27 to 62 of quadratic ones sorted by
// length.  Its x addresses come from scalar loads, so the x loads leave with
// the values' (one dependent memory round trip less) and read contiguous
// lines; 2 of 6 (FP32), 4 (FP16) or 10 (FP64) bytes an entry are not read at
// all.  A row's entries stay in order: the same sums.
// Against column indices: 1.37M rows FP64 33.6 -> 27.9 us, FP32 20.3 -> 18.1
// us, a factor's FP16 halves 13.5 and 15.8 -> 10.5 and 12.6 us (of which the
// masks in place of row lengths made 1 us); 275k rows FP64 10.7 -> 7.7 us.
// 1/8 more steps cost at most 1 byte an entry (FP64), half of what its index
// takes.  Slices of unstructured numberings find no shared offsets and keep
// their indices.
// Slower: 12 or 16 steps in flight (8 here), values loaded past the caches
// (28 -> 41 us), the next slice's bounds fetched early (no gain).
constexpr int kSlice = 64;
constexpr int kSellWindow = 2048;
constexpr int kSellRun = 256;
constexpr int kSellAhead = 8;  // masks and offsets read past the last slice's

template <typename AV, typename CT>
struct SellOp {
    int nsl, n;             // slices, rows
    const int32_t* sptr;    // nsl+1 first slots (multiples of 64), + 1 on a diagonal slice's
    const CT* col;          // per slot of the other slices
    const AV* val;          // per slot
    const float* rs;        // optional row scale: y_i = rs_i (A x)_i
    const int32_t* rows;    // rows of the slices when sorted (-1 past the last), or null: in order
    const int32_t* off;     // per 64 slots of a diagonal slice: col - row
    const uint64_t* mask;   // per 64 slots: the lanes whose row has an entry there
};

// The row of a lane of slice sl (n past the last) and the row its column
// indices count from.
template <typename AV, typename CT>
__device__ __forceinline__ int sell_row(const SellOp<AV, CT>& m, int sl, int lane, int& r0) {
    if (!m.rows) {
        r0 = sl * kSlice;
        return min(r0 + lane, m.n);
    }
    const int row = m.rows[sl * kSlice + lane];
    r0 = sl / (kSellWindow / kSlice) * kSellWindow;
    return row < 0 ? m.n : row;
}

// What a wave knows of its slice (sl the same in every lane).
struct SellSlice {
    int row, r0, base, w;
    bool dia;
};

template <typename AV, typename CT>
__device__ __forceinline__ SellSlice sell_slice(const SellOp<AV, CT>& m, int sl, int lane) {
    SellSlice s;
    const int b = m.sptr[sl];
    s.base = b & ~(kSlice - 1);
    s.dia = b & 1;
    s.w = (m.sptr[sl + 1] - s.base) / kSlice;
    s.row = sell_row(m, sl, lane, s.r0);
    return s;
}

// What a product takes of x: the values as they are, or (GMRES) scaled ones,
// the scale formed by begin() while the first step's loads are in flight.
struct SellX {
    __device__ __forceinline__ void begin() {}
    template <typename V>
    __device__ __forceinline__ V operator()(V v) const {
        return v;
    }
};

// The lane's row sum: its products in entry order, each rounded before the
// addition (no contraction), the same sums as k_csr_stream.  Every load is
// unconditional (a step past the slice's width re-reads its last slot,
// padding holds an in-range column), so the U loads of a step are all in
// flight together; only the additions are predicated.
template <typename V, typename AV, typename CT, typename XV, typename F>
__device__ __forceinline__ V sell_row_sum(const SellOp<AV, CT>& m, const SellSlice& s, int lane, const XV* x, F& fx) {
#pragma clang fp contract(off)
    // (past a slice's last step: the next slice's, or the arrays' padding)
    const uint64_t* mask = m.mask + s.base / kSlice;
    constexpr int U = kSellAhead;
    V acc = (V)0;
    if (s.dia) {
        const int32_t* off = m.off + s.base / kSlice;
        const int rc = min(s.row, m.n - 1);
        for (int j0 = 0; j0 < s.w; j0 += U) {
            AV av[U];
            XV xv[U];
            bool in[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const uint64_t mk = j0 + u < s.w ? mask[j0 + u] : 0;
                const int d = off[j0 + u];
                in[u] = __builtin_amdgcn_inverse_ballot_w64(mk);
                av[u] = m.val[s.base + min(j0 + u, s.w - 1) * kSlice + lane];
                xv[u] = x[in[u] ? rc + d : rc];
            }
            if (j0 == 0) fx.begin();
#pragma unroll
            for (int u = 0; u < U; u++) {
                const V pv = (V)av[u] * fx((V)xv[u]);
                if (in[u]) acc += pv;
            }
        }
        return acc;
    }
    for (int j0 = 0; j0 < s.w; j0 += U) {
        int cj[U];
        AV av[U];
        XV xv[U];
        bool in[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int slot = s.base + min(j0 + u, s.w - 1) * kSlice + lane;
            in[u] = __builtin_amdgcn_inverse_ballot_w64(j0 + u < s.w ? mask[j0 + u] : 0);
            cj[u] = csr_col(m.col, slot, s.r0);
            av[u] = m.val[slot];
        }
#pragma unroll
        for (int u = 0; u < U; u++) xv[u] = x[cj[u]];
        if (j0 == 0) fx.begin();
#pragma unroll
        for (int u = 0; u < U; u++) {
            const V pv = (V)av[u] * fx((V)xv[u]);
            if (in[u]) acc += pv;
        }
    }
    return acc;
}

// y = A x (or y = bsub - A x) over slices (sell_row_sum).  Dot products as
// k_csr_stream.  Slices go to waves in groups of kRowBlock/64 through
// RowBlocks, so each XCD takes a contiguous share.
template <typename V, typename AV, typename CT, typename XV, typename YV, int DOTS>
__global__ void __launch_bounds__(kRowBlock)
k_sell(SellOp<AV, CT> m, const XV* __restrict__ x, YV* __restrict__ y, const double* __restrict__ bsub,
       const V* __restrict__ dr, const V* __restrict__ dw, double* __restrict__ partials,
       const int* __restrict__ done_flag) {
#pragma clang fp contract(off)
    const int done = done_flag ? *done_flag : 0;
    constexpr int WPB = kRowBlock / kSlice;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kSlice), lane = threadIdx.x % kSlice;
    double d0 = 0.0, d1 = 0.0, d2 = 0.0;
    const RowBlocks it((m.nsl + WPB - 1) / WPB);
    for (int g = it.b; g < it.hi; g += it.step) {
        const int sl = g * WPB + wave;
        if (sl >= m.nsl) continue;
        const SellSlice s = sell_slice(m, sl, lane);
        if (done) break;  // (after the slice's own loads, which are in flight with the flag's)
        SellX fx;
        V acc = sell_row_sum<V>(m, s, lane, x, fx);
        const int row = s.row;
        if (row < m.n) {
            if (m.rs) acc = acc * (V)m.rs[row];
            double yv = (double)acc;
            if (bsub) yv = bsub[row] - yv;
            const YV yo = (YV)yv;
            y[row] = yo;
            if (DOTS == DOT_XY) {
                d0 += (double)x[row] * yv;
                d1 += yv * yv;
            } else if (DOTS == DOT_PC) {
                const double z = (double)yo;
                d0 += (double)dr[row] * z;
                d1 += z * z;
                d2 += z * (double)dw[row];
            }
        }
    }
    if (done) return;
    if (DOTS == DOT_XY) {
        double v[2] = {d0, d1};
        block_partials<2>(v, partials);
    } else if (DOTS == DOT_PC) {
        double v[3] = {d0, d1, d2};
        block_partials<3>(v, partials);
    }
}

// Slots of the sliced ELL form of a CSR matrix over its entries, rows in
// order (window 0) or sorted by length within windows of that many.
inline double sell_fill(const int32_t* rowptr, int n, int window) {
    int64_t slots = 0;
    std::vector<int32_t> count;  // of a window's rows by length
    for (int w0 = 0; w0 < n; w0 += window ? window : kSlice) {
        const int w1 = std::min(n, w0 + (window ? window : kSlice));
        int top = 0;
        for (int r = w0; r < w1; r++) top = std::max(top, rowptr[r + 1] - rowptr[r]);
        if (!window) {
            slots += (int64_t)kSlice * top;
            continue;
        }
        count.assign((size_t)top + 1, 0);
        for (int r = w0; r < w1; r++) count[rowptr[r + 1] - rowptr[r]]++;
        for (int q = 0, l = top; q < w1 - w0; q += kSlice) {  // the length of sorted row q
            int before = 0;
            for (int d = top; d > l; d--) before += count[d];
            while (before + count[l] <= q) before += count[l--];
            slots += (int64_t)kSlice * l;
        }
    }
    return n > 0 && rowptr[n] > 0 ? (double)slots / (double)rowptr[n] : 1.0;
}

// The form that a matrix's products take.  In order where that pads to at
// most kSellMaxFill times the entries; sorted where that does and either
//   - the order itself pads to at most 1.75: linear tetrahedra and triangles
//     of unstructured meshes (1.30 to 1.37), quadratic elements of lattices
//     (1.28 to 1.68), whose rows move little; or
//   - the matrix has at most a million entries: then every x is near, and the
//     CSR product is bound by its chain of barriers (8.5 us) and not by loads;
// and the CSR stream product otherwise.  Quadratic elements of unstructured
// meshes pad to 2.07 (triangles) and 2.98 (tetrahedra) in order; sorted, the
// rows of a slice come from all over the window and no two lanes share a line
// of x.  CSR against sorted slices, FP64 and FP32: linear tetrahedra, 301k
// rows, 18.7 and 16.0 -> 15.0 and 11.1 us, 804k rows 35.8 and 32.9 -> 34.4
// and 25.7; a lattice's quadratic ones, 531k rows, 41.0 and 38.8 -> 34.7 and
// 25.1; quadratic triangles, 40k rows, 9.0 and 9.0 -> 5.0 and 4.8, but 1.2M
// rows 36.4 and 32.8 -> 41.0 and 31.7, numbered at random 398k rows 28.4 and
// 25.0 -> 36.8 and 28.5.  Runs of 512 and 2048 rows keep more of the
// tetrahedra within the padding and are slower: unstructured quadratic ones,
// 223k rows, CSR 23.4 and 22.4, sorted 30.8 and 24.2, and 54.2 and 37.0 us;
// linear ones, 804k rows, 36.5 and 25.9, and 49.0 and 32.0 us.  A matrix of
// one window is one run: its x is in one CU's cache, and short runs' remainders
// would pad it past the limit (324 rows: the one-workgroup GMRES cycle, 0.32
// against 0.57 ms a step, takes slices).
constexpr double kSellMaxFill = 1.2;
enum SellOrder { SELL_NONE, SELL_IN_ORDER, SELL_SORTED };

// The rows' own padding decides; what diagonal slices add to it (1/8 at most)
// costs less than the indices they save.
inline bool sell_fits(const int32_t* rowptr, int n, double* fill = nullptr) {
    const double f = sell_fill(rowptr, n, 0);
    if (fill) *fill = f;
    return f <= kSellMaxFill;
}

// Rows that are sorted together.
inline int sell_run(int n) { return n <= kSellWindow ? kSellWindow : kSellRun; }

inline SellOrder sell_order(const int32_t* rowptr, int n) {
    double fill;
    if (sell_fits(rowptr, n, &fill)) return SELL_IN_ORDER;
    if (fill > 1.75 && rowptr[n] > 1000000) return SELL_NONE;
    return sell_fill(rowptr, n, sell_run(n)) <= kSellMaxFill ? SELL_SORTED : SELL_NONE;
}

// out[t] = src[t] >= 0 ? in[src[t]] : 0 (a value array in slot order)
template <typename SV, typename DV>
__global__ void __launch_bounds__(256)
k_sell_gather(int64_t m, const int32_t* __restrict__ src, const SV* __restrict__ in, DV* __restrict__ out) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < m) {
        const int32_t k = src[t];
        out[t] = k >= 0 ? (DV)in[k] : (DV)0;
    }
}

// Fixed grid of k_sell.
inline int sell_grid(int nsl);

// int16 column offsets from each row block's first row; false (and out
// untouched) when an offset does not fit.
inline bool compress_columns(const int32_t* rowptr, const int32_t* col, const std::vector<int32_t>& rb,
                             std::vector<int16_t>& out) {
    const int nrb = (int)rb.size() - 1;
    std::vector<int16_t> c16((size_t)rowptr[rb[nrb]]);
    for (int b = 0; b < nrb; b++) {
        const int r0 = rb[b];
        for (int k = rowptr[r0]; k < rowptr[rb[b + 1]]; k++) {
            const int d = col[k] - r0;
            if (d < -32768 || d > 32767) return false;
            c16[k] = (int16_t)d;
        }
    }
    out.swap(c16);
    return true;
}

// Fixed grid for k_csr_stream: a multiple of 8, at most kMaxRowGrid.
inline int stream_grid(int nrb) {
    static const int cap = [] {
        const char* e = getenv("FLGPU_STREAM_GRID");
        const int v = e ? atoi(e) : kMaxRowGrid;
        return v >= 8 && v <= kMaxRowGrid ? v : kMaxRowGrid;
    }();
    if (nrb < 8) return nrb > 0 ? nrb : 1;
    const int g = nrb < cap ? nrb : cap;
    return g & ~7;
}

// The groups of slices over as many workgroups as give each the same number
// of them (a workgroup with one more would double a short product's time).
inline int sell_grid(int nsl) {
    constexpr int per = kRowBlock / kSlice;
    const int groups = (nsl + per - 1) / per;
    if (groups < 8) return std::max(1, groups);
    const int rounds = (groups + stream_grid(kMaxRowGrid) - 1) / stream_grid(kMaxRowGrid);
    return ((groups + rounds - 1) / rounds + 7) & ~7;
}

template <typename V, typename AV, typename CT, typename XV, typename YV, int DOTS>
inline void sell_product(hipStream_t stream, const SellOp<AV, CT>& m, const XV* x, YV* y, const double* bsub,
                         const V* dr, const V* dw, double* partials, const int* done_flag) {
    hipLaunchKernelGGL((k_sell<V, AV, CT, XV, YV, DOTS>), dim3(sell_grid(m.nsl)), dim3(kRowBlock), 0, stream, m, x, y,
                       bsub, dr, dw, partials, done_flag);
}

}  // namespace flgpu
