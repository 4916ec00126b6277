// Krylov solve of the assembled system on gfx950.
//
// The hand-off reproduces petsc_solve (femtools/Solvers.F90:111-187):
//   - inactive (strong Dirichlet) rows become "ghost" rows holding only the
//     diagonal ghost_pivot = sqrt((maxdiag+mindiag)*maxdiag/2) over all
//     |A_ii| (femtools/Petsc_Tools.F90:959-984, :1045-1057);
//   - inactive columns are dropped and lifted into the rhs,
//     b = rhs - A*ghost_rhs (femtools/Solvers.F90:1072-1099), and ghost rows
//     get b = 0;
//   - after the solve the ghost entries of x take the rhs values
//     (femtools/Petsc_Tools.F90:724-731).
// Methods: KSPCG-style preconditioned CG, flexible CG (Polak-Ribiere beta)
// for the learned preconditioner, restarted GMRES with left Jacobi.
// Precision: FP64, or FP32 inner iterations with FP64 dot-product
// accumulation and FP64 true-residual replacement ("reliable updates",
// iterative refinement without restarting CG); the FP32 iterations add
// their steps alpha p to an FP32 increment that is added to the FP64
// solution at every replacement (and at the end), so x itself is FP64.
// Every reduction has a fixed order: results repeat bit for bit.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

#include "flgpu_internal.h"
#include "krylov_common.h"
#include "learned.h"
#include "sell_plan.h"

namespace flgpu {


struct KrylovWork {
    int n = 0;
    int64_t nnz = 0;
    DevBuf<double> val64, b, x, r, z, p, w, dinv, y, rt;
    DevBuf<float> val32, r32, z32, p32, w32, dinv32, y32, rt32;
    DevBuf<double> s;        // single-reduction CG: s = A p by recurrence
    DevBuf<float> s32;
    DevBuf<float> dx32;      // mixed CG: the FP32 increment of x since the last replacement
    bool dx_on = false;      // dx32 holds steps not yet added to x
    int npc = 0;             // partial sums of the last preconditioner apply
    DevBuf<double> partials;
    DevBuf<Scal> scal;       // two slots, see carry_if_done
    int cur = 0;             // slot holding the current state
    DevBuf<int32_t> rb, rbk; // row blocks of the streamed CSR product
    DevBuf<int16_t> col16;   // int16 column offsets (when use16)
    bool use16 = false;
    int nrb = 0;
    int64_t rb_key = -1;     // sparsity generation rb was built for
    // sliced ELL copy of the solver matrix, used by spmv when there is a plan
    SellPlan sell;
    DevBuf<double> sval64;
    DevBuf<float> sval32;
    Scal* h_scal = nullptr;  // host copy of the current slot (pinned when h_scal_owned)
    bool h_scal_owned = false;
    int64_t* word = nullptr;   // the CG loops' progress, 2 its + done, behind h_scal when that is pinned,
    int64_t* d_word = nullptr; // its address for the device,
    int64_t* pub = nullptr;    // and what a batch's iterations write to (null: not published)
    int nblk = 1;
    Scal* S() { return scal.p + cur; }
    double* part(int region) { return partials.p + (size_t)region * kPartStride; }
    // multicolour SSOR: the rows of a colour in slices of 64 (one wave), their
    // off-diagonal entries in slots as in a sliced ELL matrix -- those in
    // earlier colours for the forward sweep (f), all of them for the backward (b)
    struct SorHalf {
        DevBuf<int32_t> ptr, len, col, src;
        DevBuf<double> v64;
        DevBuf<float> v32;
    } mc_f, mc_b;
    DevBuf<int32_t> mc_rows, mc_dsrc, mc_cptr;
    DevBuf<double> mc_d64;
    DevBuf<float> mc_d32;
    std::vector<int32_t> mc_ptr;  // colour c owns slices mc_ptr[c] .. mc_ptr[c+1]
    int64_t mc_key = -1;          // sparsity generation of the colouring
    bool mc_one = false;          // a sweep by one workgroup
    // GMRES
    DevBuf<double> V, gm_work;  // basis; block sums, Hessenberg column, rotations
    DevBuf<float> V32;
    DevBuf<unsigned char> gm_state;
    void* gm_host = nullptr;    // the solve's progress, in pinned memory that the device writes
    bool have_x = false;
    bool prepared = false, prepared_mixed = false;
    ~KrylovWork() {
        if (h_scal && h_scal_owned) (void)hipHostFree(h_scal);
        if (gm_host) (void)hipHostFree(gm_host);
    }
};

// ---------------------------------------------------------------------
// Reduced system
// ---------------------------------------------------------------------

// Per-block min and max of |A_ii| (min/max do not depend on the order).
__global__ void __launch_bounds__(kVecBlock)
k_diag_minmax(int n, const int32_t* __restrict__ diag, const double* __restrict__ A,
              double* __restrict__ partials) {
    double mn = 1.79769313486231570e308, mx = -1.79769313486231570e308;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const int d = diag[i];
        const double v = d >= 0 ? fabs(A[d]) : 0.0;
        mn = fmin(mn, v);
        mx = fmax(mx, v);
    }
    __shared__ double sh[kVecBlock / 64][2];
    for (int off = 32; off > 0; off >>= 1) {
        mn = fmin(mn, __shfl_xor(mn, off, 64));
        mx = fmax(mx, __shfl_xor(mx, off, 64));
    }
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (lane == 0) {
        sh[wave][0] = mn;
        sh[wave][1] = mx;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int q = 1; q < (int)(blockDim.x >> 6); q++) {
            sh[0][0] = fmin(sh[0][0], sh[q][0]);
            sh[0][1] = fmax(sh[0][1], sh[q][1]);
        }
        partials[blockIdx.x] = sh[0][0];
        partials[kPartStride + blockIdx.x] = sh[0][1];
    }
}

// One wave: ghost pivot sqrt((max+min)*max/2) from the per-block extrema.
__global__ void __launch_bounds__(64)
k_pivot(int nparts, const double* __restrict__ partials, Scal* sc) {
    double a = 1.79769313486231570e308, b = -1.79769313486231570e308;
    for (int q = threadIdx.x; q < nparts; q += 64) {
        a = fmin(a, partials[q]);
        b = fmax(b, partials[kPartStride + q]);
    }
    for (int off = 32; off > 0; off >>= 1) {
        a = fmin(a, __shfl_xor(a, off, 64));
        b = fmax(b, __shfl_xor(b, off, 64));
    }
    if (threadIdx.x == 0) {
        sc->dmin = a;
        sc->dmax = b;
        sc->pivot = sqrt((b + a) * b / 2.0);
    }
}

// The reduced (PETSc-side) system, per row block: the block's entries are
// read once, coalesced, and one thread per row then finishes the row from
// LDS.  Ghost rows keep only the pivot on the diagonal, inactive columns
// are dropped and lifted into the rhs -- b_i = rhs_i - sum_k A_ik rhs_k over
// the inactive columns k, in entry order with the product rounded first,
// as the reference's csr_mult of the ghost values does -- and the Jacobi
// inverse diagonal and the initial x are set.
__global__ void __launch_bounds__(kRowBlock)
k_build(int nrb, const int32_t* __restrict__ rb, const int32_t* __restrict__ rowptr,
        const int32_t* __restrict__ col, const double* __restrict__ A, const double* __restrict__ rhs,
        const int32_t* __restrict__ inactive, int have_inactive, const Scal* __restrict__ sc,
        double* __restrict__ v64, float* __restrict__ v32, double* __restrict__ b, double* __restrict__ dinv,
        float* __restrict__ dinv32, double* __restrict__ x, int zero_x) {
    __shared__ double slift[kStreamNnz];
    __shared__ double sdiag[kRowBlock];
    __shared__ uint8_t serow[kStreamNnz];
    const double pivot = sc->pivot;
    const RowBlocks it(nrb);
    for (int blk = it.b; blk < it.hi; blk += it.step) {
        const int r0 = rb[blk], r1 = rb[blk + 1];
        const int k0 = rowptr[r0], k1 = rowptr[r1];
        const int row = r0 + threadIdx.x;
        const bool staged = k1 - k0 <= kStreamNnz;
        if (staged) {
            if (row < r1) {
                sdiag[threadIdx.x] = 0.0;
                for (int k = rowptr[row]; k < rowptr[row + 1]; k++) serow[k - k0] = (uint8_t)threadIdx.x;
            }
            __syncthreads();
#pragma unroll
            for (int j = 0; j < kStreamPerThread; j++) {
                const int k = k0 + threadIdx.x + j * kRowBlock;
                if (k < k1) {
                    const int l = serow[k - k0], i = r0 + l, cj = col[k];
                    const double a = A[k];
                    const bool ghost = have_inactive && inactive[i];
                    const bool off = have_inactive && inactive[cj];
                    double v = a;
                    if (ghost) v = (cj == i) ? pivot : 0.0;
                    else if (off) v = 0.0;
                    v64[k] = v;
                    if (v32) v32[k] = (float)v;
                    if (cj == i) sdiag[l] = v;
                    slift[k - k0] = (!ghost && off) ? a * rhs[cj] : 0.0;
                }
            }
            __syncthreads();
        }
        if (row < r1) {
            const bool ghost = have_inactive && inactive[row];
            double lift = 0.0, dval = 0.0;
            if (staged) {
                for (int k = rowptr[row]; k < rowptr[row + 1]; k++) lift = lift + slift[k - k0];
                dval = sdiag[threadIdx.x];
            } else {  // a row longer than the staging buffer (alone in its block)
                for (int k = rowptr[row]; k < rowptr[row + 1]; k++) {
                    const int cj = col[k];
                    const double a = A[k];
                    const bool off = have_inactive && inactive[cj];
                    double v = a;
                    if (ghost) v = (cj == row) ? pivot : 0.0;
                    else if (off) v = 0.0;
                    v64[k] = v;
                    if (v32) v32[k] = (float)v;
                    if (cj == row) dval = v;
                    if (!ghost && off) lift = lift + a * rhs[cj];
                }
            }
            b[row] = ghost ? 0.0 : rhs[row] - lift;
            const double di = dval != 0.0 ? 1.0 / dval : 1.0;
            dinv[row] = di;
            if (dinv32) dinv32[row] = (float)di;
            if (zero_x || ghost) x[row] = 0.0;
        }
        __syncthreads();
    }
}

// ---------------------------------------------------------------------
// PCG / FCG vector kernels
// ---------------------------------------------------------------------

// The scalars an iteration reads and changes, in registers of every thread
// (the whole Scal as a local variable would go through LDS or scratch).
struct CgState {
    double rz, rz_old, pAp, alpha, beta, rr, zz, zw, last_norm;
    int its, reason, done;
};

__device__ __forceinline__ CgState cg_state(const Scal* __restrict__ in) {
    return {in->rz, in->rz_old, in->pAp, in->alpha, in->beta, in->rr, in->zz, in->zw, in->last_norm, in->its, in->reason,
            in->done};
}

// The next slot: the state, the rest carried over.
__device__ __forceinline__ void cg_store(const Scal* __restrict__ in, Scal* __restrict__ out, const CgState& s) {
    *out = *in;
    out->rz = s.rz;
    out->rz_old = s.rz_old;
    out->pAp = s.pAp;
    out->alpha = s.alpha;
    out->beta = s.beta;
    out->rr = s.rr;
    out->zz = s.zz;
    out->zw = s.zw;
    out->last_norm = s.last_norm;
    out->its = s.its;
    out->reason = s.reason;
    out->done = s.done;
}

// The iteration's state for the host (cg_ahead); one store, nothing ordered
// after it.
__device__ __forceinline__ void cg_publish(int64_t* word, const CgState& s) {
    if (word) __hip_atomic_store(word, (int64_t)2 * s.its + s.done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Convergence test of KSPConvergedDefault on the norm chosen by norm_type,
// then beta (Fletcher-Reeves, or Polak-Ribiere when flexible).
__device__ __forceinline__ void cg_test(CgState& s, const Scal* __restrict__ in) {
    s.its += 1;
    const double nrm = in->norm_type == FLGPU_NORM_UNPRECONDITIONED ? sqrt(s.rr) : sqrt(s.zz);
    const double rnorm0 = in->rnorm0;
    s.last_norm = nrm;
    if (nrm != nrm || isinf(nrm)) {
        s.reason = KSP_DIVERGED_NANORINF;
        s.done = 1;
    } else if (nrm <= in->atol) {
        s.reason = KSP_CONVERGED_ATOL;
        s.done = 1;
    } else if (nrm <= in->rtol * rnorm0) {
        s.reason = KSP_CONVERGED_RTOL;
        s.done = 1;
    } else if (rnorm0 > 0 && nrm >= 1e5 * rnorm0) {
        s.reason = KSP_DIVERGED_DTOL;
        s.done = 1;
    } else if (s.its >= in->max_its) {
        s.reason = KSP_DIVERGED_ITS;
        s.done = 1;
    }
}

__device__ __forceinline__ void cg_test_and_beta(CgState& s, const Scal* __restrict__ in) {
    cg_test(s, in);
    if (in->flexible)
        s.beta = -s.alpha * s.zw / s.rz_old;  // z.(r_new - r_old) / (z_old.r_old)
    else
        s.beta = s.rz / s.rz_old;
    if (!s.done && s.rz < 0.0) {
        s.reason = KSP_DIVERGED_INDEFINITE_PC;
        s.done = 1;
    }
}

// The solver scalars advance through two slots: a kernel that changes
// them reads slot "in" in every block and block 0 writes the next state
// to slot "out", so no block can see a value written during its own
// kernel.  A finished solve carries the state over unchanged.

// R consecutive entries as one vector load / store (R * sizeof(T) bytes;
// the caller checks the alignment with rows_aligned)
template <typename T, int R>
using Rows = T __attribute__((ext_vector_type(R)));

template <int R, typename T>
__device__ __forceinline__ Rows<T, R> ld_rows(const T* __restrict__ a, int i) {
    return *reinterpret_cast<const Rows<T, R>*>(a + i);
}
template <int R, typename T>
__device__ __forceinline__ void st_rows(T* __restrict__ a, int i, const Rows<T, R>& v) {
    *reinterpret_cast<Rows<T, R>*>(a + i) = v;
}

// The vector kernels of an iteration are bound by latency (a launch, the
// partial sums, the rows): so one block per CU, every load in flight before
// the first is used, one barrier, and the scalar step taken by every thread.
// With 512 blocks of 512, a broadcast by thread 0 and rows loaded after it:
// update 9.9 and p 7.2 us on 274k FP64 rows, 13.6 and 12.0 us on 1.37M FP32
// rows with a factor; so 7.4 and 4.3, 11.2 and 6.8 us.
//
// pAp from the SpMV partials, alpha = rz / pAp; x += alpha p;
// r -= alpha w; [Jacobi: z = D^-1 r]; [learned: rt = D_s r, the residual in
// the preconditioner's scaled space]; partials r.z, r.r, z.z, z.w.  Each
// thread takes R consecutive rows per step with vector loads (the rows past
// the last whole group go one at a time), so several loads of every vector
// are in flight per thread.
template <typename V, int R>
__global__ void __launch_bounds__(kVecBlock)
k_cg_update(int n, V* __restrict__ x, const V* __restrict__ p, V* __restrict__ r,
            const V* __restrict__ w, V* __restrict__ z, const V* __restrict__ dinv, int jacobi,
            const float* __restrict__ dsc, V* __restrict__ rt,
            const double* __restrict__ pspmv, int nspmv, double* __restrict__ pvec,
            const Scal* __restrict__ in, Scal* __restrict__ out) {
    // The thread's first group of rows, the scalars and the partial sums are
    // in flight together; every thread takes the scalar step itself.
    const int ng = n / R, tid = blockIdx.x * blockDim.x + threadIdx.x, nt = gridDim.x * blockDim.x;
    Rows<V, R> pv = {}, wv = {}, rv = {}, dv = {}, xv = {};
    Rows<float, R> sv = {};
    auto load = [&](int i) {
        pv = ld_rows<R>(p, i);
        wv = ld_rows<R>(w, i);
        rv = ld_rows<R>((const V*)r, i);
        xv = ld_rows<R>((const V*)x, i);
        if (jacobi) dv = ld_rows<R>(dinv, i);
        if (dsc) sv = ld_rows<R>(dsc, i);
    };
    if (tid < ng) load(tid * R);
    CgState s = cg_state(in);
    double pap[1];
    part_totals<1>(pspmv, nspmv, pap);
    if (!s.done) {
        s.pAp = pap[0];
        s.rz_old = s.rz;
        if (!(pap[0] > 0.0)) {
            s.reason = (pap[0] != pap[0]) ? KSP_DIVERGED_NANORINF : KSP_DIVERGED_INDEFINITE_MAT;
            s.done = 1;
        } else {
            s.alpha = s.rz / pap[0];
        }
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) cg_store(in, out, s);
    if (s.done) return;
    const double alpha = s.alpha;
    const V a = (V)alpha;
    double s_rz = 0.0, s_rr = 0.0, s_zz = 0.0, s_zw = 0.0;
    auto row = [&](V& xi, V pi, V wi, V& ri, V di, float si, V& zi, V& ti) {
        xi = fma((V)alpha, pi, xi);
        ri = ri - a * wi;
        if (dsc) ti = ri * (V)si;
        if (jacobi) {
            zi = di * ri;
            s_rz += (double)ri * (double)zi;
            s_zz += (double)zi * (double)zi;
            s_zw += (double)zi * (double)wi;
        }
        s_rr += (double)ri * (double)ri;
    };
    for (int g = tid; g < ng; g += nt) {
        const int i = g * R;
        if (g != tid) load(i);
        Rows<V, R> zv = {}, tv = {};
#pragma unroll
        for (int u = 0; u < R; u++) {
            V xi = xv[u];
            V ri = rv[u], zi = (V)0, ti = (V)0;
            row(xi, pv[u], wv[u], ri, dv[u], sv[u], zi, ti);
            xv[u] = xi;
            rv[u] = ri;
            zv[u] = zi;
            tv[u] = ti;
        }
        st_rows<R>(x, i, xv);
        st_rows<R>(r, i, rv);
        if (jacobi) st_rows<R>(z, i, zv);
        if (dsc) st_rows<R>(rt, i, tv);
    }
    for (int i = ng * R + tid; i < n; i += nt) {
        V xi = x[i];
        V ri = r[i], zi = (V)0, ti = (V)0;
        row(xi, p[i], w[i], ri, jacobi ? dinv[i] : (V)0, dsc ? dsc[i] : 0.f, zi, ti);
        x[i] = xi;
        r[i] = ri;
        if (jacobi) z[i] = zi;
        if (dsc) rt[i] = ti;
    }
    double v[4] = {s_rz, s_rr, s_zz, s_zw};
    block_partials<4>(v, pvec);
}

// r.z, r.r, z.z, z.w from the update partials (or r.z, z.z, z.w from the
// learned apply), convergence test and beta in every block; p = z + beta p
// (R rows per thread and step, as k_cg_update).
template <typename V, int R>
__global__ void __launch_bounds__(kVecBlock)
k_cg_p(int n, const V* __restrict__ z, V* __restrict__ p, const double* __restrict__ pvec, int nvec,
       const double* __restrict__ ppc, int npc, const Scal* __restrict__ in, Scal* __restrict__ out, int64_t* word) {
    // The thread's first group of rows does not depend on the scalars: its
    // loads are issued before the scalars' and the partial sums', so the
    // three are in flight together (one memory round trip, not two).
    const int ng = n / R, tid = blockIdx.x * blockDim.x + threadIdx.x, nt = gridDim.x * blockDim.x;
    Rows<V, R> zv = {}, pv = {};
    auto load = [&](int i) {
        zv = ld_rows<R>(z, i);
        pv = ld_rows<R>((const V*)p, i);
    };
    if (tid < ng) load(tid * R);
    CgState s = cg_state(in);
    double u[4];
    if (ppc) {
        double q[3], rr[1];
        part_totals<3>(ppc, npc, q);
        part_totals<1>(pvec + kPartStride, nvec, rr);
        u[0] = q[0];
        u[1] = rr[0];
        u[2] = q[1];
        u[3] = q[2];
    } else {
        part_totals<4>(pvec, nvec, u);
    }
    if (!s.done) {
        s.rz = u[0];
        s.rr = u[1];
        s.zz = u[2];
        s.zw = u[3];
        cg_test_and_beta(s, in);
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        cg_store(in, out, s);
        cg_publish(word, s);
    }
    if (s.done) return;
    const V beta = (V)s.beta;
    for (int g = tid; g < ng; g += nt) {
        const int i = g * R;
        if (g != tid) load(i);
#pragma unroll
        for (int k = 0; k < R; k++) pv[k] = fma(beta, pv[k], zv[k]);
        st_rows<R>(p, i, pv);
    }
    for (int i = ng * R + tid; i < n; i += nt) p[i] = fma(beta, p[i], z[i]);
}

// Single-reduction CG (Chronopoulos & Gear 1989), the recurrence PETSc's
// KSPPIPECG builds on: with u = M r, w = A u, gamma = r.u and delta = u.w
// from one reduction phase,
//   beta = gamma / gamma_old, alpha = gamma / (delta - beta gamma / alpha_old),
//   p = u + beta p, s = w + beta s (s = A p), x += alpha p, r -= alpha s,
// then u = M r (Jacobi here; a factor by its own kernels) and w = A u (the
// next product).  One vector kernel an iteration instead of k_cg_update
// and k_cg_p.  The previous iteration's sums: delta (the product's u.w,
// pspmv), gamma, u.u and r.r (pg: this kernel's own region from the
// previous iteration, or the factor apply's r.z, z.z with pc_layout set,
// then r.r from prr); first: the iteration after a restart (gamma, r.r, u.u
// already in the scalars, p = u, s = w).  Partials r.u, r.r, u.u, 0 to
// pvec (a region other than pg and prr).
template <typename V, int R>
__global__ void __launch_bounds__(kVecBlock)
k_cg1_vec(int n, double* __restrict__ x, V* __restrict__ p, V* __restrict__ s, V* __restrict__ r,
          V* __restrict__ u, const V* __restrict__ w, const V* __restrict__ dinv, int jacobi,
          const float* __restrict__ dsc, V* __restrict__ rt, const double* __restrict__ pspmv, int nspmv,
          const double* __restrict__ pg, int ng, int pc_layout, const double* __restrict__ prr, int nrr, int first,
          double* __restrict__ pvec, const Scal* __restrict__ in, Scal* __restrict__ out, int64_t* word) {
    // the first group's loads in flight with the scalars' (as k_cg_p)
    const int ng_ = n / R, tid = blockIdx.x * blockDim.x + threadIdx.x, nt = gridDim.x * blockDim.x;
    Rows<V, R> pv = {}, sv = {}, rv = {}, uv = {}, wv = {}, dv = {};
    Rows<double, R> xv = {};
    Rows<float, R> fv = {};
    auto load = [&](int i) {
        pv = ld_rows<R>((const V*)p, i);
        sv = ld_rows<R>((const V*)s, i);
        rv = ld_rows<R>((const V*)r, i);
        uv = ld_rows<R>((const V*)u, i);
        wv = ld_rows<R>(w, i);
        xv = ld_rows<R>((const double*)x, i);
        if (jacobi) dv = ld_rows<R>(dinv, i);
        if (dsc) fv = ld_rows<R>(dsc, i);
    };
    if (tid < ng_) load(tid * R);
    CgState sc = cg_state(in);
    double dl[1], g[3] = {0.0, 0.0, 0.0}, q[1] = {0.0};
    part_totals<1>(pspmv, nspmv, dl);
    if (!first) {
        part_totals<3>(pg, ng, g);
        if (pc_layout) part_totals<1>(prr + kPartStride, nrr, q);
    }
    if (!sc.done) {
        if (!first) {
            sc.rz_old = sc.rz;
            sc.rz = g[0];
            sc.rr = pc_layout ? q[0] : g[1];
            sc.zz = pc_layout ? g[1] : g[2];
            cg_test(sc, in);
        }
        const double delta = dl[0];
        sc.pAp = delta;
        if (!sc.done) {
            const double beta = first ? 0.0 : sc.rz / sc.rz_old;
            const double denom = first ? delta : delta - beta * sc.rz / sc.alpha;
            if (sc.rz < 0.0) {
                sc.reason = KSP_DIVERGED_INDEFINITE_PC;
                sc.done = 1;
            } else if (!(denom > 0.0)) {
                sc.reason = (denom != denom) ? KSP_DIVERGED_NANORINF : KSP_DIVERGED_INDEFINITE_MAT;
                sc.done = 1;
            } else {
                sc.beta = beta;
                sc.alpha = sc.rz / denom;
            }
        }
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        cg_store(in, out, sc);
        cg_publish(word, sc);
    }
    if (sc.done) return;
    const double alpha = sc.alpha;
    const V a = (V)alpha, b = (V)sc.beta;
    double s_g = 0.0, s_rr = 0.0, s_uu = 0.0;
    auto row = [&](double& xi, V& pi, V& si, V ui, V wi, V& ri, V di, float dsi, V& uo, V& ti) {
        pi = first ? ui : fma(b, pi, ui);
        si = first ? wi : fma(b, si, wi);
        xi = fma(alpha, (double)pi, xi);
        ri = ri - a * si;
        if (dsc) ti = ri * (V)dsi;
        if (jacobi) {
            uo = di * ri;
            s_g += (double)ri * (double)uo;
            s_uu += (double)uo * (double)uo;
        }
        s_rr += (double)ri * (double)ri;
    };
    for (int gi = tid; gi < ng_; gi += nt) {
        const int i = gi * R;
        if (gi != tid) load(i);
        Rows<V, R> uo = {}, tv = {};
#pragma unroll
        for (int k = 0; k < R; k++) {
            double xi = xv[k];
            V pi = pv[k], si = sv[k], ri = rv[k], uk = (V)0, ti = (V)0;
            row(xi, pi, si, uv[k], wv[k], ri, dv[k], fv[k], uk, ti);
            xv[k] = xi;
            pv[k] = pi;
            sv[k] = si;
            rv[k] = ri;
            uo[k] = uk;
            tv[k] = ti;
        }
        st_rows<R>(x, i, xv);
        st_rows<R>(p, i, pv);
        st_rows<R>(s, i, sv);
        st_rows<R>(r, i, rv);
        if (jacobi) st_rows<R>(u, i, uo);
        if (dsc) st_rows<R>(rt, i, tv);
    }
    for (int i = ng_ * R + tid; i < n; i += nt) {
        double xi = x[i];
        V pi = p[i], si = s[i], ri = r[i], uk = (V)0, ti = (V)0;
        row(xi, pi, si, u[i], w[i], ri, jacobi ? dinv[i] : (V)0, dsc ? dsc[i] : 0.f, uk, ti);
        x[i] = xi;
        p[i] = pi;
        s[i] = si;
        r[i] = ri;
        if (jacobi) u[i] = uk;
        if (dsc) rt[i] = ti;
    }
    double v[4] = {s_g, s_rr, s_uu, 0.0};
    block_partials<4>(v, pvec);
}

template <typename V>
__global__ void __launch_bounds__(kVecBlock)
k_copy(int n, const V* __restrict__ a, V* __restrict__ b) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) b[i] = a[i];
}

template <typename V>
__global__ void __launch_bounds__(kVecBlock)
k_fill(int n, V v, V* __restrict__ a) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) a[i] = v;
}

// r_V = (V) r64 ; z = D^-1 r ; partials r.z, r.r, z.z
template <typename V>
__global__ void __launch_bounds__(kVecBlock)
k_restart_vecs(int n, const double* __restrict__ r64, V* __restrict__ r, V* __restrict__ z,
               const V* __restrict__ dinv, int jacobi, const float* __restrict__ dsc, V* __restrict__ rt,
               double* __restrict__ pvec) {
    double s_rz = 0.0, s_rr = 0.0, s_zz = 0.0;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const V ri = (V)r64[i];
        r[i] = ri;
        if (dsc) rt[i] = ri * (V)dsc[i];
        s_rr += (double)ri * (double)ri;
        if (jacobi) {
            const V zi = dinv[i] * ri;
            z[i] = zi;
            s_rz += (double)ri * (double)zi;
            s_zz += (double)zi * (double)zi;
        }
    }
    double v[3] = {s_rz, s_rr, s_zz};
    block_partials<3>(v, pvec);
}

__global__ void __launch_bounds__(kVecBlock)
k_dot2(int n, const double* __restrict__ a, double* __restrict__ partials) {
    double s = 0.0;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
        s += a[i] * a[i];
    double v[1] = {s};
    block_partials<1>(v, partials);
}

// One-block finalisation of the rarely used reductions, in place on the
// current scalar slot.
enum FinOp { FIN_TRUE_RR = 0, FIN_BB = 1, FIN_RESTART = 2, FIN_LEARNED = 3 };

__device__ __forceinline__ void set_norm0(Scal& s) {
    const double nrm = s.norm_type == FLGPU_NORM_UNPRECONDITIONED ? sqrt(s.rr) : sqrt(s.zz);
    s.rnorm0 = nrm;
    s.last_norm = nrm;
}

__global__ void __launch_bounds__(kVecBlock)
k_finalize(int op, const double* __restrict__ partials, int nparts, int jacobi, int norm0, Scal* sc) {
    double v[3];
    if (op == FIN_TRUE_RR || op == FIN_BB) {
        double one[1];
        sum_partials<1>(partials + (op == FIN_TRUE_RR ? kPartStride : 0), nparts, one);
        if (threadIdx.x == 0) {
            if (op == FIN_TRUE_RR)
                sc->true_rr = one[0];
            else
                sc->bb = one[0];
        }
        return;
    }
    sum_partials<3>(partials, nparts, v);
    if (threadIdx.x != 0) return;
    Scal s = *sc;
    if (op == FIN_RESTART) {  // r.z, r.r, z.z
        s.rr = v[1];
        if (jacobi) {
            s.rz = v[0];
            s.zz = v[2];
        }
    } else {  // learned apply: r.z, z.z, z.w
        s.rz = v[0];
        s.zz = v[1];
        s.zw = v[2];
    }
    if (norm0) set_norm0(s);
    *sc = s;
}

__global__ void __launch_bounds__(kVecBlock)
k_finish_x(int n, double* __restrict__ x, const double* __restrict__ rhs,
           const int32_t* __restrict__ inactive, int have_inactive) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n && have_inactive && inactive[i]) x[i] = rhs[i];
}

// ---------------------------------------------------------------------
// Multicolour SSOR (the "sor" preconditioner)
// ---------------------------------------------------------------------
//
// PETSc's PCSOR, which femtools/Solvers.F90:1844-1854 selects for "sor",
// applies one local symmetric Gauss-Seidel sweep (omega = 1) in the natural
// row order -- a sequential recurrence.  Here the rows are taken colour by
// colour, ascending inside a colour, where the colours are a first-fit
// colouring of the matrix graph in row order (rows of one colour share no
// entry, so a colour's rows update independently): the same sweep on the
// symmetrically permuted matrix, again symmetric positive definite for an
// SPD system.
//   forward:  z = 0; for c = 0 .. C-1:  z_i = (r_i - sum_{j != i} a_ij z_j) / a_ii
//   backward:        for c = C-2 .. 0:  the same with the current z
// (the last colour's backward step would recompute its forward values; the
// forward step needs only the entries in earlier colours, the others' z being
// 0).  Each row is summed by one thread in entry order with explicit fused
// multiply-adds, the order of the oracle's restatement.
// What bounds it: the chain of 2C - 1 dependent steps.  A launch per colour
// (k_sor_slices) takes 4 us with a few thousand rows a colour (12 us reading
// the CSR rows entry by entry); where z fits LDS and the entries are few, one
// workgroup takes the whole sweep with a barrier per colour (k_sor_block).
// An apply on one MI355X: 41 x 41 P2 triangles (6889 rows, 13 colours), 27
// launches 200 us -> one launch 36 us; 45^3 x 6 P1 tetrahedra (97k rows, 9
// colours) 205 -> 79 us.  Their time steps with GMRES: 2.42 -> 1.33 ms and
// 3.0 -> 1.88 ms.

// One sweep direction: slices ptr[sl] .. of 64 rows, len their entries.
template <typename V>
struct SorOp {
    const int32_t *rows, *ptr, *len, *col;
    const V *val, *dia;
};

constexpr int kSorBatch = 8;

// What a lane needs before the first z: its row, bounds, and the first
// batch of its entries (slots past a slice's width re-read its last one).
template <typename V>
struct SorLane {
    int row, len, base, w;
    V r, d;
    int cj[kSorBatch];
    V av[kSorBatch];
};

template <typename V>
__device__ __forceinline__ void sor_batch(const SorOp<V>& m, SorLane<V>& t, int j0, int lane) {
#pragma unroll
    for (int u = 0; u < kSorBatch; u++) {
        const int slot = t.base + min(j0 + u, t.w - 1) * kSlice + lane;
        t.cj[u] = m.col[slot];
        t.av[u] = m.val[slot];
    }
}

template <typename V>
__device__ __forceinline__ void sor_fetch(const SorOp<V>& m, int sl, int lane, const V* __restrict__ r, SorLane<V>& t) {
    const int q = sl * kSlice + lane;
    t.row = m.rows[q];
    t.len = m.len[q];
    t.d = m.dia[q];
    t.base = m.ptr[sl];
    t.w = (m.ptr[sl + 1] - t.base) / kSlice;
    if (t.w > 0) sor_batch(m, t, 0, lane);
    t.r = t.row >= 0 ? r[t.row] : (V)0;
}

// z of the lane's row from the fetched entries and the current z.
template <typename V>
__device__ __forceinline__ V sor_finish(const SorOp<V>& m, SorLane<V>& t, int lane, const V* z) {
    V acc = t.r;
    for (int j0 = 0; j0 < t.w; j0 += kSorBatch) {
        if (j0 > 0) sor_batch(m, t, j0, lane);
        V zv[kSorBatch];
#pragma unroll
        for (int u = 0; u < kSorBatch; u++) zv[u] = z[t.cj[u]];
#pragma unroll
        for (int u = 0; u < kSorBatch; u++)
            if (j0 + u < t.len) acc = fma(-t.av[u], zv[u], acc);
    }
    return acc / t.d;
}

// A colour's slices s0 .. s1, a wave each.
template <typename V>
__global__ void __launch_bounds__(256)
k_sor_slices(SorOp<V> m, int s0, int s1, const V* __restrict__ r, V* z, const int* __restrict__ done_flag) {
    if (done_flag && *done_flag) return;
    const int sl = s0 + (int)blockIdx.x * 4 + (int)(threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (sl >= s1) return;
    SorLane<V> t;
    sor_fetch(m, sl, lane, r, t);
    const V zi = sor_finish(m, t, lane, (const V*)z);
    if (t.row >= 0) z[t.row] = zi;
}

// Both sweeps by one workgroup, z in LDS: the entries of a wave's first slice
// of the next colour are fetched before the barrier that ends this one.
template <typename V>
__global__ void __launch_bounds__(1024)
k_sor_block(int n, int ncol, const int32_t* __restrict__ cptr, SorOp<V> f, SorOp<V> b, const V* __restrict__ r,
            V* __restrict__ z, const int* __restrict__ done_flag) {
    extern __shared__ double sor_lds[];
    V* zs = reinterpret_cast<V*>(sor_lds);
    if (done_flag && *done_flag) return;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, nw = blockDim.x >> 6, np = 2 * ncol - 1;
    for (int i = threadIdx.x; i < n; i += blockDim.x) zs[i] = (V)0;
    SorLane<V> t;
    auto colour = [&](int p) { return p < ncol ? p : 2 * ncol - 2 - p; };
    auto start = [&](int p) {
        const int q = colour(p), sl = cptr[q] + wave;
        if (sl < cptr[q + 1]) sor_fetch(p < ncol ? f : b, sl, lane, r, t);
    };
    start(0);
    __syncthreads();
    for (int p = 0; p < np; p++) {
        const SorOp<V>& m = p < ncol ? f : b;
        const int q = colour(p), s1 = cptr[q + 1];
        for (int sl = cptr[q] + wave; sl < s1; sl += nw) {
            if (sl != cptr[q] + wave) sor_fetch(m, sl, lane, r, t);
            const V zi = sor_finish(m, t, lane, zs);
            if (t.row >= 0) zs[t.row] = zi;
        }
        if (p + 1 < np) start(p + 1);
        __syncthreads();
    }
    for (int i = threadIdx.x; i < n; i += blockDim.x) z[i] = zs[i];
}

// The slices of a plan, a thread a slot of 64-row slices (rows: -1 past a
// colour's last), in two passes over the CSR rows: the entries of each sweep
// and the slices' widths (in steps), then the entries at their slots.  Built
// by the host, the plan of 1.37M rows of 15 entries took 240 ms, most of the
// first solve; so 4 (and 12 for the colouring, which is the host's).
__global__ void __launch_bounds__(256)
k_sor_count(int nslot, const int32_t* __restrict__ rows, const int32_t* __restrict__ rowptr,
            const int32_t* __restrict__ col, const int32_t* __restrict__ colour, int32_t* __restrict__ lenf,
            int32_t* __restrict__ lenb, int32_t* __restrict__ dsrc, int32_t* __restrict__ wf,
            int32_t* __restrict__ wb) {
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= nslot) return;  // whole waves
    const int i = rows[q];
    int nf = 0, nb = 0, d = -1;
    if (i >= 0) {
        const int ci = colour[i];
        for (int e = rowptr[i]; e < rowptr[i + 1]; e++) {
            const int j = col[e];
            if (j == i) d = e;
            else {
                nb++;
                nf += colour[j] < ci;
            }
        }
    }
    lenf[q] = nf;
    lenb[q] = nb;
    dsrc[q] = d;
    for (int off = 32; off > 0; off >>= 1) {
        nf = max(nf, __shfl_xor(nf, off, 64));
        nb = max(nb, __shfl_xor(nb, off, 64));
    }
    if ((threadIdx.x & 63) == 0) {
        wf[q / kSlice] = nf;
        wb[q / kSlice] = nb;
    }
}

__global__ void __launch_bounds__(256)
k_sor_fill(int nslot, const int32_t* __restrict__ rows, const int32_t* __restrict__ rowptr,
           const int32_t* __restrict__ col, const int32_t* __restrict__ colour, const int32_t* __restrict__ ptrf,
           const int32_t* __restrict__ ptrb, int32_t* __restrict__ colf, int32_t* __restrict__ srcf,
           int32_t* __restrict__ colb, int32_t* __restrict__ srcb) {
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= nslot) return;
    const int i = rows[q], sl = q / kSlice;
    int f = ptrf[sl] + q % kSlice, b = ptrb[sl] + q % kSlice;
    if (i >= 0) {
        const int ci = colour[i];
        for (int e = rowptr[i]; e < rowptr[i + 1]; e++) {
            const int j = col[e];
            if (j == i) continue;
            colb[b] = j;
            srcb[b] = e;
            b += kSlice;
            if (colour[j] < ci) {
                colf[f] = j;
                srcf[f] = e;
                f += kSlice;
            }
        }
    }
    for (; f < ptrf[sl + 1]; f += kSlice) colf[f] = 0, srcf[f] = -1;
    for (; b < ptrb[sl + 1]; b += kSlice) colb[b] = 0, srcb[b] = -1;
}

// Per-block sums r.z, z.z, z.w (w may be null: z.w = 0).
template <typename V>
__global__ void __launch_bounds__(kVecBlock)
k_pc_dots(int n, const V* __restrict__ r, const V* __restrict__ z, const V* __restrict__ w,
          double* __restrict__ partials, const int* __restrict__ done_flag) {
    if (done_flag && *done_flag) return;
    double s_rz = 0.0, s_zz = 0.0, s_zw = 0.0;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const double zi = (double)z[i];
        s_rz += (double)r[i] * zi;
        s_zz += zi * zi;
        if (w) s_zw += zi * (double)w[i];
    }
    double v[3] = {s_rz, s_zz, s_zw};
    block_partials<3>(v, partials);
}

// ---------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------

static int lanes_for(const flgpu_ctx* c) {
    const double avg = (double)c->nnz / std::max(1, c->rows);
    if (avg <= 6) return 4;
    if (avg <= 12) return 8;
    if (avg <= 24) return 16;
    if (avg <= 48) return 32;
    return 64;
}

static int spmv_grid(const flgpu_ctx* c) {
    return c->kw->sell.nsl ? sell_grid(c->kw->sell.nsl) : stream_grid(c->kw->nrb);
}

// The sliced ELL values matching a CSR value array of the solver matrix
// (null for any other array, which takes the CSR product).
static const double* sell_values(const KrylovWork* k, const double* val) {
    return k->sell.nsl && val == k->val64.p ? k->sval64.p : nullptr;
}
static const float* sell_values(const KrylovWork* k, const float* val) {
    return k->sell.nsl && val == k->val32.p ? k->sval32.p : nullptr;
}

template <typename V, typename CT, typename XV, typename YV>
static void sell_launch(flgpu_ctx* c, KrylovWork* k, const V* sval, const CT* col, const XV* x, YV* y,
                        const double* bsub, int want_dot, const int* done_flag) {
    const SellOp<V, CT> m = sell_op(k->sell, c->rows, sval, col);
    if (want_dot)
        sell_product<V, V, CT, XV, YV, DOT_XY>(c->stream, m, x, y, bsub, nullptr, nullptr, k->part(PART_SPMV), done_flag);
    else
        sell_product<V, V, CT, XV, YV, DOT_NONE>(c->stream, m, x, y, bsub, nullptr, nullptr, k->part(PART_SPMV),
                                                 done_flag);
}

template <typename AV, typename CT>
static CsrOp<AV, CT> matrix_op(flgpu_ctx* c, KrylovWork* k, const AV* val, const CT* col) {
    return CsrOp<AV, CT>{k->nrb, k->rb.p, k->rbk.p, c->rowptr.p, col, val, nullptr, nullptr};
}

template <typename V, typename CT, typename XV, typename YV>
static void spmv_launch(flgpu_ctx* c, KrylovWork* k, const V* val, const CT* col, const XV* x, YV* y,
                        const double* bsub, int want_dot, const int* done_flag) {
    const int grid = stream_grid(k->nrb);
    const CsrOp<V, CT> m = matrix_op<V, CT>(c, k, val, col);
    if (want_dot)
        hipLaunchKernelGGL((k_csr_stream<V, V, CT, XV, YV, DOT_XY>), dim3(grid), dim3(kRowBlock), 0, c->stream, m,
                           x, y, bsub, (const V*)nullptr, (const V*)nullptr, k->part(PART_SPMV), done_flag);
    else
        hipLaunchKernelGGL((k_csr_stream<V, V, CT, XV, YV, DOT_NONE>), dim3(grid), dim3(kRowBlock), 0, c->stream,
                           m, x, y, bsub, (const V*)nullptr, (const V*)nullptr, k->part(PART_SPMV), done_flag);
}

// y = A x (or y = bsub - A x); with want_dot the per-block sums x.y, y.y
// go to the PART_SPMV region, spmv_grid(c) of them.  The column indices
// are the int16 offsets when they fit.
template <typename V, typename XV, typename YV>
static int spmv(flgpu_ctx* c, KrylovWork* k, const V* val, const XV* x, YV* y, const double* bsub,
                int want_dot, const int* done_flag) {
    if (const V* sv = sell_values(k, val)) {
        if (k->sell.use16)
            sell_launch<V, int16_t, XV, YV>(c, k, sv, k->sell.col16.p, x, y, bsub, want_dot, done_flag);
        else
            sell_launch<V, int32_t, XV, YV>(c, k, sv, k->sell.col32.p, x, y, bsub, want_dot, done_flag);
    } else if (k->use16)
        spmv_launch<V, int16_t, XV, YV>(c, k, val, k->col16.p, x, y, bsub, want_dot, done_flag);
    else
        spmv_launch<V, int32_t, XV, YV>(c, k, val, c->col.p, x, y, bsub, want_dot, done_flag);
    FLGPU_HIP(hipGetLastError());
    return FLGPU_OK;
}

// The sliced ELL plan of the solver matrix, where sell_order gives it one
// (FLGPU_SPMV=csr keeps the CSR products throughout).
static int sell_setup(flgpu_ctx* c, KrylovWork* k) {
    const char* e = getenv("FLGPU_SPMV");
    k->sell.release();
    k->sval64.release();
    k->sval32.release();
    if (e && std::string(e) == "csr") return FLGPU_OK;
    const SellOrder order = sell_order(c->h_rowptr.data(), c->rows);
    if (order == SELL_NONE) return FLGPU_OK;
    return sell_build(c->stream, c->rows, c->nnz, c->rowptr.p, c->col.p, nullptr, order == SELL_SORTED, k->sell);
}

static int ensure_work(flgpu_ctx* c, bool mixed) {
    if (!c->kw) c->kw = new KrylovWork();
    KrylovWork* k = c->kw;
    const int n = c->rows;
    if (k->n != n || k->nnz != c->nnz) {
        k->n = n;
        k->nnz = c->nnz;
        k->have_x = false;
    }
    FLGPU_TRY(k->val64.alloc(c->nnz));
    FLGPU_TRY(k->b.alloc(n));
    FLGPU_TRY(k->x.alloc(n));
    FLGPU_TRY(k->r.alloc(n));
    FLGPU_TRY(k->z.alloc(n));
    FLGPU_TRY(k->p.alloc(n));
    FLGPU_TRY(k->w.alloc(n));
    FLGPU_TRY(k->dinv.alloc(n));
    FLGPU_TRY(k->y.alloc(n));
    FLGPU_TRY(k->rt.alloc(n));
    if (mixed) {
        FLGPU_TRY(k->rt32.alloc(n));
        FLGPU_TRY(k->val32.alloc(c->nnz));
        FLGPU_TRY(k->r32.alloc(n));
        FLGPU_TRY(k->z32.alloc(n));
        FLGPU_TRY(k->p32.alloc(n));
        FLGPU_TRY(k->w32.alloc(n));
        FLGPU_TRY(k->dinv32.alloc(n));
        FLGPU_TRY(k->y32.alloc(n));
    }
    FLGPU_TRY(k->partials.reserve((size_t)kPartStride * PART_COMPONENTS));
    if (k->rb_key != c->sparsity_gen) {
        std::vector<int32_t> rb, rbk;
        stream_row_blocks(c->h_rowptr.data(), n, rb, rbk);
        FLGPU_TRY(k->rb.upload(rb.data(), rb.size(), c->stream));
        FLGPU_TRY(k->rbk.upload(rbk.data(), rbk.size(), c->stream));
        std::vector<int16_t> c16;
        k->use16 = compress_columns(c->h_rowptr.data(), c->h_col.data(), rb, c16);
        if (k->use16) FLGPU_TRY(k->col16.upload(c16.data(), c16.size(), c->stream));
        else k->col16.release();
        FLGPU_HIP(hipStreamSynchronize(c->stream));  // rb and c16 are freed on return
        k->nrb = (int)rb.size() - 1;
        FLGPU_TRY(sell_setup(c, k));
        k->rb_key = c->sparsity_gen;
    }
    if (k->sell.nsl) {
        FLGPU_TRY(k->sval64.alloc((size_t)k->sell.nslot));
        if (mixed) FLGPU_TRY(k->sval32.alloc((size_t)k->sell.nslot));
    }
    FLGPU_TRY(k->scal.alloc(2));
    if (!k->h_scal) {
        FLGPU_HIP(hipHostMalloc((void**)&k->h_scal, sizeof(Scal) + sizeof(int64_t),
                                hipHostMallocMapped | hipHostMallocCoherent));
        k->h_scal_owned = true;
        k->word = reinterpret_cast<int64_t*>(k->h_scal + 1);
        void* d = nullptr;
        FLGPU_HIP(hipHostGetDevicePointer(&d, k->h_scal, 0));
        k->d_word = reinterpret_cast<int64_t*>(static_cast<Scal*>(d) + 1);
    }
    k->nblk = (int)std::min<int64_t>(kMaxVecGrid, (n + kVecBlock - 1) / kVecBlock);
    k->nblk = std::max(k->nblk, 1);
    return FLGPU_OK;
}

static int read_scal(flgpu_ctx* c, KrylovWork* k) {
    FLGPU_HIP(hipMemcpyAsync(k->h_scal, k->S(), sizeof(Scal), hipMemcpyDeviceToHost, c->stream));
    FLGPU_HIP(hipStreamSynchronize(c->stream));
    return FLGPU_OK;
}

static int write_scal(flgpu_ctx* c, KrylovWork* k) {
    FLGPU_HIP(hipMemcpyAsync(k->S(), k->h_scal, sizeof(Scal), hipMemcpyHostToDevice, c->stream));
    // a pageable host copy is read by the copy after the call returns
    if (!k->h_scal_owned) FLGPU_HIP(hipStreamSynchronize(c->stream));
    return FLGPU_OK;
}

static int finalize(flgpu_ctx* c, KrylovWork* k, int op, int region, int nparts, bool jacobi, bool norm0) {
    hipLaunchKernelGGL(k_finalize, dim3(1), dim3(kVecBlock), 0, c->stream, op, k->part(region), nparts,
                       jacobi ? 1 : 0, norm0 ? 1 : 0, k->S());
    FLGPU_HIP(hipGetLastError());
    return FLGPU_OK;
}

// Build the reduced (PETSc-side) system from the assembled one.
static int build_reduced(flgpu_ctx* c, KrylovWork* k, bool mixed, bool zero_x) {
    const int n = c->rows;
    hipLaunchKernelGGL(k_diag_minmax, dim3(k->nblk), dim3(kVecBlock), 0, c->stream, n, c->diag.p, c->A.p,
                       k->part(PART_MISC));
    hipLaunchKernelGGL(k_pivot, dim3(1), dim3(64), 0, c->stream, k->nblk, k->part(PART_MISC), k->S());
    hipLaunchKernelGGL(k_build, dim3(stream_grid(k->nrb)), dim3(kRowBlock), 0, c->stream, k->nrb, k->rb.p,
                       c->rowptr.p, c->col.p, c->A.p, c->rhs.p, c->inactive.p, c->have_inactive ? 1 : 0, k->S(),
                       k->val64.p, mixed ? k->val32.p : nullptr, k->b.p, k->dinv.p, mixed ? k->dinv32.p : nullptr,
                       k->x.p, zero_x ? 1 : 0);
    if (k->sell.nsl) {
        const SellPlan& p = k->sell;
        const unsigned g = grid_for(p.nslot, 256);
        hipLaunchKernelGGL((k_sell_gather<double, double>), dim3(g), dim3(256), 0, c->stream, p.nslot, p.src.p,
                           k->val64.p, k->sval64.p);
        if (mixed)
            hipLaunchKernelGGL((k_sell_gather<float, float>), dim3(g), dim3(256), 0, c->stream, p.nslot, p.src.p,
                               k->val32.p, k->sval32.p);
    }
    FLGPU_HIP(hipGetLastError());
    return FLGPU_OK;
}

// x += dx; dx = 0 (the mixed solves' FP32 increment into the FP64 solution)
__global__ void __launch_bounds__(kVecBlock)
k_fold_x(int n, double* __restrict__ x, float* __restrict__ dx) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        x[i] = x[i] + (double)dx[i];
        dx[i] = 0.f;
    }
}

// True residual r64 = b - A x (FP64) and its squared norm in scal.true_rr.
static int true_residual(flgpu_ctx* c, KrylovWork* k) {
    if (k->dx_on) {
        hipLaunchKernelGGL(k_fold_x, dim3(k->nblk), dim3(kVecBlock), 0, c->stream, c->rows, k->x.p, k->dx32.p);
        FLGPU_HIP(hipGetLastError());
    }
    FLGPU_TRY((spmv<double, double, double>(c, k, k->val64.p, k->x.p, k->r.p, k->b.p, 1, nullptr)));
    return finalize(c, k, FIN_TRUE_RR, PART_SPMV, spmv_grid(c), false, false);
}

static int norm_b(flgpu_ctx* c, KrylovWork* k) {
    hipLaunchKernelGGL(k_dot2, dim3(k->nblk), dim3(kVecBlock), 0, c->stream, c->rows, k->b.p, k->part(PART_MISC));
    return finalize(c, k, FIN_BB, PART_MISC, k->nblk, false, false);
}

// ------------------------- multicolour SSOR ------------------------------

// First-fit colouring of the rows of a CSR pattern in row order: row i
// takes the smallest colour that none of its columns j < i holds.  Rows are
// then listed colour by colour, ascending inside a colour.
static void colour_rows(int n, const int32_t* rowptr, const int32_t* col, std::vector<int32_t>& ptr,
                        std::vector<int32_t>& rows, std::vector<int32_t>& colour) {
    std::vector<int32_t> mark;  // mark[q] == i: colour q is taken next to row i
    colour.assign(n, -1);
    int ncol = 0;
    for (int i = 0; i < n; i++) {
        for (int k = rowptr[i]; k < rowptr[i + 1]; k++) {
            const int j = col[k];
            if (j < 0 || j >= i) continue;
            const int q = colour[j];
            if (q >= (int)mark.size()) mark.resize(q + 1, -1);
            mark[q] = i;
        }
        int q = 0;
        while (q < (int)mark.size() && mark[q] == i) q++;
        colour[i] = q;
        ncol = std::max(ncol, q + 1);
    }
    ptr.assign(ncol + 1, 0);
    for (int i = 0; i < n; i++) ptr[colour[i] + 1]++;
    for (int c = 0; c < ncol; c++) ptr[c + 1] += ptr[c];
    rows.resize(n);
    std::vector<int32_t> pos(ptr.begin(), ptr.end() - 1);
    for (int i = 0; i < n; i++) rows[pos[colour[i]]++] = i;
}

// One workgroup takes the sweeps when z fits its LDS and reading the entries
// through one CU (about 120 GB/s) plus a barrier per step (0.8 us) costs less
// than a launch per step (4 us).
constexpr size_t kSorLds = 128 << 10;
constexpr int kSorWindow = 2048;  // rows of a colour that are sorted by length together

// Rows longest first, equal ones in order (a counting sort).
static void sort_by_length(const int32_t* rowptr, int32_t* rows, int n, std::vector<int32_t>& count,
                           std::vector<int32_t>& tmp) {
    int top = 0;
    for (int t = 0; t < n; t++) top = std::max(top, rowptr[rows[t] + 1] - rowptr[rows[t]]);
    count.assign((size_t)top + 2, 0);  // count[d + 1]: rows that are d shorter than the longest
    for (int t = 0; t < n; t++) count[top - (rowptr[rows[t] + 1] - rowptr[rows[t]]) + 1]++;
    for (int d = 0; d < top; d++) count[d + 1] += count[d];
    tmp.assign(rows, rows + n);
    for (int t = 0; t < n; t++) rows[count[top - (rowptr[tmp[t] + 1] - rowptr[tmp[t]])]++] = tmp[t];
}

static int ssor_plan(flgpu_ctx* c, KrylovWork* k) {
    if (!c->all_diag) return set_error(FLGPU_EUNSUPPORTED, "sor preconditioner: a row has no diagonal entry");
    const int n = c->rows;
    if (c->cols > n) return set_error(FLGPU_EUNSUPPORTED, "sor preconditioner: a column past the rows");
    const int32_t *rp = c->h_rowptr.data(), *cl = c->h_col.data();
    std::vector<int32_t> cp, order, colour, rows, count, tmp;
    colour_rows(n, rp, cl, cp, order, colour);
    const int ncol = (int)cp.size() - 1;
    // slices: a colour's rows in order, longest first inside windows of kSorWindow
    k->mc_ptr.assign(1, 0);
    rows.reserve((size_t)n + (size_t)ncol * kSlice);
    for (int q = 0; q < ncol; q++) {
        for (int t = cp[q]; t < cp[q + 1]; t += kSorWindow)
            sort_by_length(rp, order.data() + t, std::min(cp[q + 1] - t, kSorWindow), count, tmp);
        rows.insert(rows.end(), order.begin() + cp[q], order.begin() + cp[q + 1]);
        rows.resize((rows.size() + kSlice - 1) / kSlice * kSlice, -1);
        k->mc_ptr.push_back((int32_t)(rows.size() / kSlice));
    }
    const int nslot = (int)rows.size(), nsl = nslot / kSlice;
    KrylovWork::SorHalf *F = &k->mc_f, *B = &k->mc_b;
    DevBuf<int32_t> dcolour, width;
    FLGPU_TRY(dcolour.upload(colour.data(), colour.size(), c->stream));
    FLGPU_TRY(width.alloc(2 * (size_t)nsl));
    FLGPU_TRY(k->mc_rows.upload(rows.data(), rows.size(), c->stream));
    FLGPU_TRY(k->mc_cptr.upload(k->mc_ptr.data(), k->mc_ptr.size(), c->stream));
    FLGPU_TRY(k->mc_dsrc.alloc(rows.size()));
    FLGPU_TRY(F->len.alloc(rows.size()));
    FLGPU_TRY(B->len.alloc(rows.size()));
    const unsigned grid = grid_for(nslot, 256);
    hipLaunchKernelGGL(k_sor_count, dim3(grid), dim3(256), 0, c->stream, nslot, k->mc_rows.p, c->rowptr.p, c->col.p,
                       dcolour.p, F->len.p, B->len.p, k->mc_dsrc.p, width.p, width.p + nsl);
    FLGPU_HIP(hipGetLastError());
    std::vector<int32_t> w(2 * (size_t)nsl), ptr[2];
    FLGPU_HIP(hipMemcpyAsync(w.data(), width.p, sizeof(int32_t) * w.size(), hipMemcpyDeviceToHost, c->stream));
    FLGPU_HIP(hipStreamSynchronize(c->stream));
    int64_t slots = 0;
    for (int half = 0; half < 2; half++) {
        int64_t at = 0;
        ptr[half].assign(1, 0);
        for (int sl = 0; sl < nsl; sl++) {
            at += (int64_t)w[half * nsl + sl] * kSlice;
            ptr[half].push_back((int32_t)at);
        }
        if (at > INT32_MAX)
            return set_error(FLGPU_EUNSUPPORTED, "sor preconditioner: %lld slots of entries", (long long)at);
        KrylovWork::SorHalf& H = half ? k->mc_b : k->mc_f;
        FLGPU_TRY(H.ptr.upload(ptr[half].data(), ptr[half].size(), c->stream));
        FLGPU_TRY(H.col.alloc((size_t)at));
        FLGPU_TRY(H.src.alloc((size_t)at));
        slots += at;
    }
    hipLaunchKernelGGL(k_sor_fill, dim3(grid), dim3(256), 0, c->stream, nslot, k->mc_rows.p, c->rowptr.p, c->col.p,
                       dcolour.p, F->ptr.p, B->ptr.p, F->col.p, F->src.p, B->col.p, B->src.p);
    FLGPU_HIP(hipGetLastError());
    FLGPU_HIP(hipStreamSynchronize(c->stream));  // the vectors and dcolour are freed here
    const double steps = 2.0 * ncol - 1.0;
    k->mc_one = sizeof(double) * (size_t)n <= kSorLds && 12.0 * (double)slots / 120e3 + 0.8 * steps < 4.0 * steps;
    if (k->mc_one)
        for (const void* f : {(const void*)&k_sor_block<double>, (const void*)&k_sor_block<float>})
            FLGPU_HIP(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kSorLds));
    k->mc_key = c->sparsity_gen;
    return FLGPU_OK;
}

template <typename V>
static const V* sor_values(KrylovWork::SorHalf& h);
template <>
const double* sor_values<double>(KrylovWork::SorHalf& h) { return h.v64.p; }
template <>
const float* sor_values<float>(KrylovWork::SorHalf& h) { return h.v32.p; }

// The plan of the sparsity, and the reduced values in its slots.
template <typename V>
static int ssor_prepare(flgpu_ctx* c, KrylovWork* k, const V* val) {
    if (k->mc_key != c->sparsity_gen) FLGPU_TRY(ssor_plan(c, k));
    auto gather = [&](const DevBuf<int32_t>& src, auto& out) -> int {
        FLGPU_TRY(out.alloc(src.n));
        if (src.n)
            hipLaunchKernelGGL((k_sell_gather<V, V>), dim3(grid_for((int64_t)src.n, 256)), dim3(256), 0, c->stream,
                               (int64_t)src.n, src.p, val, out.p);
        return FLGPU_OK;
    };
    if constexpr (std::is_same<V, double>::value) {
        FLGPU_TRY(gather(k->mc_f.src, k->mc_f.v64));
        FLGPU_TRY(gather(k->mc_b.src, k->mc_b.v64));
        FLGPU_TRY(gather(k->mc_dsrc, k->mc_d64));
    } else {
        FLGPU_TRY(gather(k->mc_f.src, k->mc_f.v32));
        FLGPU_TRY(gather(k->mc_b.src, k->mc_b.v32));
        FLGPU_TRY(gather(k->mc_dsrc, k->mc_d32));
    }
    FLGPU_HIP(hipGetLastError());
    return FLGPU_OK;
}

// z = M^-1 r (the forward and backward sweeps); with done_flag set the
// kernels return at once.
template <typename V>
static int ssor_sweeps(flgpu_ctx* c, KrylovWork* k, const V* r, V* z, const int* done_flag) {
    const int ncol = (int)k->mc_ptr.size() - 1;
    const V* dia;
    if constexpr (std::is_same<V, double>::value) dia = k->mc_d64.p;
    else dia = k->mc_d32.p;
    const SorOp<V> f{k->mc_rows.p, k->mc_f.ptr.p, k->mc_f.len.p, k->mc_f.col.p, sor_values<V>(k->mc_f), dia};
    const SorOp<V> b{k->mc_rows.p, k->mc_b.ptr.p, k->mc_b.len.p, k->mc_b.col.p, sor_values<V>(k->mc_b), dia};
    if (k->mc_one) {
        hipLaunchKernelGGL((k_sor_block<V>), dim3(1), dim3(1024), sizeof(V) * (size_t)c->rows, c->stream, c->rows,
                           ncol, k->mc_cptr.p, f, b, r, z, done_flag);
        FLGPU_HIP(hipGetLastError());
        return FLGPU_OK;
    }
    auto sweep = [&](const SorOp<V>& m, int q) {
        const int s0 = k->mc_ptr[q], s1 = k->mc_ptr[q + 1];
        if (s1 > s0)
            hipLaunchKernelGGL((k_sor_slices<V>), dim3((s1 - s0 + 3) / 4), dim3(256), 0, c->stream, m, s0, s1, r, z,
                               done_flag);
    };
    for (int q = 0; q < ncol; q++) sweep(f, q);
    for (int q = ncol - 2; q >= 0; q--) sweep(b, q);
    FLGPU_HIP(hipGetLastError());
    return FLGPU_OK;
}

template <typename V>
static int ssor_apply(flgpu_ctx* c, KrylovWork* k, const V* r, V* z, const V* w, double* partials,
                      int* nparts, const int* done_flag) {
    FLGPU_TRY(ssor_sweeps<V>(c, k, r, z, done_flag));
    hipLaunchKernelGGL((k_pc_dots<V>), dim3(k->nblk), dim3(kVecBlock), 0, c->stream, c->rows, r, z, w, partials,
                       done_flag);
    FLGPU_HIP(hipGetLastError());
    *nparts = k->nblk;
    return FLGPU_OK;
}

// ------------------------- (F)PCG ----------------------------------------

template <typename V>
struct CgVecs {
    V *r, *z, *p, *w, *dinv, *y, *rt;
    const V* val;
    V* s = nullptr;  // single-reduction CG only
    V* xw = nullptr; // what the vector kernels add alpha p to: x, or the FP32 increment
};

template <typename V>
static CgVecs<V> cg_vecs(KrylovWork* k);
template <>
CgVecs<double> cg_vecs<double>(KrylovWork* k) {
    return {k->r.p, k->z.p, k->p.p, k->w.p, k->dinv.p, k->y.p, k->rt.p, k->val64.p};
}
template <>
CgVecs<float> cg_vecs<float>(KrylovWork* k) {
    return {k->r32.p, k->z32.p, k->p32.p, k->w32.p, k->dinv32.p, k->y32.p, k->rt32.p, k->val32.p};
}

// The preconditioner of a (F)PCG iteration: the diagonal (Jacobi, or the
// identity as a unit diagonal), applied inside the vector kernels; or the
// learned factor or the multicolour SSOR sweeps, applied by kernels of their
// own after the residual update.
enum PcMode { PCM_DIAG = 0, PCM_LEARNED = 1, PCM_SSOR = 2 };

// z = M^-1 r for the learned factor (z = G^T (G r)) or SSOR; the per-block
// sums r.z, z.z, z.w (w = A p of this iteration) go to the PART_PC region.
// Returns the number of partial sums in *nparts.
template <typename V>
static int pc_apply(flgpu_ctx* c, KrylovWork* k, const CgVecs<V>& v, PcMode mode, const int* done_flag,
                    int* nparts) {
    if (mode == PCM_SSOR) return ssor_apply<V>(c, k, v.r, v.z, v.w, k->part(PART_PC), nparts, done_flag);
    return learned_precond_apply<V>(c, v.r, v.rt, v.z, v.y, v.w, k->part(PART_PC), nparts, done_flag);
}

// r = b - A x (FP64), r_V = r, z = M^-1 r with the sums r.z, r.r, z.z
// (and the initial norm when norm0) in the current scalar slot.
template <typename V>
static int restart_residual(flgpu_ctx* c, KrylovWork* k, const CgVecs<V>& v, PcMode mode, bool norm0,
                            bool recompute) {
    if (recompute) FLGPU_TRY(true_residual(c, k));
    const bool diag = mode == PCM_DIAG;
    const float* dsc = mode == PCM_LEARNED ? learned_scale(c) : nullptr;
    hipLaunchKernelGGL((k_restart_vecs<V>), dim3(k->nblk), dim3(kVecBlock), 0, c->stream, c->rows, k->r.p,
                       v.r, v.z, v.dinv, diag ? 1 : 0, dsc, v.rt, k->part(PART_VEC));
    FLGPU_HIP(hipGetLastError());
    FLGPU_TRY(finalize(c, k, FIN_RESTART, PART_VEC, k->nblk, diag, norm0 && diag));
    if (!diag) {
        int np = 0;
        FLGPU_TRY(pc_apply<V>(c, k, v, mode, nullptr, &np));
        k->npc = np;
        FLGPU_TRY(finalize(c, k, FIN_LEARNED, PART_PC, np, false, norm0));
    }
    return FLGPU_OK;
}

// The x the (F)PCG vector kernels update: FP64 x itself, or (mixed) the
// FP32 increment dx, zeroed here and added to x by every true residual
// (true_residual folds it first), so x is whole at each replacement and
// at the end of the solve.  (The single-reduction CG keeps its updates in
// FP64: with the FP32 increment its counts rose by 5-9% on the 3-D
// systems, against about 1 for (F)PCG.)
template <typename V>
static int x_work(flgpu_ctx* c, KrylovWork* k, CgVecs<V>& v) {
    if constexpr (std::is_same<V, float>::value) {
        FLGPU_TRY(k->dx32.alloc(c->rows));
        hipLaunchKernelGGL((k_fill<float>), dim3(k->nblk), dim3(kVecBlock), 0, c->stream, c->rows, 0.0f, k->dx32.p);
        FLGPU_HIP(hipGetLastError());
        v.xw = k->dx32.p;
        k->dx_on = true;
    } else {
        v.xw = k->x.p;
        k->dx_on = false;
    }
    return FLGPU_OK;
}

template <typename V>
static int cg_restart(flgpu_ctx* c, KrylovWork* k, const CgVecs<V>& v, PcMode mode, bool set_norm0) {
    FLGPU_TRY(restart_residual<V>(c, k, v, mode, set_norm0, true));
    hipLaunchKernelGGL((k_copy<V>), dim3(k->nblk), dim3(kVecBlock), 0, c->stream, c->rows, (const V*)v.z, v.p);
    FLGPU_HIP(hipGetLastError());
    return FLGPU_OK;
}

// True when every given array (null ones aside) starts on a multiple of R
// of its entries: the vector kernels then load R rows at once.
template <int R, typename... P>
static bool rows_aligned(const P*... ptrs) {
    return ((ptrs == nullptr || reinterpret_cast<uintptr_t>(ptrs) % (R * sizeof(P)) == 0) && ...);
}

// One (F)PCG iteration: w = A p; update x, r, z; [z = M^-1 r]; test,
// beta, p.  Four kernels (diagonal), six (learned) or 2C + 3 (SSOR over C
// colours), no host round trip.
template <typename V>
static int cg_iteration(flgpu_ctx* c, KrylovWork* k, const CgVecs<V>& v, PcMode mode) {
    const bool diag = mode == PCM_DIAG;
    FLGPU_TRY((spmv<V, V, V>(c, k, v.val, v.p, v.w, nullptr, 1, &k->S()->done)));
    Scal* in = k->S();
    k->cur ^= 1;
    const float* dsc = mode == PCM_LEARNED ? learned_scale(c) : nullptr;
    constexpr int R = 16 / sizeof(V);
    if (rows_aligned<R>(v.xw, v.p, v.r, v.w, v.z, v.dinv, dsc, v.rt))
        hipLaunchKernelGGL((k_cg_update<V, R>), dim3(k->nblk), dim3(kVecBlock), 0, c->stream, c->rows, v.xw, v.p,
                           v.r, v.w, v.z, v.dinv, diag ? 1 : 0, dsc, v.rt, k->part(PART_SPMV), spmv_grid(c),
                           k->part(PART_VEC), in, k->S());
    else
        hipLaunchKernelGGL((k_cg_update<V, 1>), dim3(k->nblk), dim3(kVecBlock), 0, c->stream, c->rows, v.xw, v.p,
                           v.r, v.w, v.z, v.dinv, diag ? 1 : 0, dsc, v.rt, k->part(PART_SPMV), spmv_grid(c),
                           k->part(PART_VEC), in, k->S());
    int npc = 0;
    if (!diag) FLGPU_TRY(pc_apply<V>(c, k, v, mode, &k->S()->done, &npc));
    in = k->S();
    k->cur ^= 1;
    if (rows_aligned<R>(v.z, v.p))
        hipLaunchKernelGGL((k_cg_p<V, R>), dim3(k->nblk), dim3(kVecBlock), 0, c->stream, c->rows, v.z, v.p,
                           k->part(PART_VEC), k->nblk, diag ? nullptr : k->part(PART_PC), npc, in, k->S(), k->pub);
    else
        hipLaunchKernelGGL((k_cg_p<V, 1>), dim3(k->nblk), dim3(kVecBlock), 0, c->stream, c->rows, v.z, v.p,
                           k->part(PART_VEC), k->nblk, diag ? nullptr : k->part(PART_PC), npc, in, k->S(), k->pub);
    FLGPU_HIP(hipGetLastError());
    return FLGPU_OK;
}

// Waits until a word that the device writes (2 its + done) has reached `its`
// or says done; a stream that ran dry or failed before that ends the wait.  The
// stream is asked some ms apart: a query puts a marker into a busy one, and
// asked every 4096 looks it made iterations 1 to 4 us longer.
static int wait_word(flgpu_ctx* c, const int64_t* word, int64_t its) {
    for (unsigned spin = 1;; spin++) {
        const int64_t w = __atomic_load_n(word, __ATOMIC_ACQUIRE);
        if ((w & 1) || w / 2 >= its) return FLGPU_OK;
        __builtin_ia32_pause();
        if (spin % (1u << 16) == 0) {
            const hipError_t e = hipStreamQuery(c->stream);
            if (e == hipErrorNotReady) continue;
            FLGPU_HIP(e);
            const int64_t w2 = __atomic_load_n(word, __ATOMIC_ACQUIRE);
            if ((w2 & 1) || w2 / 2 >= its) return FLGPU_OK;
            return set_error(FLGPU_EHIP, "flgpu_solve: stopped at iteration %lld of %lld", (long long)(w2 / 2),
                             (long long)its);
        }
    }
}

// The CG loops queue check_every iterations between two looks at the scalars;
// the ones past the last return at once, but each is three launches or more
// (8 us; with sor 2C + 3).  So the host stays at most kCgAhead iterations
// ahead of the device and queues none once that is done.  Before iteration q
// of a batch that began at iteration `its`: true if it is still wanted.  (The
// single-reduction CG counts an iteration when the next one begins.)  Solves
// of 17 iterations, 1681 rows: Jacobi 574 -> 395 us, sor 1039 -> 714 us.  Past
// kCgPublish iterations what is left over is small beside the solve, and only
// the sor sweeps' iterations, of many launches, are still published (0.3 us
// each: 0.5% of a solve of 538 on 1.37M rows).
constexpr int kCgAhead = 4, kCgPublish = 64;

static int cg_ahead(flgpu_ctx* c, KrylovWork* k, PcMode mode, int64_t its, int q, bool* wanted) {
    *wanted = true;
    if (q == 0) {  // nothing is in flight
        k->pub = its < kCgPublish || mode == PCM_SSOR ? k->d_word : nullptr;
        if (k->pub) __atomic_store_n(k->word, 2 * its, __ATOMIC_RELEASE);
        return FLGPU_OK;
    }
    if (!k->pub) return FLGPU_OK;
    FLGPU_TRY(wait_word(c, k->word, its + q - kCgAhead));
    *wanted = !(__atomic_load_n(k->word, __ATOMIC_ACQUIRE) & 1);
    return FLGPU_OK;
}

template <typename V>
static int run_cg(flgpu_ctx* c, const flgpu_solver_params* sp, flgpu_solve_info* info, bool learned) {
    KrylovWork* k = c->kw;
    const bool mixed = std::is_same<V, float>::value;
    CgVecs<V> v = cg_vecs<V>(k);
    FLGPU_TRY(x_work<V>(c, k, v));
    PcMode mode = learned ? PCM_LEARNED : sp->pc == FLGPU_PC_SOR ? PCM_SSOR : PCM_DIAG;
    bool use_learned = learned;
    const int check_every = sp->check_every > 0 ? sp->check_every : 16;
    const double stall_factor = sp->stall_factor > 0 ? sp->stall_factor : 0.9;
    const int stall_window = sp->stall_window > 0 ? sp->stall_window : 50;

    // identity preconditioner = Jacobi with dinv = 1: handled by the
    // "jacobi" kernels when pc == NONE by filling dinv with ones
    if (!learned && sp->pc == FLGPU_PC_NONE) {
        hipLaunchKernelGGL((k_fill<double>), dim3(k->nblk), dim3(kVecBlock), 0, c->stream, c->rows, 1.0, k->dinv.p);
        if (mixed)
            hipLaunchKernelGGL((k_fill<float>), dim3(k->nblk), dim3(kVecBlock), 0, c->stream, c->rows, 1.0f,
                               k->dinv32.p);
        FLGPU_HIP(hipGetLastError());
    }
    if (mode == PCM_SSOR) FLGPU_TRY(ssor_prepare<V>(c, k, v.val));
    Scal& h = *k->h_scal;
    // keep the pivot computed by build_reduced
    FLGPU_TRY(read_scal(c, k));
    {
        const double pivot = h.pivot, dmin = h.dmin, dmax = h.dmax;
        std::memset(&h, 0, sizeof h);
        h.pivot = pivot;
        h.dmin = dmin;
        h.dmax = dmax;
    }
    h.max_its = sp->max_its > 0 ? sp->max_its : 10000;
    h.rtol = sp->rtol;
    h.atol = sp->atol;
    h.norm_type = sp->norm_type;
    h.flexible = (use_learned || sp->ksp == FLGPU_KSP_FCG) ? 1 : 0;
    FLGPU_TRY(write_scal(c, k));
    FLGPU_TRY(norm_b(c, k));
    FLGPU_TRY(cg_restart<V>(c, k, v, mode, true));
    FLGPU_TRY(read_scal(c, k));
    info->refinements = 0;
    info->fallback = 0;
    const double bnorm = std::sqrt(h.bb);
    if (h.last_norm == 0.0 || h.last_norm <= sp->atol) {
        // converged before the first iteration: the device copy of the
        // scalars is what the solve reports from, so it gets the reason too
        h.reason = KSP_CONVERGED_ATOL;
        h.done = 1;
        FLGPU_TRY(write_scal(c, k));
    }
    double rmax = std::sqrt(h.rr);          // reliable-update reference
    const double delta = 0.1;
    int window_its = 0;
    double window_norm = h.last_norm;
    auto t0 = std::chrono::steady_clock::now();
    while (!h.done) {
        for (int q = 0; q < check_every; q++) {
            bool wanted;
            FLGPU_TRY(cg_ahead(c, k, mode, h.its, q, &wanted));
            if (!wanted) break;
            FLGPU_TRY(cg_iteration<V>(c, k, v, mode));
        }
        FLGPU_TRY(read_scal(c, k));
        const double rnow = std::sqrt(h.rr);
        if (mixed && (h.done ? h.reason > 0 : rnow < delta * rmax)) {
            // reliable update: replace the FP32 residual by the FP64 one
            const int reason = h.reason, done = h.done;
            FLGPU_TRY(true_residual(c, k));
            FLGPU_TRY(read_scal(c, k));
            const double tr = std::sqrt(h.true_rr);
            info->refinements++;
            const double target = std::max(sp->rtol * (sp->norm_type == FLGPU_NORM_UNPRECONDITIONED ? h.rnorm0 : bnorm),
                                           sp->atol);
            // The FP32 recurrence said converged: the FP64 true residual
            // decides (for either norm type it is the unpreconditioned
            // ||b - A x|| against rtol times ||r0|| or ||b||, the
            // criterion the solve reports in true_relres).  Short of it,
            // the iteration goes on, or at max_its the solve has diverged.
            if (done && reason > 0 && tr > target) {
                if (h.its < h.max_its) {
                    h.done = 0;
                    h.reason = 0;
                } else {
                    h.reason = KSP_DIVERGED_ITS;
                }
                FLGPU_TRY(write_scal(c, k));
            }
            if (!h.done) {
                // The FP32 recurrence drifts from the true residual by about
                // eps32 times the residual of the last replacement.  After a
                // drop of more than 1e3 since then (a fast preconditioner
                // between two host checks) that drift is no longer small
                // against r, and the old direction p is not conjugate to the
                // replaced residual: the direction restarts from z.
                const bool restart_p = rnow < 1e-3 * rmax;
                FLGPU_TRY(restart_residual<V>(c, k, v, mode, false, false));
                if (restart_p) {
                    hipLaunchKernelGGL((k_copy<V>), dim3(k->nblk), dim3(kVecBlock), 0, c->stream, c->rows,
                                       (const V*)v.z, v.p);
                    FLGPU_HIP(hipGetLastError());
                }
                FLGPU_TRY(read_scal(c, k));
                rmax = std::sqrt(h.rr);
            }
        }
        if (use_learned && !h.done) {
            window_its += check_every;
            if (window_its >= stall_window) {
                if (h.last_norm > stall_factor * window_norm) {
                    // stalled: fall back to Jacobi-PCG from the current x
                    use_learned = false;
                    mode = PCM_DIAG;
                    info->fallback = 1;
                    h.flexible = sp->ksp == FLGPU_KSP_FCG ? 1 : 0;
                    FLGPU_TRY(write_scal(c, k));
                    FLGPU_TRY(cg_restart<V>(c, k, v, PCM_DIAG, false));
                    FLGPU_TRY(read_scal(c, k));
                    rmax = std::sqrt(h.rr);
                }
                window_its = 0;
                window_norm = h.last_norm;
            }
        }
    }
    FLGPU_TRY(true_residual(c, k));
    FLGPU_TRY(read_scal(c, k));
    auto t1 = std::chrono::steady_clock::now();
    info->seconds = std::chrono::duration<double>(t1 - t0).count();
    info->its = h.its;
    info->reason = h.reason;
    info->true_relres = bnorm > 0 ? std::sqrt(h.true_rr) / bnorm : std::sqrt(h.true_rr);
    info->precond_relres = h.rnorm0 > 0 ? h.last_norm / h.rnorm0 : h.last_norm;
    return FLGPU_OK;
}

// ------------------------- single-reduction CG ---------------------------

// The restart of the single-reduction recurrence: r = b - A x (FP64), r_V,
// u = M r with gamma, r.r, u.u in the scalars (restart_residual), then
// w = A u with u.w in the PART_SPMV partials; the next iteration takes
// p = u, s = w.
template <typename V>
static int cg1_restart(flgpu_ctx* c, KrylovWork* k, const CgVecs<V>& v, PcMode mode, bool norm0, bool recompute) {
    FLGPU_TRY(restart_residual<V>(c, k, v, mode, norm0, recompute));
    return spmv<V, V, V>(c, k, v.val, v.z, v.w, nullptr, 1, &k->S()->done);
}

// One iteration: the vector update (k_cg1_vec), [the factor or SSOR
// apply], the product w = A u.  Two kernels with the diagonal
// preconditioner, four with a factor.  reg: the partial-sum region the
// previous update wrote (read here), the other one is written.
template <typename V>
static int cg1_iteration(flgpu_ctx* c, KrylovWork* k, const CgVecs<V>& v, PcMode mode, bool first, int& reg) {
    const bool diag = mode == PCM_DIAG;
    const int reg_out = reg == PART_VEC ? PART_VEC2 : PART_VEC;
    Scal* in = k->S();
    k->cur ^= 1;
    const float* dsc = mode == PCM_LEARNED ? learned_scale(c) : nullptr;
    const double* pg = diag ? k->part(reg) : k->part(PART_PC);
    const int ng = diag ? k->nblk : k->npc;
    constexpr int R = 16 / sizeof(V);
    auto launch = [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3(k->nblk), dim3(kVecBlock), 0, c->stream, c->rows, k->x.p, v.p, v.s, v.r, v.z,
                           (const V*)v.w, (const V*)v.dinv, diag ? 1 : 0, dsc, v.rt, (const double*)k->part(PART_SPMV),
                           spmv_grid(c), pg, ng, diag ? 0 : 1, (const double*)k->part(reg), k->nblk, first ? 1 : 0,
                           k->part(reg_out), (const Scal*)in, k->S(), k->pub);
    };
    if (rows_aligned<R>(k->x.p, v.p, v.s, v.r, v.z, v.w, v.dinv, dsc, v.rt))
        launch(&k_cg1_vec<V, R>);
    else
        launch(&k_cg1_vec<V, 1>);
    FLGPU_HIP(hipGetLastError());
    reg = reg_out;
    if (!diag) {
        int npc = 0;
        FLGPU_TRY(pc_apply<V>(c, k, v, mode, &k->S()->done, &npc));
        k->npc = npc;
    }
    return spmv<V, V, V>(c, k, v.val, v.z, v.w, nullptr, 1, &k->S()->done);
}

template <typename V>
static int run_cg1(flgpu_ctx* c, const flgpu_solver_params* sp, flgpu_solve_info* info, bool factor) {
    KrylovWork* k = c->kw;
    const bool mixed = std::is_same<V, float>::value;
    CgVecs<V> v = cg_vecs<V>(k);
    if (mixed) {
        FLGPU_TRY(k->s32.alloc(c->rows));
        v.s = reinterpret_cast<V*>(k->s32.p);
    } else {
        FLGPU_TRY(k->s.alloc(c->rows));
        v.s = reinterpret_cast<V*>(k->s.p);
    }
    PcMode mode = factor ? PCM_LEARNED : sp->pc == FLGPU_PC_SOR ? PCM_SSOR : PCM_DIAG;
    bool use_factor = factor;
    const int check_every = sp->check_every > 0 ? sp->check_every : 16;
    const double stall_factor = sp->stall_factor > 0 ? sp->stall_factor : 0.9;
    const int stall_window = sp->stall_window > 0 ? sp->stall_window : 50;
    if (!factor && sp->pc == FLGPU_PC_NONE) {
        hipLaunchKernelGGL((k_fill<double>), dim3(k->nblk), dim3(kVecBlock), 0, c->stream, c->rows, 1.0, k->dinv.p);
        if (mixed)
            hipLaunchKernelGGL((k_fill<float>), dim3(k->nblk), dim3(kVecBlock), 0, c->stream, c->rows, 1.0f,
                               k->dinv32.p);
        FLGPU_HIP(hipGetLastError());
    }
    if (mode == PCM_SSOR) FLGPU_TRY(ssor_prepare<V>(c, k, v.val));
    Scal& h = *k->h_scal;
    FLGPU_TRY(read_scal(c, k));
    {
        const double pivot = h.pivot, dmin = h.dmin, dmax = h.dmax;
        std::memset(&h, 0, sizeof h);
        h.pivot = pivot;
        h.dmin = dmin;
        h.dmax = dmax;
    }
    h.max_its = sp->max_its > 0 ? sp->max_its : 10000;
    h.rtol = sp->rtol;
    h.atol = sp->atol;
    h.norm_type = sp->norm_type;
    FLGPU_TRY(write_scal(c, k));
    FLGPU_TRY(norm_b(c, k));
    FLGPU_TRY(cg1_restart<V>(c, k, v, mode, true, true));
    FLGPU_TRY(read_scal(c, k));
    info->refinements = 0;
    info->fallback = 0;
    const double bnorm = std::sqrt(h.bb);
    if (h.last_norm == 0.0 || h.last_norm <= sp->atol) {
        h.reason = KSP_CONVERGED_ATOL;
        h.done = 1;
        FLGPU_TRY(write_scal(c, k));
    }
    double rmax = std::sqrt(h.rr);
    const double delta = 0.1;
    int window_its = 0;
    double window_norm = h.last_norm;
    bool first = true;
    int reg = PART_VEC;  // restart_residual's partials
    auto t0 = std::chrono::steady_clock::now();
    while (!h.done) {
        for (int q = 0; q < check_every; q++) {
            bool wanted;
            FLGPU_TRY(cg_ahead(c, k, mode, h.its, q, &wanted));
            if (!wanted) break;
            FLGPU_TRY(cg1_iteration<V>(c, k, v, mode, first, reg));
            first = false;
        }
        FLGPU_TRY(read_scal(c, k));
        const double rnow = std::sqrt(h.rr);
        if (mixed && (h.done ? h.reason > 0 : rnow < delta * rmax)) {
            // reliable update, as in the (F)PCG loop: the FP64 true residual
            // replaces the FP32 one and decides convergence
            const int reason = h.reason, done = h.done;
            FLGPU_TRY(true_residual(c, k));
            FLGPU_TRY(read_scal(c, k));
            const double tr = std::sqrt(h.true_rr);
            info->refinements++;
            const double target = std::max(sp->rtol * (sp->norm_type == FLGPU_NORM_UNPRECONDITIONED ? h.rnorm0 : bnorm),
                                           sp->atol);
            if (done && reason > 0 && tr > target) {
                if (h.its < h.max_its) {
                    h.done = 0;
                    h.reason = 0;
                } else {
                    h.reason = KSP_DIVERGED_ITS;
                }
                FLGPU_TRY(write_scal(c, k));
            }
            if (!h.done) {
                // As in the (F)PCG loop, the direction survives a drop of
                // up to 1e3 since the last replacement: s = A p is then
                // recomputed (its FP32 recurrence drifts like r's) and the
                // next update forms beta from the replaced gamma and the
                // gamma that formed p.  After a larger drop the recurrence
                // restarts from the replaced residual (p = u, s = w); the
                // update that follows tests no residual, so the count takes
                // the replaced one here.
                const bool restart_p = rnow < 1e-3 * rmax;
                const double rz_p = h.rz;
                if (!restart_p) FLGPU_TRY((spmv<V, V, V>(c, k, v.val, v.p, v.s, nullptr, 0, &k->S()->done)));
                FLGPU_TRY(cg1_restart<V>(c, k, v, mode, false, false));
                FLGPU_TRY(read_scal(c, k));
                if (restart_p)
                    h.its += 1;
                else
                    h.rz = rz_p;
                FLGPU_TRY(write_scal(c, k));
                first = restart_p;
                reg = PART_VEC;
                rmax = std::sqrt(h.rr);
            }
        }
        if (use_factor && !h.done) {
            window_its += check_every;
            if (window_its >= stall_window) {
                if (h.last_norm > stall_factor * window_norm) {
                    use_factor = false;
                    mode = PCM_DIAG;
                    info->fallback = 1;
                    FLGPU_TRY(write_scal(c, k));
                    FLGPU_TRY(cg1_restart<V>(c, k, v, PCM_DIAG, false, true));
                    FLGPU_TRY(read_scal(c, k));
                    h.its += 1;
                    FLGPU_TRY(write_scal(c, k));
                    first = true;
                    reg = PART_VEC;
                    rmax = std::sqrt(h.rr);
                }
                window_its = 0;
                window_norm = h.last_norm;
            }
        }
    }
    FLGPU_TRY(true_residual(c, k));
    FLGPU_TRY(read_scal(c, k));
    auto t1 = std::chrono::steady_clock::now();
    info->seconds = std::chrono::duration<double>(t1 - t0).count();
    info->its = h.its;
    info->reason = h.reason;
    info->true_relres = bnorm > 0 ? std::sqrt(h.true_rr) / bnorm : std::sqrt(h.true_rr);
    info->precond_relres = h.rnorm0 > 0 ? h.last_norm / h.rnorm0 : h.last_norm;
    return FLGPU_OK;
}

// ------------------------- GMRES ------------------------------------------
//
// Restarted GMRES with left preconditioning and classical Gram-Schmidt done
// twice, driven from the device: the Hessenberg column, its Givens rotations
// and the convergence test are taken by one wave beside the next iteration's
// dot products, so an iteration is four kernels and no host round trip:
//   k_gm_sell / k_gm_csr  normalises the last w into basis vector v_k and
//                         forms w = D^-1 A v_k (SSOR: A v_k, then the sweeps)
//   k_gm_dots             h1_j = w . v_j; one more workgroup closes the
//                         column before this one
//   k_gm_orth<.., DOTS>   w -= sum h1_j v_j and, from the same registers,
//                         h2_j = w . v_j (the second pass's coefficients)
//   k_gm_orth<.., NORM>   w -= sum h2_j v_j and |w|^2
// The basis is read three times an iteration instead of five, and the sums
// over blocks are taken by every consumer block in the same fixed order.
// The iteration counter and the done flag reach the host through a word in
// pinned memory, which it polls a few iterations behind what it has queued.
// What bounds it: small systems, the chain of four launches (each two or
// three dependent memory round trips, 4-7 us); large ones, reading the basis
// (17 to 30 vectors of 373k rows: 15-17 us a pass, 4.2 to 4.7 TB/s).  A column
// is closed beside the next iteration's dot products, so a solve runs one
// product (and one pair of sweeps) past the last column.  Whole time steps on
// one MI355X, with ten launches and three waits for the host an iteration and
// now (the sliced products' share included): 64 x 64 P1 triangles, 17
// iterations, 2.08 -> 0.62 ms; 71^3 x 6 P1 tetrahedra, 29 iterations, 5.87 ->
// 2.77 ms; 40^3 x 6 P2, 52 iterations, 14.4 -> 7.4 ms.

constexpr int kGmGrid = 256;    // blocks of the basis kernels: one per CU, so that a consumer block can sum the
                                // partial sums of every basis vector itself (256 x 31 doubles)
constexpr int kGmReg = 32;      // basis vectors held in registers; longer bases are read more often
constexpr int kGmAhead = 3;     // iterations queued beyond the last one known to be finished

// Threads of the basis kernels for NB vectors in registers: as many as the
// registers allow, since a block per CU has to cover the memory latency.
constexpr int gm_block(int NB) { return NB <= 16 ? 1024 : 512; }

// Device state of a solve.
struct GmState {
    double rnorm0, last;
    double rtol, atol;
    int32_t its, max_its, kk, reason, done, first;
};

// What the host sees of it, in pinned memory: word = 2 its + done while the
// solve runs (one store, nothing ordered after it), the state after it.
struct GmHost {
    int64_t word;
    GmState st;
};

// Where the kernels find the solve's small arrays (m: restart length).
struct GmDev {
    GmState* st;
    GmHost* host;
    double *p1, *p2, *pn;   // block sums: h1 and h2 per basis vector, |w|^2
    double *h1, *h2;        // the column's coefficients
    double *R, *g, *cs, *sn, *y;
    int m, nb;              // nb: blocks of the basis kernels
};

__device__ __forceinline__ int gm_done(const GmDev& d) {
    return __hip_atomic_load(&d.st->done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Lane `lane`'s value (the same lane in the whole wave), without the
// latency of a shuffle through LDS.
__device__ __forceinline__ double gm_lane(double v, int lane) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                            __builtin_amdgcn_readlane(__double2loint(v), lane));
}

__device__ __forceinline__ double gm_wave_sum(double t) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) t += __shfl_xor(t, off, 64);
    return t;
}

// A lane's share of nb <= kGmGrid block sums; gm_wave_sum of it is their
// total, in the same order in every wave.
__device__ __forceinline__ double gm_share(const double* __restrict__ p, int nb) {
    const int lane = threadIdx.x & 63;
    double v[kGmGrid / 64];
#pragma unroll
    for (int q = 0; q < kGmGrid / 64; q++) v[q] = q * 64 < nb ? p[min(lane + 64 * q, nb - 1)] : 0.0;
    double t = 0.0;
#pragma unroll
    for (int q = 0; q < kGmGrid / 64; q++) t += lane + 64 * q < nb ? v[q] : 0.0;
    return t;
}

__device__ __forceinline__ void gm_publish(const GmDev& d, const GmState& s) {
    __hip_atomic_store(&d.host->word, (int64_t)2 * s.its + s.done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// One wave: the norm of the last w closes column kk - 1 (rotations,
// residual estimate, convergence test), or opens a cycle when kk = 0.  Lane
// j holds entry j of the column and rotation j, 64 entries at a time.
__device__ __forceinline__ void gm_close_column(const GmDev& d, int kk) {
    const int lane = threadIdx.x & 63, c = kk - 1;
    const double nn = gm_share(d.pn, d.nb);
    GmState s = *d.st;
    const double gc = c >= 0 ? d.g[c] : 0.0;
    if (s.done) return;
    if (kk == 0) {
        const double hn = sqrt(gm_wave_sum(nn));
        if (lane == 0) {
            s.kk = 0;
            d.g[0] = hn;
            if (s.first) {
                s.first = 0;
                s.rnorm0 = s.last = hn;
                if (hn == 0.0 || hn <= s.atol) {
                    s.reason = KSP_CONVERGED_ATOL;
                    s.done = 1;
                }
            }
            *d.st = s;
            gm_publish(d, s);
        }
        return;
    }
    double* Rc = d.R + (size_t)c * (d.m + 1);
    double a = 0.0;  // the entry that the next rotation takes, the same in every lane
    for (int j0 = 0; j0 <= c; j0 += 64) {
        const int j = j0 + lane;
        const double h = j <= c ? d.h1[j] + d.h2[j] : 0.0;
        const double cj = j < c ? d.cs[j] : 0.0, sj = j < c ? d.sn[j] : 0.0;
        double r = 0.0;
        for (int q = 0; q < min(64, c + 1 - j0); q++) {
            const double b = gm_lane(h, q);  // entry j0 + q, rotated against a by rotation j0 + q - 1
            if (j0 + q == 0) {
                a = b;
                continue;
            }
            const double cq = q > 0 ? gm_lane(cj, q - 1) : d.cs[j0 - 1], sq = q > 0 ? gm_lane(sj, q - 1) : d.sn[j0 - 1];
            const double up = cq * a + sq * b;
            if (q > 0) {
                if (lane == q - 1) r = up;
            } else if (lane == 0) {
                Rc[j0 - 1] = up;
            }
            a = -sq * a + cq * b;
        }
        if (j < c && lane < 63) Rc[j] = r;
    }
    const double hn = sqrt(gm_wave_sum(nn));
    if (lane == 0) {
        const double den = sqrt(a * a + hn * hn);
        const double cc = den == 0.0 ? 1.0 : a / den, sc = den == 0.0 ? 0.0 : hn / den;
        d.cs[c] = cc;
        d.sn[c] = sc;
        Rc[c] = cc * a + sc * hn;
        d.g[c + 1] = -sc * gc;
        d.g[c] = cc * gc;
        s.its += 1;
        s.kk = c + 1;
        s.last = fabs(-sc * gc);
        if (s.last != s.last) s.reason = KSP_DIVERGED_NANORINF;
        else if (s.last <= s.atol) s.reason = KSP_CONVERGED_ATOL;
        else if (s.last <= s.rtol * s.rnorm0) s.reason = KSP_CONVERGED_RTOL;
        else if (s.its >= s.max_its) s.reason = KSP_DIVERGED_ITS;
        s.done = s.reason != 0;
        *d.st = s;
        gm_publish(d, s);
    }
}

__global__ void k_gm_begin(GmDev d, double rtol, double atol, int max_its, int resume) {
    GmState s = *d.st;
    if (!resume) {
        s.rnorm0 = s.last = 0.0;
        s.rtol = rtol;
        s.atol = atol;
        s.its = 0;
        s.max_its = max_its;
        s.first = 1;
    }
    s.kk = 0;
    s.reason = s.done = 0;
    *d.st = s;
    gm_publish(d, s);
}

// The scale that normalises w, from |w|^2 (0 for w = 0).
__device__ __forceinline__ double gm_scale(double share) {
    const double nrm = sqrt(gm_wave_sum(share));
    return nrm > 0.0 ? 1.0 / nrm : 0.0;
}

// w / |w| from |w|^2's block sums, in two steps.  The product takes FP32
// entries scaled by the power of two next to 1 / |w| (exact), so that its
// range is the matrix's, whatever the units and the size of the residual (a
// product that left it lost the solve); what remains, between 1/2 and 1, is
// applied to the row's sum.  FP64 has the range, and takes the whole scale
// at the end.  Normalising every gathered FP32 entry in FP64 instead: 1% of
// a step on 104k quadratic rows.
template <typename V>
struct GmUnit {
    double share, s, t;
    int e;
    __device__ __forceinline__ explicit GmUnit(double sh) : share(sh), s(0.0), t(0.0), e(0) {}
    __device__ __forceinline__ void begin() {
        s = t = gm_scale(share);
        if (sizeof(V) == 4) {
            e = __builtin_amdgcn_frexp_exp(s);
            t = __builtin_amdgcn_ldexp(s, -e);
        }
    }
    __device__ __forceinline__ V operator()(V w) const {  // an entry for the product
        if constexpr (sizeof(V) == 4) return __builtin_amdgcn_ldexpf(w, e);
        else return w;
    }
    __device__ __forceinline__ V row(V acc) const { return (V)((double)acc * t); }  // its sum
    __device__ __forceinline__ V entry(V w) const { return (V)((double)w * s); }    // of the basis vector
};

// v = w / |w| and y = D^-1 A v (D^-1 absent: y = A v) over the slices of the
// solver matrix.  The scale is formed with the first slice's loads in flight.
// The kernel holds nothing else: closing the column here took it from 8 to 5
// waves a SIMD (15 -> 22 us on 373k rows).
template <typename V, typename CT>
__global__ void __launch_bounds__(kRowBlock)
k_gm_sell(SellOp<V, CT> m, const V* __restrict__ w, V* __restrict__ v, V* __restrict__ y,
          const V* __restrict__ dinv, GmDev d) {
    GmUnit<V> unit(gm_share(d.pn, d.nb));
    if (gm_done(d)) return;
    constexpr int WPB = kRowBlock / kSlice;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kSlice), lane = threadIdx.x % kSlice;
    const RowBlocks it((m.nsl + WPB - 1) / WPB);
    for (int g = it.b; g < it.hi; g += it.step) {
        const int sl = g * WPB + wave;
        if (sl >= m.nsl) continue;
        const SellSlice c = sell_slice(m, sl, lane);
        const int rc = min(c.row, m.n - 1);
        const V wi = w[rc], di = dinv ? dinv[rc] : (V)1;
        if (c.w == 0) unit.begin();
        const V acc = sell_row_sum<V>(m, c, lane, w, unit);
        if (c.row < m.n) {
            v[c.row] = unit.entry(wi);
            y[c.row] = di * unit.row(acc);
        }
    }
}

// The same over the CSR matrix, L lanes a row.
template <int L, typename V>
__global__ void __launch_bounds__(kRowBlock)
k_gm_csr(int n, const int32_t* __restrict__ rowptr, const int32_t* __restrict__ col, const V* __restrict__ val,
         const V* __restrict__ w, V* __restrict__ v, V* __restrict__ y, const V* __restrict__ dinv, GmDev d) {
    GmUnit<V> unit(gm_share(d.pn, d.nb));
    if (gm_done(d)) return;
    unit.begin();
    constexpr int ROWS = kRowBlock / L;
    const int lane = threadIdx.x % L, rloc = threadIdx.x / L;
    for (int grp = blockIdx.x; grp * ROWS < n; grp += gridDim.x) {
        const int row = grp * ROWS + rloc;
        V acc = (V)0;
        if (row < n)
            for (int k = rowptr[row] + lane; k < rowptr[row + 1]; k += L) acc += val[k] * unit(w[col[k]]);
        for (int off = L >> 1; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
        if (row < n && lane == 0) {
            v[row] = unit.entry(w[row]);
            y[row] = (dinv ? dinv[row] : (V)1) * unit.row(acc);
        }
    }
}

// One step of gm_block_sums on the first 2 HALF values: lane pairs at
// distance MASK exchange, each keeps HALF sums; then the steps below it.
template <int HALF, int MASK, int NB>
__device__ __forceinline__ void gm_halve(double (&a)[NB], int lane, int& j) {
    if constexpr (HALF > 0) {
        const bool hi = lane & MASK;
#pragma unroll
        for (int q = 0; q < HALF; q++) {
            const double keep = hi ? a[q + HALF] : a[q], send = hi ? a[q] : a[q + HALF];
            a[q] = keep + __shfl_xor(send, MASK, 64);
        }
        j += hi ? HALF : 0;
        gm_halve<HALF / 2, MASK / 2, NB>(a, lane, j);
    } else if constexpr (MASK > 0) {
        a[0] += __shfl_xor(a[0], MASK, 64);
        gm_halve<0, MASK / 2, NB>(a, lane, j);
    }
}

// Sums NB (8, 16 or 32) per-thread values over the block: each step of a
// wave halves the values a lane still carries (it sends the half its partner
// keeps), so NB sums take about 2 NB shuffles and not 12 NB.  out[j] for j < nv.
template <int NB, int B>
__device__ __forceinline__ void gm_block_sums(double (&a)[NB], int nv, double* __restrict__ out, int stride) {
    __shared__ double sh[B / 64][NB];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int j = 0;
    gm_halve<NB / 2, 32, NB>(a, lane, j);
    __syncthreads();  // the last use of sh
    if ((lane & (64 / NB - 1)) == 0) sh[wave][j] = a[0];
    __syncthreads();
    if ((int)threadIdx.x < NB && (int)threadIdx.x < nv) {
        double t = sh[0][threadIdx.x];
#pragma unroll
        for (int q = 1; q < B / 64; q++) t += sh[q][threadIdx.x];
        out[(size_t)threadIdx.x * stride] = t;
    }
}

// Totals of the block sums of nv <= NB basis vectors, into LDS (zero past
// nv): 16 lanes a vector when there are at most 16 blocks, a wave a vector
// otherwise, every load issued before the first sum.
template <int NB, int B>
__device__ __forceinline__ void gm_totals(const double* __restrict__ p, int nv, int nb, double (&sh)[NB],
                                          double* __restrict__ h) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (nb <= 16) {
        const int j = threadIdx.x >> 4, b = threadIdx.x & 15;
        double t = j < nv && b < nb ? p[(size_t)j * nb + b] : 0.0;
#pragma unroll
        for (int off = 8; off > 0; off >>= 1) t += __shfl_xor(t, off, 64);
        if (b == 0 && j < NB) sh[j] = t;
    } else {
        constexpr int W = B / 64, R = (NB + W - 1) / W;
        double t[R];
#pragma unroll
        for (int r = 0; r < R; r++) {
            const int j = wave + r * W;
            t[r] = j < nv ? gm_share(p + (size_t)j * nb, nb) : 0.0;
        }
#pragma unroll
        for (int r = 0; r < R; r++) {
            t[r] = gm_wave_sum(t[r]);
            const int j = wave + r * W;
            if (lane == 0 && j < NB) sh[j] = t[r];
        }
    }
    __syncthreads();
    if (blockIdx.x == 0 && (int)threadIdx.x < nv) h[threadIdx.x] = sh[threadIdx.x];
}

// Row i of basis vectors 0 .. nv-1 (1 <= nv <= 8 for NB = 8, NB / 2 < nv <= NB
// beyond; past nv the last one again): unconditional loads, all in flight
// together.
template <typename V, int NB>
__device__ __forceinline__ void gm_load(const V* __restrict__ Vb, size_t ldv, int nv, int i, V (&t)[NB]) {
    const V* q = Vb + i;
#pragma unroll
    for (int j = 0; j < NB; j++) {
        t[j] = *q;
        if ((NB > 8 && j < NB / 2) || j + 1 < nv) q += ldv;
    }
}

// p1_j = block sums of w . v_j for j < nv; the last workgroup closes the
// previous column.
template <typename V, int NB>
__global__ void __launch_bounds__(gm_block(NB))
k_gm_dots(int n, size_t ldv, int nv, const V* __restrict__ Vb, const V* __restrict__ w, GmDev d) {
    constexpr int B = gm_block(NB);
    if ((int)blockIdx.x == d.nb) {
        if (threadIdx.x < 64) gm_close_column(d, nv - 1);
        return;
    }
    const int done = gm_done(d), step = d.nb * B;
    const int i0 = blockIdx.x * B + threadIdx.x;
    V t[NB], wi = (V)0;
    if (i0 < n) {
        gm_load<V, NB>(Vb, ldv, nv, i0, t);
        wi = w[i0];
    }
    if (done) return;
    double acc[NB];
#pragma unroll
    for (int j = 0; j < NB; j++) acc[j] = 0.0;
    for (int i = i0; i < n; i += step) {
        if (i != i0) {
            gm_load<V, NB>(Vb, ldv, nv, i, t);
            wi = w[i];
        }
#pragma unroll
        for (int j = 0; j < NB; j++) acc[j] = fma((double)wi, (double)t[j], acc[j]);
    }
    gm_block_sums<NB, B>(acc, nv, d.p1 + blockIdx.x, d.nb);
}

// w -= sum_j h_j v_j (j < nv), h the totals of the block sums p; then, from
// the vectors still in registers, the block sums of w . v_j (DOTS) or of
// |w|^2 (otherwise).  The first rows' loads are issued before the totals.
template <typename V, int NB, bool DOTS>
__global__ void __launch_bounds__(gm_block(NB))
k_gm_orth(int n, size_t ldv, int nv, const V* __restrict__ Vb, V* __restrict__ w, const double* __restrict__ p,
          double* __restrict__ h, double* __restrict__ out, GmDev d) {
    constexpr int B = gm_block(NB);
    __shared__ double sh[NB];
    const int done = gm_done(d);
    const int i0 = blockIdx.x * B + threadIdx.x;
    V t[NB], wi = (V)0;
    if (i0 < n) {
        gm_load<V, NB>(Vb, ldv, nv, i0, t);
        wi = w[i0];
    }
    if (done) return;
    gm_totals<NB, B>(p, nv, d.nb, sh, h);
    double acc[DOTS ? NB : 1];
#pragma unroll
    for (int j = 0; j < (DOTS ? NB : 1); j++) acc[j] = 0.0;
    for (int i = i0; i < n; i += gridDim.x * B) {
        if (i != i0) {
            gm_load<V, NB>(Vb, ldv, nv, i, t);
            wi = w[i];
        }
        double a = (double)wi;
#pragma unroll
        for (int j = 0; j < NB; j++) a = fma(-sh[j], (double)t[j], a);
        const V o = (V)a;
        w[i] = o;
        if (DOTS) {
#pragma unroll
            for (int j = 0; j < NB; j++) acc[j] = fma((double)o, (double)t[j], acc[j]);
        } else {
            acc[0] = fma((double)o, (double)o, acc[0]);
        }
    }
    if constexpr (DOTS) {
        gm_block_sums<NB, B>(acc, nv, out + blockIdx.x, d.nb);
    } else {
        __shared__ double sn[B / 64][1];
        block_sum<1>(acc, sn);
        if (threadIdx.x == 0) out[blockIdx.x] = acc[0];
    }
}

// The same for a basis longer than the registers hold, kGmReg vectors at a
// time (h given), and the totals by a launch of their own.
template <typename V>
__global__ void __launch_bounds__(gm_block(kGmReg))
k_gm_dots_long(int n, size_t ldv, int nv, const V* __restrict__ Vb, const V* __restrict__ w, double* __restrict__ out,
               GmDev d) {
    constexpr int B = gm_block(kGmReg);
    if ((int)blockIdx.x == d.nb) {
        if (threadIdx.x < 64) gm_close_column(d, nv - 1);
        return;
    }
    if (gm_done(d)) return;
    for (int c0 = 0; c0 < nv; c0 += kGmReg) {
        double acc[kGmReg];
#pragma unroll
        for (int j = 0; j < kGmReg; j++) acc[j] = 0.0;
        for (int i = blockIdx.x * B + threadIdx.x; i < n; i += d.nb * B) {
            const double wi = (double)w[i];
#pragma unroll
            for (int j = 0; j < kGmReg; j++) acc[j] = fma(wi, (double)Vb[ldv * min(c0 + j, nv - 1) + i], acc[j]);
        }
        gm_block_sums<kGmReg, B>(acc, nv - c0, out + (size_t)c0 * d.nb + blockIdx.x, d.nb);
    }
}

template <typename V>
__global__ void __launch_bounds__(gm_block(kGmReg))
k_gm_orth_long(int n, size_t ldv, int nv, const V* __restrict__ Vb, V* __restrict__ w, const double* __restrict__ h,
               double* __restrict__ pn, GmDev d) {
    constexpr int B = gm_block(kGmReg);
    if (gm_done(d)) return;
    double acc[1] = {0.0};
    for (int i = blockIdx.x * B + threadIdx.x; i < n; i += gridDim.x * B) {
        double a = (double)w[i];
#pragma unroll 8
        for (int j = 0; j < nv; j++) a = fma(-h[j], (double)Vb[ldv * j + i], a);
        const V o = (V)a;
        w[i] = o;
        acc[0] = fma((double)o, (double)o, acc[0]);
    }
    __shared__ double sn[B / 64][1];
    block_sum<1>(acc, sn);
    if (threadIdx.x == 0) pn[blockIdx.x] = acc[0];
}

__global__ void __launch_bounds__(64)
k_gm_reduce(GmDev d, const double* __restrict__ p, double* __restrict__ h) {
    const double t = gm_wave_sum(gm_share(p + (size_t)blockIdx.x * d.nb, d.nb));
    if (!gm_done(d) && threadIdx.x == 0) h[blockIdx.x] = t;
}

constexpr int kGmNormBlock = 1024;

// w = D^-1 r64 (D^-1 absent: r64) in the working precision, and |w|^2.
template <typename V>
__global__ void __launch_bounds__(kGmNormBlock)
k_gm_precres_norm(int n, const double* __restrict__ r64, const double* __restrict__ dinv, V* __restrict__ out,
                  GmDev d) {
    double nn = 0.0;
    for (int i = blockIdx.x * kGmNormBlock + threadIdx.x; i < n; i += gridDim.x * kGmNormBlock) {
        const V o = dinv ? (V)(dinv[i] * r64[i]) : (V)r64[i];
        out[i] = o;
        nn += (double)o * (double)o;
    }
    double a[1] = {nn};
    __shared__ double sn[kGmNormBlock / 64][1];
    block_sum<1>(a, sn);
    if (threadIdx.x == 0) d.pn[blockIdx.x] = a[0];
}

template <typename V>
__global__ void __launch_bounds__(kGmNormBlock)
k_gm_norm(int n, const V* __restrict__ w, GmDev d) {
    double nn = 0.0;
    for (int i = blockIdx.x * kGmNormBlock + threadIdx.x; i < n; i += gridDim.x * kGmNormBlock)
        nn += (double)w[i] * (double)w[i];
    double a[1] = {nn};
    __shared__ double sn[kGmNormBlock / 64][1];
    block_sum<1>(a, sn);
    if (threadIdx.x == 0) d.pn[blockIdx.x] = a[0];
}

// One wave: closes column kk - 1 if the solve has not finished before it,
// then y = R^-1 g over the cycle's columns.  Up to 64 columns, lane j keeps
// g_j and the triangle is staged in LDS; y_i = g_i / R_ii by the reciprocals,
// formed together, and one correction.
__global__ void __launch_bounds__(64)
k_gm_cycle_end(GmDev d, int kk) {
    constexpr int N = 64;
    __shared__ double sR[N * (N + 1) / 2];
    if (kk > 0) gm_close_column(d, kk);
    __syncthreads();
    const int nc = __hip_atomic_load(&d.st->kk, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT), lane = threadIdx.x;
    const int ld = d.m + 1;
    if (nc <= N) {
        for (int i = 0; i < nc; i++)
            if (lane <= i) sR[i * (i + 1) / 2 + lane] = d.R[(size_t)i * ld + lane];
        double g = lane < nc ? d.g[lane] : 0.0;
        __syncthreads();
        const double rd = lane < nc ? sR[lane * (lane + 1) / 2 + lane] : 1.0, inv = 1.0 / rd;
        double y = 0.0;
        for (int i = nc - 1; i >= 0; i--) {
            const double gi = gm_lane(g, i), ri = gm_lane(rd, i), vi = gm_lane(inv, i);
            double yi = gi * vi;
            const double e = fma(-yi, ri, gi) * vi;
            if (e == e) yi += e;
            if (lane == i) y = yi;
            if (lane < i) g = fma(-sR[i * (i + 1) / 2 + lane], yi, g);
        }
        if (lane < nc) d.y[lane] = y;
        return;
    }
    for (int j = lane; j < nc; j += 64) d.y[j] = d.g[j];
    __syncthreads();
    for (int i = nc - 1; i >= 0; i--) {
        const double yi = d.y[i] / d.R[(size_t)i * ld + i];
        __syncthreads();
        for (int j = lane; j < i; j += 64) d.y[j] -= d.R[(size_t)i * ld + j] * yi;
        if (lane == 0) d.y[i] = yi;
        __syncthreads();
    }
}

// x += sum_j y_j v_j over the cycle's columns
template <typename V>
__global__ void __launch_bounds__(kVecBlock)
k_gm_update_x(int n, size_t ldv, const V* __restrict__ Vb, GmDev d, double* __restrict__ x) {
    const int kk = d.st->kk;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        double acc = x[i];
#pragma unroll 8
        for (int j = 0; j < kk; j++) acc += d.y[j] * (double)Vb[ldv * j + i];
        x[i] = acc;
    }
}

// z = D^-1 r64 or r64 (pc_apply_host)
template <typename V>
__global__ void __launch_bounds__(kVecBlock)
k_gm_precres(int n, const double* __restrict__ r64, const double* __restrict__ dinv, V* __restrict__ out) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
        out[i] = dinv ? (V)(dinv[i] * r64[i]) : (V)r64[i];
}

// One workgroup takes a whole cycle of a small system: the residual's norm,
// the iterations, the triangular solve and the update of x in one launch,
// with a barrier where the other path has a launch.  w and A v are in LDS
// (the product gathers there); a thread keeps the same rows of every basis
// vector, which stay in this CU's caches, and with at most one row a thread
// it reads them once an iteration.  Bound by the latency of the block sums
// (6 us an iteration) and by what one CU reads (gm_small_fits): 324 rows 7.3
// us an iteration, 4225 rows 32 us, where the four launches take 21 us.
// Time step on 17 x 17 P1 triangles: 0.56 -> 0.32 ms.
constexpr int kGmSmallBlock = 512;

// Gram-Schmidt of w against nv vectors, twice; |w|^2 to every thread.
template <typename V, int NB, bool ONE>
__device__ __forceinline__ double gm_small_orth(int n, size_t ldv, int nv, const V* Vb, V* w, double* h1, double* h2) {
    constexpr int B = kGmSmallBlock;
    __shared__ double total;
    V t[NB];
    double acc[NB], nn[1] = {0.0};
#pragma unroll
    for (int j = 0; j < NB; j++) acc[j] = 0.0;
    for (int i = threadIdx.x; i < n; i += B) {
        gm_load<V, NB>(Vb, ldv, nv, i, t);
        const double wi = (double)w[i];
#pragma unroll
        for (int j = 0; j < NB; j++) acc[j] = fma(wi, (double)t[j], acc[j]);
    }
    gm_block_sums<NB, B>(acc, nv, h1, 1);
    __syncthreads();
#pragma unroll
    for (int j = 0; j < NB; j++) acc[j] = 0.0;
    for (int i = threadIdx.x; i < n; i += B) {
        if (!ONE) gm_load<V, NB>(Vb, ldv, nv, i, t);
        double a = (double)w[i];
#pragma unroll
        for (int j = 0; j < NB; j++)
            if (j < nv) a = fma(-h1[j], (double)t[j], a);
        const V o = (V)a;
        w[i] = o;
#pragma unroll
        for (int j = 0; j < NB; j++) acc[j] = fma((double)o, (double)t[j], acc[j]);
    }
    gm_block_sums<NB, B>(acc, nv, h2, 1);
    __syncthreads();
    for (int i = threadIdx.x; i < n; i += B) {
        if (!ONE) gm_load<V, NB>(Vb, ldv, nv, i, t);
        double a = (double)w[i];
#pragma unroll
        for (int j = 0; j < NB; j++)
            if (j < nv) a = fma(-h2[j], (double)t[j], a);
        const V o = (V)a;
        w[i] = o;
        nn[0] = fma((double)o, (double)o, nn[0]);
    }
    __shared__ double sn[B / 64][1];
    block_sum<1>(nn, sn);
    if (threadIdx.x == 0) total = nn[0];
    __syncthreads();
    return total;
}

template <typename V, bool ONE>
__global__ void __launch_bounds__(kGmSmallBlock)
k_gm_small(SellOp<V, int16_t> m, size_t ldv, V* __restrict__ Vb, const double* __restrict__ r64,
           const double* __restrict__ dinv64, const V* __restrict__ dinv, double* __restrict__ x, GmDev d) {
    constexpr int B = kGmSmallBlock, N = kGmReg;
    extern __shared__ double gm_lds[];
    V* w = reinterpret_cast<V*>(gm_lds);
    V* w2 = w + ((m.n + 1) & ~1);
    __shared__ double h1[N], h2[N], cs[N], sn[N], g[N + 1], R[N][N + 1], y[N], s_nn;
    __shared__ int s_done;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, n = m.n;
    GmState st = *d.st;
    double nn[1] = {0.0};
    for (int i = tid; i < n; i += B) {
        const V o = (V)(dinv64[i] * r64[i]);
        w[i] = o;
        nn[0] = fma((double)o, (double)o, nn[0]);
    }
    __shared__ double sred[B / 64][1];
    block_sum<1>(nn, sred);
    if (tid == 0) s_nn = nn[0];
    __syncthreads();
    double hn = sqrt(s_nn);
    if (tid == 0) g[0] = hn;
    st.kk = 0;
    if (st.first) {
        st.first = 0;
        st.rnorm0 = st.last = hn;
        if (hn == 0.0 || hn <= st.atol) {
            st.reason = KSP_CONVERGED_ATOL;
            st.done = 1;
        }
    }
    int kk = 0;
    while (kk < d.m && !st.done) {
        const double sc = hn > 0.0 ? 1.0 / hn : 0.0;
        for (int i = tid; i < n; i += B) {
            const V v = (V)((double)w[i] * sc);
            Vb[ldv * kk + i] = v;
            w[i] = v;
        }
        __syncthreads();
        for (int sl = __builtin_amdgcn_readfirstlane(wave); sl < m.nsl; sl += B / 64) {
            const SellSlice c = sell_slice(m, sl, lane);
            const V di = dinv[min(c.row, n - 1)];
            SellX fx;
            const V acc = sell_row_sum<V>(m, c, lane, (const V*)w, fx);
            if (c.row < n) w2[c.row] = di * acc;
        }
        __syncthreads();
        V* q = w;
        w = w2;
        w2 = q;
        const int nv = kk + 1;
        const double s2 = nv <= 8 ? gm_small_orth<V, 8, ONE>(n, ldv, nv, Vb, w, h1, h2)
                        : nv <= 16 ? gm_small_orth<V, 16, ONE>(n, ldv, nv, Vb, w, h1, h2)
                                   : gm_small_orth<V, N, ONE>(n, ldv, nv, Vb, w, h1, h2);
        hn = sqrt(s2);
        if (wave == 0) {  // close the column: lane j holds entry j and rotation j
            const double h = lane <= kk ? h1[lane] + h2[lane] : 0.0;
            const double cj = lane < kk ? cs[lane] : 0.0, sj = lane < kk ? sn[lane] : 0.0;
            double a = gm_lane(h, 0), r = 0.0;
            for (int j = 0; j < kk; j++) {
                const double b = gm_lane(h, j + 1), cq = gm_lane(cj, j), sq = gm_lane(sj, j);
                const double up = cq * a + sq * b;
                if (lane == j) r = up;
                a = -sq * a + cq * b;
            }
            const double den = sqrt(a * a + hn * hn);
            const double cc = den == 0.0 ? 1.0 : a / den, ss = den == 0.0 ? 0.0 : hn / den;
            if (lane == kk) r = cc * a + ss * hn;
            if (lane <= kk) R[kk][lane] = r;
            if (lane == 0) {
                const double gc = g[kk];
                cs[kk] = cc;
                sn[kk] = ss;
                g[kk + 1] = -ss * gc;
                g[kk] = cc * gc;
            }
        }
        __syncthreads();
        kk++;
        st.its += 1;
        st.kk = kk;
        st.last = fabs(g[kk]);
        if (st.last != st.last) st.reason = KSP_DIVERGED_NANORINF;
        else if (st.last <= st.atol) st.reason = KSP_CONVERGED_ATOL;
        else if (st.last <= st.rtol * st.rnorm0) st.reason = KSP_CONVERGED_RTOL;
        else if (st.its >= st.max_its) st.reason = KSP_DIVERGED_ITS;
        st.done = st.reason != 0;
    }
    if (wave == 0) {  // y = R^-1 g, as in k_gm_cycle_end
        double gl = lane < kk ? g[lane] : 0.0, yl = 0.0;
        const double rd = lane < kk ? R[lane][lane] : 1.0, inv = 1.0 / rd;
        for (int i = kk - 1; i >= 0; i--) {
            const double gi = gm_lane(gl, i), ri = gm_lane(rd, i), vi = gm_lane(inv, i);
            double yi = gi * vi;
            const double e = fma(-yi, ri, gi) * vi;
            if (e == e) yi += e;
            if (lane == i) yl = yi;
            if (lane < i) gl = fma(-R[i][lane], yi, gl);
        }
        if (lane < kk) y[lane] = yl;
    }
    __syncthreads();
    for (int i = tid; i < n; i += B) {
        double acc = x[i];
#pragma unroll 8
        for (int j = 0; j < kk; j++) acc += y[j] * (double)Vb[ldv * j + i];
        x[i] = acc;
    }
    if (tid == 0) {
        *d.st = st;
        gm_publish(d, st);
    }
}

// A cycle goes to one workgroup when its vectors fit LDS, the basis its
// registers, and an iteration -- 6 us of block sums, then the matrix and
// three passes over ten vectors read by one CU at 55 GB/s -- stays below the
// 20 us of the four launches (P1 triangles: up to 2200 rows).  Column indices
// of so few rows have 16 bits.
static bool gm_small_fits(const KrylovWork* k, int n, int64_t nnz, int m, size_t value) {
    const double bytes = (double)nnz * (double)(value + 2) + 30.0 * (double)n * (double)value;
    return k->sell.nsl && k->sell.use16 && m <= kGmReg && 2 * value * ((size_t)n + 2) <= ((size_t)96 << 10) && 6.0 + bytes / 55e3 < 18.0;
}

template <typename V>
static int run_gmres(flgpu_ctx* c, const flgpu_solver_params* sp, flgpu_solve_info* info) {
    KrylovWork* k = c->kw;
    const int n = c->rows;
    const int m = sp->restart > 0 ? sp->restart : 30;
    const bool mixed = std::is_same<V, float>::value;
    const V* val = mixed ? (const V*)k->val32.p : (const V*)k->val64.p;
    const V* dinv = mixed ? (const V*)k->dinv32.p : (const V*)k->dinv.p;
    const size_t ldv = ((size_t)n + 31) & ~(size_t)31;  // basis vectors start on whole lines
    V* Vb;
    V* wb[2];  // the product reads one and writes the other
    if (mixed) {
        FLGPU_TRY(k->V32.alloc(ldv * m));
        Vb = (V*)k->V32.p;
        wb[0] = (V*)k->w32.p;
        wb[1] = (V*)k->z32.p;
    } else {
        FLGPU_TRY(k->V.alloc(ldv * m));
        Vb = (V*)k->V.p;
        wb[0] = (V*)k->w.p;
        wb[1] = (V*)k->z.p;
    }
    if (sp->pc == FLGPU_PC_NONE) {
        hipLaunchKernelGGL((k_fill<double>), dim3(k->nblk), dim3(kVecBlock), 0, c->stream, n, 1.0, k->dinv.p);
        if (mixed)
            hipLaunchKernelGGL((k_fill<float>), dim3(k->nblk), dim3(kVecBlock), 0, c->stream, n, 1.0f, k->dinv32.p);
        FLGPU_HIP(hipGetLastError());
    }
    // left SSOR: the product and the residual go through tmp, then the sweeps
    const bool ssor = sp->pc == FLGPU_PC_SOR;
    if (ssor) FLGPU_TRY(ssor_prepare<V>(c, k, val));
    V* tmp = mixed ? (V*)k->rt32.p : (V*)k->rt.p;
    const int nb = std::max(1, (int)std::min<int64_t>(kGmGrid, ((int64_t)n + 511) / 512));
    const size_t mm = (size_t)m + 1;
    FLGPU_TRY(k->gm_work.reserve((2 * mm + 1) * kGmGrid + 7 * mm + mm * m));
    FLGPU_TRY(k->gm_state.reserve(sizeof(GmState)));
    if (!k->gm_host) {
        FLGPU_HIP(hipHostMalloc((void**)&k->gm_host, sizeof(GmHost), hipHostMallocMapped | hipHostMallocCoherent));
        std::memset(k->gm_host, 0, sizeof(GmHost));
    }
    GmHost* host = static_cast<GmHost*>(k->gm_host);
    GmDev d{};
    d.st = reinterpret_cast<GmState*>(k->gm_state.p);
    FLGPU_HIP(hipHostGetDevicePointer((void**)&d.host, host, 0));
    d.m = m;
    d.nb = nb;
    d.p1 = k->gm_work.p;
    d.p2 = d.p1 + mm * kGmGrid;
    d.pn = d.p2 + mm * kGmGrid;
    d.h1 = d.pn + kGmGrid;
    d.h2 = d.h1 + mm;
    d.g = d.h2 + mm;
    d.cs = d.g + mm;
    d.sn = d.cs + mm;
    d.y = d.sn + mm;
    d.R = d.y + mm;
    const int L = lanes_for(c);
    const int rows_per_blk = kRowBlock / L;
    const int mgrid = std::max(1, (int)std::min<int64_t>(kMaxRowGrid, (n + rows_per_blk - 1) / rows_per_blk));
    const V* sval = sell_values(k, val);
    auto product = [&](const V* w, V* v, V* out) -> int {
        const V* dv = ssor ? nullptr : dinv;
        V* y = ssor ? tmp : out;
        if (sval) {
            const int grid = sell_grid(k->sell.nsl);
            if (k->sell.use16) {
                const SellOp<V, int16_t> op = sell_op(k->sell, n, sval, k->sell.col16.p);
                hipLaunchKernelGGL((k_gm_sell<V, int16_t>), dim3(grid), dim3(kRowBlock), 0, c->stream, op, w, v, y, dv,
                                   d);
            } else {
                const SellOp<V, int32_t> op = sell_op(k->sell, n, sval, k->sell.col32.p);
                hipLaunchKernelGGL((k_gm_sell<V, int32_t>), dim3(grid), dim3(kRowBlock), 0, c->stream, op, w, v, y, dv,
                                   d);
            }
        } else {
            auto launch = [&](auto kern) {
                hipLaunchKernelGGL(kern, dim3(mgrid), dim3(kRowBlock), 0, c->stream, n, c->rowptr.p, c->col.p, val,
                                   w, v, y, dv, d);
            };
            switch (L) {
                case 4: launch(&k_gm_csr<4, V>); break;
                case 8: launch(&k_gm_csr<8, V>); break;
                case 16: launch(&k_gm_csr<16, V>); break;
                case 32: launch(&k_gm_csr<32, V>); break;
                default: launch(&k_gm_csr<64, V>); break;
            }
        }
        if (ssor) FLGPU_TRY(ssor_sweeps<V>(c, k, tmp, out, &d.st->done));
        return FLGPU_OK;
    };
    // Gram-Schmidt of w against nv basis vectors, twice, and |w|^2
    auto orthogonalise = [&](V* w, int nv) {
        auto pass = [&](auto nbc) {
            constexpr int NB = decltype(nbc)::value;
            const dim3 grid(nb), block(gm_block(NB));
            hipLaunchKernelGGL((k_gm_dots<V, NB>), dim3(nb + 1), block, 0, c->stream, n, ldv, nv, Vb, w, d);
            hipLaunchKernelGGL((k_gm_orth<V, NB, true>), grid, block, 0, c->stream, n, ldv, nv, Vb, w, d.p1, d.h1,
                               d.p2, d);
            hipLaunchKernelGGL((k_gm_orth<V, NB, false>), grid, block, 0, c->stream, n, ldv, nv, Vb, w, d.p2, d.h2,
                               d.pn, d);
        };
        if (nv <= 8) return pass(std::integral_constant<int, 8>());
        if (nv <= 16) return pass(std::integral_constant<int, 16>());
        if (nv <= kGmReg) return pass(std::integral_constant<int, kGmReg>());
        const dim3 grid(nb), block(gm_block(kGmReg));
        for (int q = 0; q < 2; q++) {
            double *pq = q ? d.p2 : d.p1, *hq = q ? d.h2 : d.h1;
            hipLaunchKernelGGL((k_gm_dots_long<V>), dim3(q ? nb : nb + 1), block, 0, c->stream, n, ldv, nv, Vb, w, pq, d);
            hipLaunchKernelGGL(k_gm_reduce, dim3(nv), dim3(64), 0, c->stream, d, pq, hq);
            hipLaunchKernelGGL((k_gm_orth_long<V>), grid, block, 0, c->stream, n, ldv, nv, Vb, w, hq, d.pn, d);
        }
    };
    const int max_its = sp->max_its > 0 ? sp->max_its : 10000;
    Scal& h = *k->h_scal;
    std::memset(&h, 0, sizeof h);
    FLGPU_TRY(write_scal(c, k));
    FLGPU_TRY(norm_b(c, k));
    host->word = 0;
    hipLaunchKernelGGL(k_gm_begin, dim3(1), dim3(1), 0, c->stream, d, sp->rtol, sp->atol, max_its, 0);
    auto t0 = std::chrono::steady_clock::now();
    int refinements = 0;
    bool have_residual = false;
    const bool small = !ssor && sval && gm_small_fits(k, n, c->nnz, m, sizeof(V));
    auto small_cycle = [&]() -> int {
        const size_t lds = 2 * sizeof(V) * (((size_t)n + 1) & ~(size_t)1);
        const SellOp<V, int16_t> op = sell_op(k->sell, n, sval, (const int16_t*)k->sell.col16.p);
        auto launch = [&](auto kern) -> int {
            FLGPU_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                          hipFuncAttributeMaxDynamicSharedMemorySize, 100 << 10));
            hipLaunchKernelGGL(kern, dim3(1), dim3(kGmSmallBlock), lds, c->stream, op, ldv, Vb, (const double*)k->r.p,
                               (const double*)k->dinv.p, dinv, k->x.p, d);
            FLGPU_HIP(hipGetLastError());
            return FLGPU_OK;
        };
        return n <= kGmSmallBlock ? launch(&k_gm_small<V, true>) : launch(&k_gm_small<V, false>);
    };
    for (;;) {
        // residual in FP64, preconditioned, in the working precision
        if (!have_residual) FLGPU_TRY(true_residual(c, k));
        have_residual = false;
        if (small) {
            refinements++;
            FLGPU_TRY(small_cycle());
            FLGPU_TRY(true_residual(c, k));
            FLGPU_HIP(hipMemcpyAsync(&host->st, d.st, sizeof(GmState), hipMemcpyDeviceToHost, c->stream));
            FLGPU_TRY(read_scal(c, k));
            have_residual = true;
            if (!host->st.reason) continue;
            if (!mixed || host->st.reason <= 0 ||
                std::sqrt(h.true_rr) <= std::max(sp->rtol * std::sqrt(h.bb), sp->atol) || host->st.its >= max_its)
                break;
            hipLaunchKernelGGL(k_gm_begin, dim3(1), dim3(1), 0, c->stream, d, sp->rtol, sp->atol, max_its, 1);
            continue;
        }
        int cur = 0;
        hipLaunchKernelGGL((k_gm_precres_norm<V>), dim3(nb), dim3(kGmNormBlock), 0, c->stream, n, k->r.p,
                           ssor ? nullptr : k->dinv.p, ssor ? tmp : wb[0], d);
        if (ssor) {
            FLGPU_TRY(ssor_sweeps<V>(c, k, tmp, wb[0], nullptr));
            hipLaunchKernelGGL((k_gm_norm<V>), dim3(nb), dim3(kGmNormBlock), 0, c->stream, n, wb[0], d);
        }
        FLGPU_HIP(hipGetLastError());
        refinements++;
        const int64_t before = host->word / 2;  // closed columns of the earlier cycles: none is in flight
        int kk = 0;
        for (; kk < m; kk++) {
            FLGPU_TRY(wait_word(c, &host->word, before + kk - kGmAhead));
            if (__atomic_load_n(&host->word, __ATOMIC_ACQUIRE) & 1) break;
            FLGPU_TRY(product(wb[cur], Vb + ldv * kk, wb[cur ^ 1]));
            cur ^= 1;
            orthogonalise(wb[cur], kk + 1);
            FLGPU_HIP(hipGetLastError());
        }
        hipLaunchKernelGGL(k_gm_cycle_end, dim3(1), dim3(64), 0, c->stream, d, kk);
        hipLaunchKernelGGL((k_gm_update_x<V>), dim3(k->nblk), dim3(kVecBlock), 0, c->stream, n, ldv, Vb, d, k->x.p);
        FLGPU_HIP(hipGetLastError());
        FLGPU_TRY(wait_word(c, &host->word, before + kk));
        if (!(__atomic_load_n(&host->word, __ATOMIC_ACQUIRE) & 1)) continue;
        FLGPU_TRY(true_residual(c, k));
        FLGPU_HIP(hipMemcpyAsync(&host->st, d.st, sizeof(GmState), hipMemcpyDeviceToHost, c->stream));
        FLGPU_TRY(read_scal(c, k));
        // mixed: the FP32 estimate converged, the FP64 residual decides
        if (!mixed || host->st.reason <= 0 || std::sqrt(h.true_rr) <= std::max(sp->rtol * std::sqrt(h.bb), sp->atol) ||
            host->st.its >= max_its)
            break;
        host->word = (int64_t)2 * host->st.its;
        hipLaunchKernelGGL(k_gm_begin, dim3(1), dim3(1), 0, c->stream, d, sp->rtol, sp->atol, max_its, 1);
        have_residual = true;
    }
    auto t1 = std::chrono::steady_clock::now();
    const double bnorm = std::sqrt(h.bb);
    info->seconds = std::chrono::duration<double>(t1 - t0).count();
    info->its = host->st.its;
    info->reason = host->st.reason;
    info->true_relres = bnorm > 0 ? std::sqrt(h.true_rr) / bnorm : std::sqrt(h.true_rr);
    info->precond_relres = host->st.rnorm0 > 0 ? host->st.last / host->st.rnorm0 : host->st.last;
    info->refinements = mixed ? refinements : 0;
    info->fallback = 0;
    return FLGPU_OK;
}

int solve(flgpu_ctx* c, const flgpu_solver_params* sp, double* x_host, flgpu_solve_info* info_out) {
    flgpu_solve_info info{};
    const bool mixed = sp->precision == FLGPU_MIXED;
    if (sp->precision != FLGPU_FP64 && sp->precision != FLGPU_MIXED)
        return set_error(FLGPU_EINVAL, "flgpu_solve: precision %d", sp->precision);
    if (sp->ksp != FLGPU_KSP_CG && sp->ksp != FLGPU_KSP_GMRES && sp->ksp != FLGPU_KSP_FCG &&
        sp->ksp != FLGPU_KSP_PIPECG)
        return set_error(FLGPU_EINVAL, "flgpu_solve: ksp %d", sp->ksp);
    if (sp->pc != FLGPU_PC_NONE && sp->pc != FLGPU_PC_JACOBI && sp->pc != FLGPU_PC_LEARNED && sp->pc != FLGPU_PC_SOR &&
        sp->pc != FLGPU_PC_FSAI)
        return set_error(FLGPU_EINVAL, "flgpu_solve: pc %d", sp->pc);
    const bool factor = sp->pc == FLGPU_PC_LEARNED || sp->pc == FLGPU_PC_FSAI;
    if (factor && sp->ksp == FLGPU_KSP_GMRES)
        return set_error(FLGPU_EUNSUPPORTED, "flgpu_solve: the learned and fsai preconditioners run with cg/fcg/pipecg");
    FLGPU_TRY(ensure_work(c, mixed));
    KrylovWork* k = c->kw;
    const bool zero_x = sp->start_from_zero || !x_host;
    if (x_host && !sp->start_from_zero)
        FLGPU_HIP(hipMemcpyAsync(k->x.p, x_host, sizeof(double) * c->rows, hipMemcpyHostToDevice, c->stream));
    FLGPU_TRY(build_reduced(c, k, mixed, zero_x));
    k->prepared = true;
    k->prepared_mixed = mixed;
    if (factor) FLGPU_TRY(learned_prepare(c, mixed, sp->pc == FLGPU_PC_FSAI));
    k->dx_on = false;  // set by the mixed CG loops for their FP32 increment
    if (sp->ksp == FLGPU_KSP_GMRES) {
        FLGPU_TRY(mixed ? run_gmres<float>(c, sp, &info) : run_gmres<double>(c, sp, &info));
    } else if (sp->ksp == FLGPU_KSP_PIPECG) {
        FLGPU_TRY(mixed ? run_cg1<float>(c, sp, &info, factor) : run_cg1<double>(c, sp, &info, factor));
    } else {
        FLGPU_TRY(mixed ? run_cg<float>(c, sp, &info, factor) : run_cg<double>(c, sp, &info, factor));
    }
    k->dx_on = false;  // the loops end with a true residual, which adds the increment to x
    hipLaunchKernelGGL(k_finish_x, dim3(grid_for(c->rows, kVecBlock)), dim3(kVecBlock), 0, c->stream, c->rows,
                       k->x.p, c->rhs.p, c->inactive.p, c->have_inactive ? 1 : 0);
    FLGPU_HIP(hipGetLastError());
    if (x_host) FLGPU_TRY(copy_out(c, x_host, k->x.p, sizeof(double) * c->rows));
    FLGPU_HIP(hipStreamSynchronize(c->stream));
    k->have_x = true;
    if (info_out) *info_out = info;
    return FLGPU_OK;
}

void krylov_invalidate(flgpu_ctx* c) {
    if (c->kw) c->kw->prepared = c->kw->prepared_mixed = false;
}

void krylov_free(flgpu_ctx* c) {
    delete c->kw;
    c->kw = nullptr;
}

// ---------------------------------------------------------------------
// The solve without allocation
// ---------------------------------------------------------------------
//
// Every buffer of the FP64 (F)PCG -- reduced matrix values, the vectors,
// per-block partial sums, the two solver-scalar slots and the row blocks of
// the streamed product -- is carved out of one file-scope device array.
// The host code never names the array itself (in host code its name is a
// host-side stand-in): it takes the array's device address once per GPU
// from hipGetSymbolAddress (noalloc_setup, called by flgpu_init with the
// device current) and passes that address on.  Every context on a GPU
// shares that GPU's array, so solves that overlap on one GPU race.

constexpr size_t kNoAllocBytes = (size_t)64 << 20;
static __device__ __align__(256) unsigned char scratch[kNoAllocBytes];
static std::mutex g_scratch_mu;
static unsigned char* g_scratch_ptr[kMaxDevices] = {};

int noalloc_setup(int device) {
    if (device < 0 || device >= kMaxDevices)
        return set_error(FLGPU_EUNSUPPORTED, "flgpu_init: device %d beyond the %d the library tracks", device,
                         kMaxDevices);
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (g_scratch_ptr[device]) return FLGPU_OK;
    void* p = nullptr;
    FLGPU_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    if (!p) return set_error(FLGPU_EHIP, "flgpu_init: no device address for the solver work array");
    g_scratch_ptr[device] = static_cast<unsigned char*>(p);
    return FLGPU_OK;
}

static unsigned char* noalloc_ptr(int device) {
    if (device < 0 || device >= kMaxDevices) return nullptr;
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    return g_scratch_ptr[device];
}

// Row blocks of a fixed number of rows, rows_per * maxlen <= kStreamNnz
// (or one row per block): computed on the device, no host table.
__global__ void __launch_bounds__(256)
k_fixed_row_blocks(int n, int rows_per, int nrb, const int32_t* __restrict__ rowptr, int32_t* __restrict__ rb,
                   int32_t* __restrict__ rbk) {
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b > nrb) return;
    const int r = (int)std::min<int64_t>((int64_t)b * rows_per, n);
    rb[b] = r;
    rbk[b] = rowptr[r];
}

// Carves the work of an n-row, nnz-entry FP64 (F)PCG out of the array;
// false when it does not fit (*need gets the bytes it would take).
static bool noalloc_carve(unsigned char* base, int n, int64_t nnz, int nrb, KrylovWork& k, size_t* need) {
    size_t off = 0;
    auto take = [&](size_t bytes) {
        const size_t at = off;
        off = (off + bytes + 255) & ~(size_t)255;
        return at;
    };
    const size_t o_val = take(sizeof(double) * (size_t)nnz);
    size_t o_vec[7];
    for (size_t& o : o_vec) o = take(sizeof(double) * (size_t)n);
    const size_t o_part = take(sizeof(double) * (size_t)kPartStride * PART_COMPONENTS);
    const size_t o_scal = take(sizeof(Scal) * 2);
    const size_t o_rb = take(sizeof(int32_t) * ((size_t)nrb + 1));
    const size_t o_rbk = take(sizeof(int32_t) * ((size_t)nrb + 1));
    *need = off;
    if (off > kNoAllocBytes) return false;
    k.val64.borrow(reinterpret_cast<double*>(base + o_val), (size_t)nnz);
    DevBuf<double>* vecs[7] = {&k.b, &k.x, &k.r, &k.z, &k.p, &k.w, &k.dinv};
    for (int q = 0; q < 7; q++) vecs[q]->borrow(reinterpret_cast<double*>(base + o_vec[q]), (size_t)n);
    k.partials.borrow(reinterpret_cast<double*>(base + o_part), (size_t)kPartStride * PART_COMPONENTS);
    k.scal.borrow(reinterpret_cast<Scal*>(base + o_scal), 2);
    k.rb.borrow(reinterpret_cast<int32_t*>(base + o_rb), (size_t)nrb + 1);
    k.rbk.borrow(reinterpret_cast<int32_t*>(base + o_rbk), (size_t)nrb + 1);
    return true;
}

int solve_noalloc(flgpu_ctx* c, const flgpu_solver_params* sp, double* x_host, flgpu_solve_info* info_out) {
    if (!x_host) return set_error(FLGPU_EINVAL, "flgpu_solve_noalloc: x is required (host, rows values)");
    if (sp->precision != FLGPU_FP64)
        return set_error(FLGPU_EUNSUPPORTED, "flgpu_solve_noalloc: FP64 only (precision %d)", sp->precision);
    if (sp->ksp != FLGPU_KSP_CG && sp->ksp != FLGPU_KSP_FCG)
        return set_error(FLGPU_EUNSUPPORTED, "flgpu_solve_noalloc: cg or fcg only (ksp %d)", sp->ksp);
    if (sp->pc != FLGPU_PC_NONE && sp->pc != FLGPU_PC_JACOBI)
        return set_error(FLGPU_EUNSUPPORTED, "flgpu_solve_noalloc: pc none or jacobi only (pc %d)", sp->pc);
    unsigned char* base = noalloc_ptr(c->device);
    if (!base) return set_error(FLGPU_EINVAL, "flgpu_solve_noalloc: device %d was not set up by flgpu_init", c->device);
    const int n = c->rows;
    int maxlen = 0;
    for (int i = 0; i < n; i++) maxlen = std::max(maxlen, c->h_rowptr[i + 1] - c->h_rowptr[i]);
    const int rows_per = std::max(1, std::min(kRowBlock, kStreamNnz / std::max(1, maxlen)));
    const int nrb = (int)(((int64_t)n + rows_per - 1) / rows_per);
    KrylovWork k;  // every buffer a view of the array; nothing allocated or freed
    size_t need = 0;
    if (!noalloc_carve(base, n, c->nnz, nrb, k, &need))
        return set_error(FLGPU_EUNSUPPORTED,
                         "flgpu_solve_noalloc: a system of %d rows and %lld entries needs %zu bytes of solver work, "
                         "more than the %zu bytes of its fixed array",
                         n, (long long)c->nnz, need, kNoAllocBytes);
    Scal h_scal;  // pageable: read_scal / write_scal synchronise
    k.n = n;
    k.nnz = c->nnz;
    k.use16 = false;
    k.nrb = nrb;
    k.h_scal = &h_scal;
    k.h_scal_owned = false;
    k.nblk = std::max(1, (int)std::min<int64_t>(kMaxVecGrid, ((int64_t)n + kVecBlock - 1) / kVecBlock));
    flgpu_solve_info info{};
    KrylovWork* saved = c->kw;
    c->kw = &k;
    const int rc = [&]() -> int {
        hipLaunchKernelGGL(k_fixed_row_blocks, dim3(grid_for((int64_t)nrb + 1, 256)), dim3(256), 0, c->stream, n,
                           rows_per, nrb, c->rowptr.p, k.rb.p, k.rbk.p);
        FLGPU_HIP(hipGetLastError());
        if (!sp->start_from_zero)
            FLGPU_HIP(hipMemcpyAsync(k.x.p, x_host, sizeof(double) * n, hipMemcpyHostToDevice, c->stream));
        FLGPU_TRY(build_reduced(c, &k, false, sp->start_from_zero != 0));
        FLGPU_TRY(run_cg<double>(c, sp, &info, false));
        hipLaunchKernelGGL(k_finish_x, dim3(grid_for(n, kVecBlock)), dim3(kVecBlock), 0, c->stream, n, k.x.p,
                           c->rhs.p, c->inactive.p, c->have_inactive ? 1 : 0);
        FLGPU_HIP(hipGetLastError());
        FLGPU_HIP(hipMemcpyAsync(x_host, k.x.p, sizeof(double) * n, hipMemcpyDeviceToHost, c->stream));
        FLGPU_HIP(hipStreamSynchronize(c->stream));
        return FLGPU_OK;
    }();
    c->kw = saved;
    if (rc != FLGPU_OK) {
        (void)hipStreamSynchronize(c->stream);  // no kernel still reads the views
        return rc;
    }
    if (info_out) *info_out = info;
    return FLGPU_OK;
}

int solution_get(flgpu_ctx* c, double* x) {
    if (!c->kw || !c->kw->have_x) return set_error(FLGPU_EINVAL, "flgpu_solution_get: no solution");
    FLGPU_TRY(copy_out(c, x, c->kw->x.p, sizeof(double) * c->rows));
    FLGPU_HIP(hipStreamSynchronize(c->stream));
    return FLGPU_OK;
}

int csr_mult(flgpu_ctx* c, const double* x, double* y) {
    FLGPU_TRY(ensure_work(c, false));
    KrylovWork* k = c->kw;
    DevBuf<double> dx, dy;
    FLGPU_TRY(dx.upload(x, c->cols, c->stream));
    FLGPU_TRY(dy.alloc(c->rows));
    FLGPU_TRY((spmv<double, double, double>(c, k, c->A.p, dx.p, dy.p, nullptr, 0, nullptr)));
    FLGPU_HIP(hipMemcpyAsync(y, dy.p, sizeof(double) * c->rows, hipMemcpyDeviceToHost, c->stream));
    FLGPU_HIP(hipStreamSynchronize(c->stream));
    return FLGPU_OK;
}

// rt = D r (the residual in the factor's scaled space)
__global__ void __launch_bounds__(kVecBlock)
k_scale_res(int n, const double* __restrict__ r, const float* __restrict__ dsq, double* __restrict__ rt) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
        rt[i] = r[i] * (double)dsq[i];
}

int pc_apply_host(flgpu_ctx* c, const flgpu_solver_params* sp, const double* r, double* z) {
    if (sp->pc != FLGPU_PC_NONE && sp->pc != FLGPU_PC_JACOBI && sp->pc != FLGPU_PC_SOR &&
        sp->pc != FLGPU_PC_LEARNED && sp->pc != FLGPU_PC_FSAI)
        return set_error(FLGPU_EUNSUPPORTED, "flgpu_pc_apply: pc %d", sp->pc);
    FLGPU_TRY(ensure_work(c, false));
    KrylovWork* k = c->kw;
    FLGPU_TRY(build_reduced(c, k, false, true));
    k->prepared = true;
    k->prepared_mixed = false;
    const int n = c->rows;
    FLGPU_HIP(hipMemcpyAsync(k->r.p, r, sizeof(double) * n, hipMemcpyHostToDevice, c->stream));
    if (sp->pc == FLGPU_PC_SOR) {
        FLGPU_TRY(ssor_prepare<double>(c, k, k->val64.p));
        FLGPU_TRY(ssor_sweeps<double>(c, k, k->r.p, k->z.p, nullptr));
    } else if (sp->pc == FLGPU_PC_LEARNED || sp->pc == FLGPU_PC_FSAI) {
        FLGPU_TRY(learned_prepare(c, false, sp->pc == FLGPU_PC_FSAI));
        hipLaunchKernelGGL(k_scale_res, dim3(k->nblk), dim3(kVecBlock), 0, c->stream, n, k->r.p, learned_scale(c),
                           k->rt.p);
        FLGPU_HIP(hipGetLastError());
        int np = 0;
        FLGPU_TRY(learned_precond_apply<double>(c, k->r.p, k->rt.p, k->z.p, k->y.p, k->r.p, k->part(PART_PC), &np,
                                                nullptr));
    } else {
        hipLaunchKernelGGL((k_gm_precres<double>), dim3(k->nblk), dim3(kVecBlock), 0, c->stream, n, k->r.p,
                           sp->pc == FLGPU_PC_JACOBI ? k->dinv.p : nullptr, k->z.p);
        FLGPU_HIP(hipGetLastError());
    }
    FLGPU_HIP(hipMemcpyAsync(z, k->z.p, sizeof(double) * n, hipMemcpyDeviceToHost, c->stream));
    FLGPU_HIP(hipStreamSynchronize(c->stream));
    return FLGPU_OK;
}

const double* reduced_values(flgpu_ctx* c) { return c->kw ? c->kw->val64.p : nullptr; }

int reduced_prepare(flgpu_ctx* c) {
    if (c->kw && c->kw->prepared && c->kw->prepared_mixed) return FLGPU_OK;
    return solver_prepare(c, FLGPU_MIXED);
}

int solver_prepare(flgpu_ctx* c, int precision) {
    const bool mixed = precision == FLGPU_MIXED;
    FLGPU_TRY(ensure_work(c, mixed));
    FLGPU_TRY(build_reduced(c, c->kw, mixed, true));
    FLGPU_HIP(hipMemsetAsync(c->kw->p.p, 0, sizeof(double) * c->rows, c->stream));
    if (mixed) FLGPU_HIP(hipMemsetAsync(c->kw->p32.p, 0, sizeof(float) * c->rows, c->stream));
    FLGPU_HIP(hipStreamSynchronize(c->stream));
    c->kw->prepared_mixed = mixed;
    c->kw->prepared = true;
    return FLGPU_OK;
}

// Streams through a buffer (read and write) to evict the SpMV's operands
// from the L2 caches and the Infinity Cache before a cold timing.
__global__ void __launch_bounds__(256) k_flush(uint4* __restrict__ buf, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        uint4 v = buf[i];
        v.x += 1u;
        buf[i] = v;
    }
}

// reps products, each after a flush of flush_mib MiB and timed alone
// between its own events; *ms = their mean.
int time_spmv_cold(flgpu_ctx* c, int precision, int reps, int flush_mib, double* ms) {
    const bool mixed = precision == FLGPU_MIXED;
    if (!c->kw || !c->kw->prepared || (mixed && !c->kw->prepared_mixed))
        FLGPU_TRY(solver_prepare(c, precision));
    KrylovWork* k = c->kw;
    const int64_t n16 = (int64_t)flush_mib * (1 << 20) / 16;
    DevBuf<uint4> fb;
    FLGPU_TRY(fb.alloc((size_t)n16));
    FLGPU_HIP(hipMemsetAsync(fb.p, 0, sizeof(uint4) * n16, c->stream));
    std::vector<hipEvent_t> ev(2 * (size_t)reps, nullptr);
    int rc = FLGPU_OK;
    for (auto& e : ev)
        if (hipEventCreate(&e) != hipSuccess) rc = set_error(FLGPU_EHIP, "flgpu_time_spmv_cold: hipEventCreate");
    for (int r = 0; r < reps && rc == FLGPU_OK; r++) {
        hipLaunchKernelGGL(k_flush, dim3(2048), dim3(256), 0, c->stream, fb.p, n16);
        if (hipEventRecord(ev[2 * r], c->stream) != hipSuccess) rc = set_error(FLGPU_EHIP, "hipEventRecord");
        if (rc == FLGPU_OK)
            rc = mixed ? spmv<float, float, float>(c, k, k->val32.p, k->p32.p, k->w32.p, nullptr, 0, nullptr)
                       : spmv<double, double, double>(c, k, k->val64.p, k->p.p, k->w.p, nullptr, 0, nullptr);
        if (rc == FLGPU_OK && hipEventRecord(ev[2 * r + 1], c->stream) != hipSuccess)
            rc = set_error(FLGPU_EHIP, "hipEventRecord");
    }
    if (rc == FLGPU_OK && hipStreamSynchronize(c->stream) != hipSuccess)
        rc = set_error(FLGPU_EHIP, "flgpu_time_spmv_cold: hipStreamSynchronize");
    double sum = 0.0;
    for (int r = 0; r < reps && rc == FLGPU_OK; r++) {
        float t = 0.f;
        if (hipEventElapsedTime(&t, ev[2 * r], ev[2 * r + 1]) != hipSuccess)
            rc = set_error(FLGPU_EHIP, "hipEventElapsedTime");
        sum += t;
    }
    for (auto& e : ev)
        if (e) (void)hipEventDestroy(e);
    if (rc == FLGPU_OK) *ms = sum / reps;
    return rc;
}

// Bare solver-matrix SpMV w = A p, timed with HIP events on the stream.
int time_spmv(flgpu_ctx* c, int precision, int reps, double* ms) {
    const bool mixed = precision == FLGPU_MIXED;
    if (!c->kw || !c->kw->prepared || (mixed && !c->kw->prepared_mixed))
        FLGPU_TRY(solver_prepare(c, precision));
    KrylovWork* k = c->kw;
    hipEvent_t e0, e1;
    FLGPU_HIP(hipEventCreate(&e0));
    FLGPU_HIP(hipEventCreate(&e1));
    FLGPU_HIP(hipEventRecord(e0, c->stream));
    for (int r = 0; r < reps; r++) {
        if (mixed)
            FLGPU_TRY((spmv<float, float, float>(c, k, k->val32.p, k->p32.p, k->w32.p, nullptr, 0, nullptr)));
        else
            FLGPU_TRY((spmv<double, double, double>(c, k, k->val64.p, k->p.p, k->w.p, nullptr, 0, nullptr)));
    }
    FLGPU_HIP(hipEventRecord(e1, c->stream));
    FLGPU_HIP(hipEventSynchronize(e1));
    float t = 0.f;
    FLGPU_HIP(hipEventElapsedTime(&t, e0, e1));
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    *ms = (double)t / reps;
    return FLGPU_OK;
}

}  // namespace flgpu
