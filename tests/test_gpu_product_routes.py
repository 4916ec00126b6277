"""The forms that a matrix's products take -- slices in order or sorted,
diagonal slices, column indices of 16 and 32 bits, the CSR products with each
number of lanes a row -- against each other and against numpy, on patterns
that are no mesh's.

The matrices, right-hand sides and first iterates are small integers, so that
every sum of one CG or GMRES step is exact in FP32 and FP64 (below 2^24), in
any order: a step's result is the same bits whichever form the product takes,
and one wrong, missing or doubled entry changes it.
"""
import ctypes as C

import numpy as np
import pytest

import oracle as O
from fluidity_amd import cg, lib as L, meshgen as M

pytestmark = pytest.mark.gpu


def pattern(rows):
    """Sparsity from each row's sorted columns (0-based), the diagonal among them."""
    lens = np.array([len(r) for r in rows])
    colm = np.concatenate(rows)
    findrm = np.concatenate([[1], 1 + np.cumsum(lens)]).astype(np.int32)
    row = np.repeat(np.arange(len(rows)), lens)
    centrm = (np.nonzero(colm == row)[0] + 1).astype(np.int32)
    assert centrm.size == len(rows)
    return cg.Sparsity(findrm, (colm + 1).astype(np.int32), centrm)


def banded(n, offsets):
    """Shared offsets: diagonal slices."""
    return [np.array([i + d for d in offsets if 0 <= i + d < n]) for i in range(n)]


def lengths(n, lens, seed, near=None):
    """Random columns, lens[i % len(lens)] of them a row, anywhere or within `near`."""
    g = np.random.default_rng(seed)
    out = []
    for i in range(n):
        lo, hi = (0, n) if near is None else (max(0, i - near), min(n, i + near + 1))
        k = min(lens[i % len(lens)], hi - lo)
        c = np.unique(np.append(g.integers(lo, hi, k), i))
        out.append(c)
    return out


def mixed_slices(n, seed):
    """Banded and random rows by turns of 100, so that slices of both kinds alternate."""
    b, r = banded(n, (-40, -3, -1, 0, 1, 3, 40)), lengths(n, [7], seed)
    return [b[i] if i // 100 % 2 else r[i] for i in range(n)]


PATTERNS = {
    "two rows": lambda: [np.array([0, 1])] * 2,
    "diagonal only": lambda: [np.array([i]) for i in range(300)],
    "one slice": lambda: banded(64, (-7, -1, 0, 1, 7)),
    "slices and a row": lambda: banded(641, (-7, -1, 0, 1, 7)),
    "banded": lambda: banded(5000, (-70, -69, -1, 0, 1, 69, 70)),
    "random, 16 bits": lambda: lengths(30000, [9], 1),
    "random, 32 bits": lambda: lengths(40000, [9], 2),
    "alternating, 32 bits": lambda: mixed_slices(50000, 3),
    "sorted, a window": lambda: lengths(256, [4, 4, 4, 12], 4),
    "sorted, windows and a row": lambda: lengths(2561, [4, 4, 4, 12], 5),
    "sorted, near": lambda: lengths(20000, [4, 4, 12], 6, near=400),
    "sorted, 32 bits": lambda: lengths(40000, [4, 4, 12], 7),
    "sorted, banded": lambda: [r if i % 2 else r[np.abs(r - i) < 50] for i, r in
                               enumerate(banded(9000, (-90, -80, -9, -1, 0, 1, 9, 80, 90)))],
    "csr, 4 lanes, grid strides": lambda: lengths(140000, [1, 1, 12], 8, near=3000),
    "csr, 8 lanes": lambda: lengths(60000, [2, 2, 27], 9, near=3000),
    "csr, 16 lanes": lambda: lengths(70000, [3, 3, 60], 10, near=3000),
    "csr, 32 lanes, grid strides": lambda: lengths(30000, [6, 6, 120], 11),
    "csr, 64 lanes, grid strides": lambda: lengths(12000, [20, 20, 260], 12),
    "csr, a long row": lambda: lengths(3000, [4], 13)[:-1] + [np.arange(3000)],
}


def system(sp, seed):
    g = np.random.default_rng(seed)
    n = sp.findrm.size - 1
    A = g.choice([-1.0, 1.0], sp.nnz)
    A[sp.centrm - 1] = 64.0
    return A, g.integers(-8, 9, n).astype(np.float64), g.integers(-2, 3, n).astype(np.float64)


def one_step(sp, A, b, x0, ksp, precision):
    n = b.size
    pr = cg.CGProblem(M.interval_mesh(n - 1), sparsity=sp)
    L.check(pr.lib.flgpu_matrix_set(pr.ctx, L.ptr(A), L.ptr(b), None), "flgpu_matrix_set")
    so = cg.SolverOptions(ksp, "none", relative_error=1e-14, max_iterations=1, restart=33, precision=precision,
                          start_from_zero=False)
    x, info = cg.petsc_solve(pr, so, x0)
    pr.close()
    assert info.its == 1
    return x


@pytest.mark.parametrize("name", list(PATTERNS))
def test_a_step_is_the_same_in_every_form(require_gpu, monkeypatch, name):
    print(f"\n[case] products of: {name}", flush=True)
    sp = pattern(PATTERNS[name]())
    A, b, x0 = system(sp, 17)
    n = b.size
    row = np.repeat(np.arange(n), np.diff(sp.findrm))
    mult = lambda v: np.bincount(row, A * v[sp.colm - 1], n)
    r = b - mult(x0)
    w = mult(r)
    assert np.max(np.abs(w)) < 2 ** 24
    want = {"cg": x0 + (r @ r) / (r @ w) * r, "gmres": x0 + (r @ w) / (w @ w) * r}  # least |b - A x| along r
    for ksp in ("cg", "gmres"):
        for precision in ("fp64", "mixed"):
            monkeypatch.delenv("FLGPU_SPMV", raising=False)
            x = one_step(sp, A, b, x0, ksp, precision)
            monkeypatch.setenv("FLGPU_SPMV", "csr")
            xc = one_step(sp, A, b, x0, ksp, precision)
            assert np.array_equal(x, xc), (ksp, precision)
            # x0, the step's length and the direction rounded to the precision
            tol = 8 * (2.0 ** -53 if precision == "fp64" else 2.0 ** -24) * (np.abs(x0) + np.abs(want[ksp] - x0))
            assert np.all(np.abs(x - want[ksp]) <= tol + 1e-300), (ksp, precision, np.max(np.abs(x - want[ksp])))


def regular_pairs(m, r, seed):
    """2m nodes, each of the last m joined to r of the first m and each of the
    first to r of the last, at random: rows of both triangular halves have one
    length in a slice and share no offsets."""
    g = np.random.default_rng(seed)
    pi, shift = g.permutation(m), np.sort(g.choice(m, r, replace=False))
    lo = (pi[:, None] + shift) % m                     # of node m + j
    rows = [[] for _ in range(2 * m)]
    for j in range(m):
        rows[m + j] = list(lo[j]) + [m + j]
        for c in lo[j]:
            rows[c].append(m + j)
    return [np.sort(np.array(q if i >= m else q + [i])) for i, q in enumerate(rows)]


@pytest.mark.parametrize("m", [32, 200, 5000, 35000])  # 32-bit columns in the last
@pytest.mark.parametrize("pc", ["fsai", "learned"])
def test_factor_halves_without_shared_offsets(require_gpu, monkeypatch, pc, m):
    from fluidity_amd import learned
    print(f"\n[case] {pc} halves of {2 * m} rows", flush=True)
    sp = pattern(regular_pairs(m, 6, m))
    n = 2 * m
    row = np.repeat(np.arange(n), np.diff(sp.findrm))
    A = np.where(row == sp.colm - 1, 7.0 + np.random.default_rng(1).uniform(0.5, 1.0, n)[row], -1.0)
    x = np.random.default_rng(2).standard_normal(n)
    b = np.bincount(row, A * x[sp.colm - 1], n)
    z = []
    for spmv in ("", "csr"):
        monkeypatch.setenv("FLGPU_SPMV", spmv)
        pr = cg.CGProblem(M.interval_mesh(n - 1), sparsity=sp)
        L.check(pr.lib.flgpu_matrix_set(pr.ctx, L.ptr(A), L.ptr(b), None), "flgpu_matrix_set")
        if pc == "learned":
            learned.set_params(pr, learned.load())
        zi = np.zeros(n)
        L.check(pr.lib.flgpu_pc_apply(pr.ctx, C.byref(cg.SolverOptions("cg", pc).params()), L.ptr(b), L.ptr(zi)),
                "flgpu_pc_apply")
        z.append(zi)
        for precision in ("fp64", "mixed"):
            got, info = cg.petsc_solve(pr, cg.SolverOptions("fcg", pc, relative_error=1e-10, precision=precision,
                                                            norm="unpreconditioned"))
            # diagonally dominant: eigenvalues within (0.5, 14.5), condition number below 29
            assert info.reason > 0 and np.linalg.norm(got - x) <= 29 * 1.1e-10 * np.linalg.norm(x), precision
        pr.close()
    assert np.any(z[0]) and np.array_equal(z[0], z[1])  # entry order is kept: the same sums


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_long_bases_over_more_rows_than_the_grid(require_gpu, precision):
    """GMRES bases past the 32 vectors held in registers, with more rows than
    256 blocks of 512 threads."""
    cfg = M.config("c2", seed=37, scale=51)  # 140608 rows
    print(f"\n[case] long basis, rows {cfg.mesh.nnodes}", flush=True)
    ref = O.reference_system(cfg)
    xr, _, reason, _, _ = O.petsc_solve("cg", "jacobi", 1e-12, ref["sparsity"], ref["A"], ref["inactive"], ref["rhs"])
    assert reason > 0
    pr = cg.problem_from_config(cfg)
    cg.assemble_advection_diffusion_cg(pr, cg.options_from_config(cfg), cfg.dt)
    cg.apply_dirichlet_conditions(pr, cfg.mesh.boundary, 0.0, cfg.dt)
    x, info = cg.petsc_solve(pr, cg.SolverOptions("gmres", "jacobi", relative_error=1e-7, restart=60,
                                                  precision=precision, max_iterations=400))
    # condition number below 0.7 (cells a side)^2, as in test_gpu_cg_sizes.py
    assert info.reason > 0 and info.its > 33
    assert np.linalg.norm(x - xr) <= 0.7 * 51 ** 2 * 1e-7 * np.linalg.norm(xr)
    pr.close()
