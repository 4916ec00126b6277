"""CG, flexible CG with a factor and the single-reduction CG where the block
sums and grids of their kernels change: one block, one row more than a
block, one block per CU and more than one row group a thread; products of
one slice, of uneven groups, and of several rounds.  The reference is the
oracle's Jacobi-CG to a relative residual of 1e-13; the difference is bounded
by cond(D^-1 A) (1e-13 + rtol), and these Poisson systems' condition numbers
are below 0.7 (cells a side)^2.
"""
import numpy as np
import pytest

import oracle as O
from fluidity_amd import cg, meshgen as M

pytestmark = pytest.mark.gpu

METHODS = [("cg", "jacobi", "fp64"), ("cg", "jacobi", "mixed"), ("cg", "none", "fp64"), ("cg", "fsai", "fp64"),
           ("fcg", "fsai", "mixed"), ("cg", "sor", "fp64"), ("pipecg", "jacobi", "fp64"), ("pipecg", "fsai", "mixed")]


@pytest.mark.parametrize("scale", [2, 3, 9, 10, 39, 64])  # 27, 64, 1000, 1331, 64000 and 274625 rows
def test_cg_against_oracle(require_gpu, scale):
    cfg = M.config("c2", seed=23, scale=scale)
    ref = O.reference_system(cfg)
    xr, _, reason, _, _ = O.petsc_solve("cg", "jacobi", 1e-13, ref["sparsity"], ref["A"], ref["inactive"], ref["rhs"])
    assert reason > 0
    pr = cg.problem_from_config(cfg)
    cg.assemble_advection_diffusion_cg(pr, cg.options_from_config(cfg), cfg.dt)
    cg.apply_dirichlet_conditions(pr, cfg.mesh.boundary, 0.0, cfg.dt)
    rtol = 1e-10
    tol = 0.7 * max(scale, 3) ** 2 * (rtol + 1e-13)
    for ksp, pc, precision in METHODS:
        print(f"\n[case] {ksp} {pc} {precision} rows {cfg.mesh.nnodes}", flush=True)
        so = cg.SolverOptions(ksp, pc, relative_error=rtol, precision=precision, norm="unpreconditioned")
        x, info = cg.petsc_solve(pr, so)
        assert info.reason > 0 and info.true_relres <= rtol * (1 + 1e-6), (ksp, pc, precision, info.true_relres)
        assert np.linalg.norm(x - xr) <= tol * np.linalg.norm(xr), (ksp, pc, precision)
        x2, info2 = cg.petsc_solve(pr, so)
        assert np.array_equal(x, x2) and info2.its == info.its  # fixed order of every sum
    pr.close()


def renumbered(cfg, seed):
    """The linear mesh with its nodes numbered at random: rows share no
    column offsets, so the products keep their column indices."""
    m = cfg.mesh
    perm = np.random.default_rng(seed).permutation(m.nnodes)  # old node -> new
    inv = np.argsort(perm)
    assert np.array_equal(m.ndglno, m.ndglno_x)
    m.ndglno = (perm[m.ndglno - 1] + 1).astype(m.ndglno.dtype)
    m.ndglno_x = m.ndglno.copy()
    m.X, m.node_pos = m.X[inv].copy(), m.node_pos[inv].copy()
    m.boundary = np.sort(perm[m.boundary - 1] + 1).astype(m.boundary.dtype)
    cfg.T = cfg.T[inv].copy()
    if cfg.U is not None:
        cfg.U = cfg.U[inv].copy()
    return cfg


# rows in order with and without shared column offsets, and quadratic rows
# sorted in one window, at a window's 2048 rows and over several.  The
# quadratic systems are mass-dominated: condition numbers below 1e3.
@pytest.mark.parametrize("name,scale,shuffle", [("c2", 3, True), ("c2", 13, True), ("c2", 13, False),
                                                ("c3", 5, False), ("c3", 7, False), ("c3", 9, False)])
def test_products_by_numbering(require_gpu, name, scale, shuffle):
    cfg = M.config(name, seed=29, scale=scale)
    if shuffle:
        cfg = renumbered(cfg, 5)
    print(f"\n[case] {name} rows {cfg.mesh.nnodes} shuffled {shuffle}", flush=True)
    ref = O.reference_system(cfg)
    meth = "cg" if name == "c2" else "gmres"
    xr, _, reason, _, _ = O.petsc_solve(meth, "jacobi", 1e-13, ref["sparsity"], ref["A"], ref["inactive"], ref["rhs"])
    assert reason > 0
    pr = cg.problem_from_config(cfg)
    cg.assemble_advection_diffusion_cg(pr, cg.options_from_config(cfg), cfg.dt)
    cg.apply_dirichlet_conditions(pr, cfg.mesh.boundary, 0.0, cfg.dt)
    tol = (0.7 * max(scale, 3) ** 2 if name == "c2" else 1e3) * (1e-10 + 1e-13)
    for precision in ("fp64", "mixed"):
        x, info = cg.petsc_solve(pr, cg.SolverOptions(meth, "jacobi", relative_error=1e-10, precision=precision,
                                                      norm="unpreconditioned" if meth == "cg" else "preconditioned"))
        assert info.reason > 0 and np.linalg.norm(x - xr) <= tol * np.linalg.norm(xr), precision
    pr.close()


# Quadratic elements numbered at random on both sides of a million entries:
# rows sorted into slices, and the CSR products.
@pytest.mark.parametrize("scale", [15, 17])  # 29791 rows of 807661 entries; 42875 rows of 1170281
def test_quadratic_products_numbered_at_random(require_gpu, scale):
    cfg = M.config("c3", seed=31, scale=scale)
    m = cfg.mesh
    perm = np.random.default_rng(7).permutation(m.nnodes)
    inv = np.argsort(perm)
    m.ndglno = (perm[m.ndglno - 1] + 1).astype(m.ndglno.dtype)
    m.node_pos = m.node_pos[inv].copy()
    m.boundary = np.sort(perm[m.boundary - 1] + 1).astype(m.boundary.dtype)
    cfg.T, cfg.U = cfg.T[inv].copy(), cfg.U[inv].copy()
    print(f"\n[case] c3 numbered at random, rows {m.nnodes}", flush=True)
    ref = O.reference_system(cfg)
    xr, _, reason, _, _ = O.petsc_solve("gmres", "jacobi", 1e-13, ref["sparsity"], ref["A"], ref["inactive"],
                                        ref["rhs"])
    assert reason > 0
    pr = cg.problem_from_config(cfg)
    cg.assemble_advection_diffusion_cg(pr, cg.options_from_config(cfg), cfg.dt)
    cg.apply_dirichlet_conditions(pr, cfg.mesh.boundary, 0.0, cfg.dt)
    for precision in ("fp64", "mixed"):
        x, info = cg.petsc_solve(pr, cg.SolverOptions("gmres", "jacobi", relative_error=1e-10, precision=precision))
        # mass-dominated: condition numbers below 1e3
        assert info.reason > 0 and np.linalg.norm(x - xr) <= 1e3 * 1e-10 * np.linalg.norm(xr), precision
    pr.close()


@pytest.mark.parametrize("ksp,pc", [("cg", "jacobi"), ("cg", "sor"), ("fcg", "fsai"), ("pipecg", "jacobi"),
                                    ("pipecg", "fsai")])
def test_batches_of_iterations_change_nothing(require_gpu, ksp, pc):
    """The iterations that are queued between two looks at the scalars, few or
    more than the solve takes, and ended by convergence or by the limit."""
    cfg = M.config("c2", seed=41, scale=12)
    pr = cg.problem_from_config(cfg)
    cg.assemble_advection_diffusion_cg(pr, cg.options_from_config(cfg), cfg.dt)
    cg.apply_dirichlet_conditions(pr, cfg.mesh.boundary, 0.0, cfg.dt)
    for limit in (1, 2, 5, 16, 17, 10000):
        seen = []
        for every in (1, 2, 5, 16, 300):
            print(f"\n[case] {ksp} {pc} limit {limit} batches of {every}", flush=True)
            so = cg.SolverOptions(ksp, pc, relative_error=1e-9, max_iterations=limit, check_every=every)
            x, info = cg.petsc_solve(pr, so)
            assert info.reason == (2 if limit == 10000 else -3) and (limit == 10000 or info.its == limit)
            seen.append((info.its, x))
        assert all(its == seen[0][0] and np.array_equal(x, seen[0][1]) for its, x in seen)
    pr.close()
