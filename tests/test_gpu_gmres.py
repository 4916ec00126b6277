"""The device-driven GMRES at the sizes where its kernels change: systems of
one block, of at most 16 and of more blocks (how the block sums are taken),
bases of up to 8, 16 and 32 vectors in registers and longer ones, restarts
that end a cycle mid-way, sliced ELL and CSR products, FP64 and mixed.

The reference is the oracle's own solve of the same system to a relative
residual of 1e-13; both residuals bound the difference by
cond(D^-1 A) (1e-13 + rtol), and these systems' condition numbers are below
1e3 (mass-dominated) and 2e4 (the Poisson one), hence the tolerances.
"""
import numpy as np
import pytest

import oracle as O
from fluidity_amd import cg, meshgen as M

pytestmark = pytest.mark.gpu

# name, cells a side, restart, precision, preconditioner, rtol, tolerance on x
CASES = [
    ("c1", 2, 30, "fp64", "jacobi", 1e-11, 1e-8),     # 9 rows: one partly filled block
    ("c1", 21, 30, "fp64", "jacobi", 1e-11, 1e-8),    # 484 rows: one workgroup, one row a thread
    ("c1", 22, 30, "fp64", "jacobi", 1e-11, 1e-8),    # 529 rows: more
    ("c1", 22, 7, "mixed", "none", 1e-9, 1e-6),       # and several cycles
    ("c1", 45, 32, "fp64", "jacobi", 1e-11, 1e-8),    # 2116 rows: the most
    ("c1", 47, 30, "fp64", "jacobi", 1e-11, 1e-8),    # 2304 rows: a launch a step
    ("c1p2", 9, 30, "fp64", "jacobi", 1e-11, 1e-8),   # quadratic triangles, rows sorted by length
    ("c1", 90, 30, "fp64", "jacobi", 1e-11, 1e-8),    # 8281 rows: 17 blocks
    ("c1", 90, 1, "fp64", "jacobi", 1e-9, 1e-6),      # a cycle an iteration
    ("c1", 40, 8, "fp64", "jacobi", 1e-11, 1e-8),     # register bases of 8 and cycles of exactly that
    ("c1", 40, 9, "fp64", "sor", 1e-11, 1e-8),
    ("c1", 40, 17, "mixed", "jacobi", 1e-9, 1e-6),
    ("c2", 9, 33, "fp64", "jacobi", 1e-11, 1e-7),     # Poisson: bases beyond the registers
    ("c2", 9, 65, "fp64", "none", 1e-11, 1e-7),
    ("c2", 20, 100, "fp64", "jacobi", 1e-11, 1e-7),
    ("c2", 20, 70, "mixed", "jacobi", 1e-8, 1e-5),
    ("c3", 3, 30, "fp64", "jacobi", 1e-11, 1e-8),     # quadratic: not the sliced ELL of equal rows
    ("c3", 3, 30, "mixed", "sor", 1e-9, 1e-6),
]


@pytest.mark.parametrize("name,scale,restart,precision,pc,rtol,tol", CASES)
def test_gmres_against_oracle(require_gpu, name, scale, restart, precision, pc, rtol, tol):
    print(f"\n[case] gmres {name} {scale} restart {restart} {precision} {pc}", flush=True)
    cfg = M.config(name, seed=17, scale=scale)
    ref = O.reference_system(cfg)
    pr = cg.problem_from_config(cfg)
    cg.assemble_advection_diffusion_cg(pr, cg.options_from_config(cfg), cfg.dt)
    cg.apply_dirichlet_conditions(pr, cfg.mesh.boundary, 0.0, cfg.dt)
    so = cg.SolverOptions("gmres", pc, relative_error=rtol, restart=restart, precision=precision)
    x, info = cg.petsc_solve(pr, so)
    xr, _, reason, _, _ = O.petsc_solve("gmres", "jacobi", 1e-13, ref["sparsity"], ref["A"], ref["inactive"],
                                        ref["rhs"])
    assert info.reason > 0 and reason > 0
    assert np.max(np.abs(x - xr)) <= tol * np.max(np.abs(xr))
    x2, info2 = cg.petsc_solve(pr, so)  # a second solve on the same work arrays repeats it bit for bit
    assert np.array_equal(x, x2) and info2.its == info.its
    pr.close()


def test_gmres_iteration_limit_and_zero_rhs(require_gpu):
    """max_its ends the solve inside a cycle with PETSc's KSP_DIVERGED_ITS
    and that many iterations; a zero right-hand side converges at once."""
    cfg = M.config("c2", seed=17, scale=8)
    pr = cg.problem_from_config(cfg)
    cg.assemble_advection_diffusion_cg(pr, cg.options_from_config(cfg), cfg.dt)
    cg.apply_dirichlet_conditions(pr, cfg.mesh.boundary, 0.0, cfg.dt)
    for limit in (1, 5, 13):
        _, info = cg.petsc_solve(pr, cg.SolverOptions("gmres", "jacobi", relative_error=1e-14, restart=6,
                                                      max_iterations=limit))
        assert (info.reason, info.its) == (-3, limit)
    import ctypes as C
    from fluidity_amd import lib as L
    A, rhs, inact = pr.matrix()
    zero = np.zeros_like(rhs)
    L.check(pr.lib.flgpu_matrix_set(pr.ctx, L.ptr(A), L.ptr(zero), L.ptr(inact)), "flgpu_matrix_set")
    x, info = cg.petsc_solve(pr, cg.SolverOptions("gmres", "jacobi", relative_error=1e-10))
    assert info.reason == 3 and info.its == 0 and not np.any(x)
    pr.close()


# A matrix scaled by 2^a and a solution by 2^x change no rounding in the
# solver while nothing leaves the range: the same iterations and exactly the
# scaled solution, also where the FP32 residual times the matrix would leave
# it (below 1e-38 once the residual has fallen, above 3e38).
@pytest.mark.parametrize("n,spmv", [(40, ""), (90, ""), (47, "csr")])
@pytest.mark.parametrize("a,x", [(-60, -40), (60, 85)])
def test_mixed_gmres_in_any_units(require_gpu, monkeypatch, n, spmv, a, x):
    from fluidity_amd import lib as L
    print(f"\n[case] mixed gmres {n} {spmv} matrix 2^{a} solution 2^{x}", flush=True)
    if spmv:
        monkeypatch.setenv("FLGPU_SPMV", spmv)
    cfg = M.config("c1", seed=17, scale=n)
    pr = cg.problem_from_config(cfg)
    cg.assemble_advection_diffusion_cg(pr, cg.options_from_config(cfg), cfg.dt)
    cg.apply_dirichlet_conditions(pr, cfg.mesh.boundary, 0.0, cfg.dt)
    so = cg.SolverOptions("gmres", "jacobi", relative_error=1e-9, precision="mixed")
    A, rhs, inact = pr.matrix()
    # entries of one size (the prescribed values, taken as they are, zero), so that none is below the range by itself
    rhs = np.where(inact != 0, 0.0, np.max(np.abs(rhs)) * np.random.default_rng(3).uniform(0.5, 1.5, rhs.size))
    for sa, sb in ((0, 0), (a, a + x)):
        As, bs = np.ldexp(A, sa), np.ldexp(rhs, sb)
        L.check(pr.lib.flgpu_matrix_set(pr.ctx, L.ptr(As), L.ptr(bs), L.ptr(inact)), "flgpu_matrix_set")
        got, info = cg.petsc_solve(pr, so)
        if sa == 0:
            want, its = got, info.its
    assert info.reason == 2 and info.its == its
    assert np.array_equal(got, np.ldexp(want, x))
    pr.close()
