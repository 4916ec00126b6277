"""The SSOR sweeps on each side of the choice between one workgroup (z in
LDS) and a launch per colour, and at the edges of slices and batches: the
preconditioner applied equals the oracle's sweep bit for bit (as in
test_gpu_sor.py, whose systems all take one workgroup).
"""
import ctypes as C

import numpy as np
import pytest

import oracle as O
from fluidity_amd import cg, lib as L, meshgen as M
from test_gpu_sor import gpu_system, reduced_full_pattern

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,scale", [
    ("c1", 2),     # 9 rows
    ("c1", 126),   # 16129 rows: z just fits the workgroup's LDS
    ("c1", 128),   # 16641 rows: it does not
    ("c2", 24),    # 15625 rows of 15 entries
    ("c2", 31),    # 32768 rows: a launch per colour
    ("c3", 13),    # 19683 rows of up to 65 entries, sorted by length
])
def test_sweep_is_the_oracles(require_gpu, name, scale):
    cfg = M.config(name, seed=12, scale=scale)
    print(f"\n[case] ssor {name} scale {scale} rows {cfg.mesh.nnodes}", flush=True)
    pr = gpu_system(cfg)
    A, rhs, inact = pr.matrix()
    sp = pr.sparsity
    findrm, colm, val = reduced_full_pattern({"sparsity": (sp.findrm, sp.colm, sp.centrm), "A": A, "rhs": rhs,
                                              "inactive": inact})
    r = np.random.default_rng(3).standard_normal(cfg.mesh.nnodes)
    z = np.zeros_like(r)
    L.check(pr.lib.flgpu_pc_apply(pr.ctx, C.byref(cg.SolverOptions("cg", "sor").params()), L.ptr(r), L.ptr(z)),
            "flgpu_pc_apply")
    pr.close()
    zo = O.ssor_apply(findrm, colm, val, r)
    assert np.array_equal(z, zo), np.max(np.abs(z - zo))
