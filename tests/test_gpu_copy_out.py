"""Results copied to the caller through the pinned slots: sizes below, at and
past the size where that path starts and its chunks, exact values, fresh and
reused destinations, and copies of two contexts on two threads at once."""
import threading

import numpy as np
import pytest

from fluidity_amd import cg, lib as L, meshgen as M

pytestmark = pytest.mark.gpu


def bound(n):
    mesh = M.square_tris(n)
    pr = cg.CGProblem(mesh)
    return pr, pr.sparsity.nnz


# entries: below 4 MiB, just past it (a short last chunk), several chunks a thread
@pytest.mark.parametrize("n", [200, 274, 275, 520])
def test_values_arrive_whole(require_gpu, n):
    pr, nnz = bound(n)
    print(f"\n[case] copy of {8 * nnz} bytes", flush=True)
    rhs = np.arange(pr.mesh.nnodes, dtype=np.float64)
    back = np.empty(nnz)
    for seed in (1, 2):
        A = np.random.default_rng(seed).standard_normal(nnz)
        L.check(pr.lib.flgpu_matrix_set(pr.ctx, L.ptr(A), L.ptr(rhs), None), "flgpu_matrix_set")
        got, r, _ = pr.matrix()
        assert np.array_equal(got, A) and np.array_equal(r, rhs)
        L.check(pr.lib.flgpu_matrix_get(pr.ctx, L.ptr(back), None, None), "flgpu_matrix_get")
        assert np.array_equal(back, A)
    pr.close()


def test_two_contexts_on_two_threads(require_gpu):
    prs = [bound(n)[0] for n in (400, 520)]
    want = [np.random.default_rng(k).standard_normal(p.sparsity.nnz) for k, p in enumerate(prs)]
    for p, A in zip(prs, want):
        L.check(p.lib.flgpu_matrix_set(p.ctx, L.ptr(A), L.ptr(np.zeros(p.mesh.nnodes)), None), "flgpu_matrix_set")
    ok = [True, True]

    def read(k):
        for _ in range(10):
            ok[k] = ok[k] and np.array_equal(prs[k].matrix()[0], want[k])

    threads = [threading.Thread(target=read, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert ok == [True, True]
    for p in prs:
        p.close()


@pytest.mark.parametrize("n", [4, 8])  # checked on the host, on the device
def test_cmc_pattern_check(require_gpu, n):
    """The first column out of range is named, and the last accepted pattern
    stays in place."""
    mesh = M.cube_tets(n)
    pr = cg.CGProblem(mesh)
    pm = cg.vertex_pressure_mesh(pr)
    cg.bind_pressure_mesh(pr, pm)
    cg.construct_momentum_ct(pr, pm)
    f, c = cg.cmc_sparsity(pm, mesh.nnodes)
    good = cg.assemble_masslumped_cmc(pr, f, c)
    for bad in (0, mesh.nnodes + 1, -5):
        broken = c.copy()
        broken[[17, 40]] = bad
        with pytest.raises(L.FlgpuError, match=rf"colm\(18\) = {bad} out of 1"):
            cg.assemble_masslumped_cmc(pr, f, broken)
    assert np.array_equal(cg.assemble_masslumped_cmc(pr, f, c), good)
    pr.close()


def test_pinned_destination(require_gpu):
    """Memory that the caller has pinned, at an offset too, takes the direct
    transfer at every size."""
    import ctypes as C
    pr, nnz = bound(520)
    path = next(ln.split()[-1] for ln in open("/proc/self/maps") if "libamdhip64" in ln)  # the library's runtime
    hip = C.CDLL(path)
    p = C.c_void_p()
    assert hip.hipHostMalloc(C.byref(p), C.c_size_t(8 * (nnz + 3)), 0) == 0
    dst = np.frombuffer((C.c_double * (nnz + 3)).from_address(p.value), np.float64)
    A = np.random.default_rng(4).standard_normal(nnz)
    L.check(pr.lib.flgpu_matrix_set(pr.ctx, L.ptr(A), L.ptr(np.zeros(pr.mesh.nnodes)), None), "flgpu_matrix_set")
    for off in (0, 3):
        dst[:] = -1.0
        L.check(pr.lib.flgpu_matrix_get(pr.ctx, C.c_void_p(p.value + 8 * off), None, None), "flgpu_matrix_get")
        assert np.array_equal(dst[off:off + nnz], A)
    pr.close()
    assert hip.hipHostFree(p) == 0
