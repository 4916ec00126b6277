"""The host arrays that results are copied to: what the library does not write
is zero, and a pattern that is longer than its column array is refused before
the library would read and write past the arrays.  On the CPU, with the
library's calls replaced by ones that write what the C entry points write.
"""
import ctypes as C
from types import SimpleNamespace

import numpy as np
import pytest

from fluidity_amd import cg, lib as L

FINDRM = np.array([1, 3, 6], np.int32)  # 5 entries


def _fill(p, n, value):
    (C.c_double * n).from_address(p.value)[:] = [value] * n


class Library:
    def flgpu_matrix_get(self, ctx, A, rhs, inactive):
        _fill(A, 5, 1.0)
        _fill(rhs, 2, 2.0)
        (C.c_int32 * 2).from_address(inactive.value)[:] = [0, 1]
        return 0

    def flgpu_ct_assemble(self, ctx, ibp, const, rho, ct, ml):
        _fill(ct, 2 * 5, 3.0)
        _fill(ml, 2, 4.0)
        return 0

    def flgpu_cmc_assemble(self, ctx, im, rows, findrm, colm, out):
        _fill(out, 5, 5.0)
        return 0


@pytest.fixture
def garbage(monkeypatch):
    """np.empty memory that is never zero by luck."""
    monkeypatch.setattr(cg.np, "empty", lambda shape, dtype=np.float64: np.full(shape, -7, dtype))


def _problem(entries):
    pr = cg.CGProblem.__new__(cg.CGProblem)
    pr.lib, pr.ctx = Library(), None
    pr.mesh = SimpleNamespace(nnodes=2, dim=2)
    pr.sparsity = cg.Sparsity(FINDRM, np.ones(entries, np.int32), np.ones(2, np.int32))
    return pr


@pytest.mark.parametrize("entries", [5, 9])
def test_what_is_not_written_is_zero(garbage, entries):
    pr, tail = _problem(entries), [0.0] * (entries - 5)
    A, rhs, inactive = pr.matrix()
    assert list(A) == [1.0] * 5 + tail and list(rhs) == [2.0] * 2 and list(inactive) == [0, 1]
    pm = cg.PressureMesh(None, 3, 2, None, FINDRM, np.ones(entries, np.int32))
    ct, ml = cg.construct_momentum_ct(pr, pm)
    assert list(ct.ravel()) == [3.0] * 10 + 2 * tail and list(ml) == [4.0] * 2
    cmc = cg.assemble_masslumped_cmc(pr, FINDRM, np.ones(entries, np.int32))
    assert list(cmc) == [5.0] * 5 + tail


def test_short_column_arrays_are_refused():
    pr = _problem(4)
    pm = cg.PressureMesh(None, 3, 2, None, FINDRM, np.ones(4, np.int32))
    for call in (pr.matrix, lambda: cg.construct_momentum_ct(pr, pm),
                 lambda: cg.assemble_masslumped_cmc(pr, FINDRM, np.ones(4, np.int32))):
        with pytest.raises(ValueError, match="5 entries"):
            call()
