"""The training gradient where its per-block sums change shape: fewer rows
than one chunk, exactly one, ragged last chunks and edge blocks, and odd
probe counts, against the numpy restatement (BF16 operands emulated).  The
tolerances are those of the small-system gradient test: FP32 against FP64
sums can move an activation across a bfloat16 rounding boundary, one 2^-8
step of one operand, hence 5e-3 of a parameter block's largest entry.
"""
import numpy as np
import pytest

import learned_ref as LR
from test_gpu_learned import perturbed_params, system
from fluidity_amd import learned

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,scale,probes", [("c1", 5, 1), ("c4", 3, 8), ("c4", 4, 3), ("c4", 12, 16),
                                               ("c4", 20, 5)])
def test_gradient_over_block_shapes(require_gpu, name, scale, probes):
    print(f"\n[case] gradient {name} {scale}, {probes} probes", flush=True)
    cfg, pr, g = system(name, scale=scale, seed=9)
    th = perturbed_params()
    learned.set_params(pr, th)
    loss, grad = learned.loss_grad(pr, nprobe=probes, seed=42)
    lref, gref, _ = LR.loss_and_grad(th, g, LR.probes(g.n, probes, 42), rb=True)
    assert abs(loss - lref) <= 1e-4 * abs(lref)
    for lo, hi in [(0, LR.W_IN + LR.H * LR.NFEAT), (LR.B_IN, LR.L0), (LR.layer(0), LR.layer(1)),
                   (LR.layer(1), LR.layer(2)), (LR.layer(2), LR.OUT), (LR.OUT, LR.G1), (LR.G1, LR.TOTAL)]:
        assert np.max(np.abs(grad[lo:hi] - gref[lo:hi])) <= 5e-3 * max(np.max(np.abs(gref[lo:hi])), 1e-30), (lo, hi)
    loss2, grad2 = learned.loss_grad(pr, nprobe=probes, seed=42)
    assert loss2 == loss and np.array_equal(grad, grad2)  # fixed partition and order
    pr.close()
