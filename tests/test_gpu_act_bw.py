"""The activation backward in the epilogue of the bf16 backward's hidden-
gradient product: every kind of hidden, rows and widths at the edges of its
32-row blocks and 64-column parts, against the float64 restatement."""
import numpy as np
import pytest

from mixlab_amd.op import MoEFeedForward
from mixlab_amd.workloads import bf16_bits, round_bf16
from oracle.backward import backward64
from tests.moe_testutil import random_case, rel_l2

pytestmark = pytest.mark.gpu


# (one slot part, a padded width, several tiles of 128 and of 256 columns;
# experts of 0, 1, 31..33 and many rows come from the small and large N)
@pytest.mark.parametrize("etype,act", [(0, 0), (1, 0), (2, 0), (2, 1), (2, 2), (2, 3)])
@pytest.mark.parametrize("N,D,E,K,F", [
    (3, 128, 8, 2, 64), (33, 128, 1, 1, 128), (97, 256, 3, 2, 200), (700, 256, 4, 2, 512)])
def test_hidden_gradient_epilogue(gpu_lib, N, D, E, K, F, etype, act):
    x, wr, experts = random_case(N + F, N, D, E, F, expert_type=etype, wscale=0.1)
    x, wr = round_bf16(x), round_bf16(wr)
    experts = [[round_bf16(w) for w in ws] for ws in experts]
    dD = np.random.default_rng(7).standard_normal((N, D), dtype=np.float32)
    with MoEFeedForward([1, N, D, E, K, etype, F, act], [0.25], compute_dtype="bf16") as op:
        op.set_weights(bf16_bits(wr), [[bf16_bits(w) for w in ws] for ws in experts])
        dx, dwr, dw = op.backward_host(x, dD, 0.1, 0.2)
        top = op.routing()["top_idx"]
    wx, wwr, ww = backward64(x, wr, experts, top, dD, 0.1, 0.2, etype, act, 0.25)
    # bf16 intermediates (2^-9 each over a few products); dwr holds the gate
    # gradients, summed over the width's parts
    tol = 2e-2
    assert rel_l2(dx, wx) <= tol and rel_l2(dwr, wwr) <= tol
    for e in range(E):
        for a, b in zip(dw[e], ww[e]):
            if (np.asarray(top) == e).any():
                assert rel_l2(a, b) <= tol
            else:
                assert not np.any(a)
