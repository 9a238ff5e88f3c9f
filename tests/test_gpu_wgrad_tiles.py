"""Weight gradients on 256 x 256 tiles that reach past the output's rows or
columns (widths of 128 modulo 256), on the bf16 backward and on the plane
pairs of the fp32 one, against the float64 restatement."""
import numpy as np
import pytest

from mixlab_amd.op import MoEFeedForward
from mixlab_amd.workloads import bf16_bits, round_bf16
from oracle.backward import backward64
from tests.moe_testutil import random_case, rel_l2

pytestmark = pytest.mark.gpu


# D 384 and 640 (rows past the output), plain mlp of ffn 640 (columns past
# it), a padded ffn, a split hidden, plane pairs at D 600, and D 128 (kept on
# 128 x 128 tiles)
@pytest.mark.parametrize("N,D,E,K,F,etype,act,dtype", [
    (200, 384, 2, 1, 256, 0, 0, "bf16"), (150, 640, 3, 1, 640, 2, 0, "bf16"),
    (130, 640, 2, 1, 333, 1, 1, "bf16"), (140, 600, 2, 1, 380, 0, 0, "fp32"),
    (150, 128, 2, 2, 640, 2, 2, "bf16")])
def test_wgrad_past_the_edge(gpu_lib, N, D, E, K, F, etype, act, dtype):
    bf16 = dtype == "bf16"
    x, wr, experts = random_case(N + D, N, D, E, F, expert_type=etype, wscale=0.1)
    if bf16:
        x, wr = round_bf16(x), round_bf16(wr)
        experts = [[round_bf16(w) for w in ws] for ws in experts]
    dD = np.random.default_rng(6).standard_normal((N, D), dtype=np.float32)
    up = bf16_bits if bf16 else (lambda a: np.ascontiguousarray(a, np.float32))
    with MoEFeedForward([1, N, D, E, K, etype, F, act], [0.0], compute_dtype=dtype) as op:
        op.set_weights(up(wr), [[up(w) for w in ws] for ws in experts])
        dx, dwr, dw = op.backward_host(x, dD, 0.1, 0.2)
        top = op.routing()["top_idx"]
    wx, wwr, ww = backward64(x, wr, experts, top, dD, 0.1, 0.2, etype, act, 0.0)
    # bf16 intermediates (2^-9 each over a few products); three plane pairs of
    # 2^-16 for fp32
    tol = 2e-2 if bf16 else 1e-4
    assert rel_l2(dx, wx) <= tol
    for e in range(E):
        for a, b in zip(dw[e], ww[e]):
            assert np.isfinite(a).all() and rel_l2(a, b) <= tol
