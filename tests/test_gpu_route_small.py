"""The one-launch router with four tokens per workgroup: batches around the line
where it starts and of every remainder of four, every number of expert groups,
widths past whole chunks -- routing bit for bit against the CPU restatement, over
calls of one op on x of their own (the ticket is left zero for the next call, and
no result of the call before stands in for this one's)."""
import numpy as np
import pytest

from mixlab_amd.op import MoEFeedForward
from mixlab_amd.workloads import bf16_bits, round_bf16
from tests.moe_testutil import assert_routing_equal, random_case, run_oracle, same_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,D,E,K,bf16", [
    (256, 128, 8, 2, True), (257, 128, 8, 2, True), (258, 136, 70, 3, True), (259, 200, 130, 2, True),
    (511, 1024, 200, 4, True), (767, 65, 5, 5, False), (1022, 72, 64, 8, False),
    (640, 3072, 16, 2, True), (640, 3080, 16, 2, True), (301, 3, 256, 1, False)])
def test_route_small_four_tokens(gpu_lib, monkeypatch, N, D, E, K, bf16):
    monkeypatch.setenv("MXM_SMALL_ROUTE", "1")
    F = 16
    x, wr, experts = random_case(N + D + E, N, D, E, F)
    if bf16:
        x, wr = round_bf16(x), round_bf16(wr)
        experts = [[round_bf16(m) for m in ws] for ws in experts]
    conv = bf16_bits if bf16 else (lambda a: np.ascontiguousarray(a, np.float32))
    with MoEFeedForward([1, N, D, E, K, 0, F, 0], [0.0],
                        compute_dtype="bf16" if bf16 else "fp32") as op:
        op.set_weights(conv(wr), [[conv(w) for w in ws] for ws in experts])
        for call in range(3):
            xc = np.roll(x, 5 * call, axis=0) * np.float32((-1) ** call)
            want = run_oracle(xc, wr, experts, K=K, bf16=bf16)
            delta, aux, ent = op.forward_host(conv(xc))
            assert op.info()["route_flow"] == 1
            assert_routing_equal(op.routing(), want)
            # (F below the matrix-core tiles: the exact-order products)
            assert same_bits(delta, want["delta"])
            # fp32 sums of N probabilities (bf16: the means rounded to bf16, 2^-9)
            assert abs(aux - want["aux"]) <= (1e-2 if bf16 else 1e-5) * abs(want["aux"])
            assert abs(ent - want["entropy"]) <= 1e-4 * abs(want["entropy"])
