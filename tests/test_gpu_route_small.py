"""The one-launch router with four tokens per workgroup: batches around the line
where it starts and of every remainder of four, every number of expert groups,
widths past whole chunks -- routing bit for bit against the CPU restatement, and
repeated calls (the ticket is left zero)."""
import pytest

from mixlab_amd.workloads import round_bf16
from tests.moe_testutil import assert_routing_equal, random_case, run_gpu, run_oracle, same_bits

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
    want = run_oracle(x, wr, experts, K=K, bf16=bf16)
    for _ in range(2):
        delta, aux, ent, routing, info = run_gpu(x, wr, experts, B=1, T=N, K=K, bf16=bf16)
        assert info["route_flow"] == 1
        assert_routing_equal(routing, want)
        # (F below the matrix-core tiles: the exact-order products)
        assert same_bits(delta, want["delta"])
        # fp32 sums of N probabilities (bf16: the means rounded to bf16, 2^-9)
        assert abs(aux - want["aux"]) <= (1e-2 if bf16 else 1e-5) * abs(want["aux"])
        assert abs(ent - want["entropy"]) <= 1e-4 * abs(want["entropy"])
