"""The tiled router's matrix-core logits for up to 32 experts, its tiles of 16
and 64 tokens, and the one-launch dispatch: against the vector-unit logits
(MXM_ROUTER_MFMA=0) bit for bit, and the routing bit for bit against the CPU
restatement."""
import numpy as np
import pytest

from mixlab_amd.workloads import round_bf16
from tests.moe_testutil import assert_routing_equal, random_case, run_gpu, run_oracle, same_bits

pytestmark = pytest.mark.gpu

# one to four expert groups of 16, chunks that do not fill a round (D 64, 72,
# 320, 1000), last tiles of 1 and 15 tokens, tiles of 64 from 16385 tokens on
CASES = [
    (1025, 64, 4, 2, "fp32"), (1039, 72, 16, 3, "fp32"), (1100, 1000, 17, 2, "fp32"),
    (2000, 320, 32, 8, "bf16"), (1031, 200, 8, 2, "bf16"), (1500, 2048, 5, 5, "bf16"),
    (1300, 128, 1, 1, "bf16"), (16384, 64, 20, 2, "bf16"), (16385, 72, 12, 2, "bf16"),
    (16449, 136, 30, 4, "fp32"), (17000, 64, 4, 1, "fp32"),
]


@pytest.mark.parametrize("N,D,E,K,dtype", CASES)
def test_router_tiles(gpu_lib, monkeypatch, N, D, E, K, dtype):
    bf16 = dtype == "bf16"
    F = 128 if bf16 else 32
    x, wr, experts = random_case(50 + N + D + E, N, D, E, F)
    if bf16:
        x, wr = round_bf16(x), round_bf16(wr)
        experts = [[round_bf16(w) for w in ws] for ws in experts]
    runs = []
    for mf in ("1", "0"):
        monkeypatch.setenv("MXM_ROUTER_MFMA", mf)
        runs.append(run_gpu(x, wr, experts, B=1, T=N, K=K, bf16=bf16, want_probs=True))
    (d1, a1, e1, r1, _), (d0, a0, e0, r0, _) = runs
    for key in ("probs", "top_idx", "gates", "counts", "offsets", "perm"):
        assert same_bits(r1[key], r0[key]), key
    assert same_bits(d1, d0)
    assert same_bits(np.float32(a1), np.float32(a0)) and same_bits(np.float32(e1), np.float32(e0))
    rows = np.arange(0, N, max(1, N // 64), dtype=np.int32)
    want = run_oracle(x, wr, experts, K=K, bf16=bf16, rows=rows)
    assert same_bits(r1["probs"], want["probs"])
    assert_routing_equal(r1, want)
    # fp32 sums of N probabilities (bf16: the means rounded to bf16, 2^-9)
    assert abs(a1 - want["aux"]) <= (1e-2 if bf16 else 1e-5) * abs(want["aux"])
    assert abs(e1 - want["entropy"]) <= 1e-4 * abs(want["entropy"]) + 1e-7


def test_dispatch_of_many_tiles(gpu_lib):
    """More than 2^18 histogram entries (1101 tiles of 256 experts): the
    dispatch reads sums over groups of 32 tiles."""
    N, D, E, K, F = 70407, 8, 256, 2, 8
    x, wr, experts = random_case(9, N, D, E, F)
    wr = wr * np.float32(20.0)
    _, aux, ent, routing, _ = run_gpu(x, wr, experts, B=1, T=N, K=K)
    want = run_oracle(x, wr, experts, K=K, rows=np.arange(4, dtype=np.int32))
    assert_routing_equal(routing, want)
    assert abs(aux - want["aux"]) <= 1e-5 * abs(want["aux"])
    assert abs(ent - want["entropy"]) <= 1e-4 * abs(want["entropy"])


@pytest.mark.parametrize("N,D,dtype,tile", [
    (1100, 127, "fp32", 64), (1100, 128, "fp32", 16), (1500, 130, "bf16", 16),
    (1500, 65, "bf16", 64), (16385, 128, "fp32", 64)])
def test_tile_tokens(gpu_lib, N, D, dtype, tile):
    """Tiles of 16 tokens only for rows that the matrix cores take (whole 16-byte
    pieces of x, or of its padded copy for the matrix-core experts)."""
    bf16 = dtype == "bf16"
    E, K, F = 6, 2, 16 if D == 65 else 128
    x, wr, experts = random_case(N + D, N, D, E, F)
    if bf16:
        x, wr = round_bf16(x), round_bf16(wr)
        experts = [[round_bf16(w) for w in ws] for ws in experts]
    _, aux, ent, routing, info = run_gpu(x, wr, experts, B=1, T=N, K=K, bf16=bf16)
    assert info["route_flow"] == 0 and info["router_tiles"] == -(-N // tile)
    want = run_oracle(x, wr, experts, K=K, bf16=bf16, rows=np.arange(4, dtype=np.int32))
    assert_routing_equal(routing, want)
    # fp32 sums of N probabilities (bf16: the means rounded to bf16, 2^-9)
    assert abs(aux - want["aux"]) <= (1e-2 if bf16 else 1e-5) * abs(want["aux"])
    assert abs(ent - want["entropy"]) <= 1e-4 * abs(want["entropy"])


@pytest.mark.parametrize("N,E", [(6144, 256), (6145, 256), (16384, 100), (16383, 97)])
def test_dispatch_groups_of_small_tiles(gpu_lib, N, E):
    """Both sides of the line from which the dispatch reads sums over groups of
    tiles, with tiles of 16 tokens and a last group of one or of all its tiles."""
    D, K, F = 8, 3, 8
    x, wr, experts = random_case(N + E, N, D, E, F)
    wr = wr * np.float32(20.0)
    _, aux, ent, routing, info = run_gpu(x, wr, experts, B=1, T=N, K=K)
    assert info["router_tiles"] == -(-N // 16)
    want = run_oracle(x, wr, experts, K=K, rows=np.arange(4, dtype=np.int32))
    assert_routing_equal(routing, want)
    assert abs(aux - want["aux"]) <= 1e-5 * abs(want["aux"])  # fp32 sums of N terms
    assert abs(ent - want["entropy"]) <= 1e-4 * abs(want["entropy"])
