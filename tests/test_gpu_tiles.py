"""The MFMA grouped GEMM's tile plan (256 x 256 and 128 x 128 tiles of one
launch, pairs of 128 x 128 tiles) at the edges of its tiles: the op without a
family flag against the 128 x 128 family, bit for bit (every output is one sum
over k in ascending order whichever tile it falls in), and against the CPU
restatement on a sample of rows."""
import numpy as np
import pytest

from mixlab_amd import _lib
from mixlab_amd.workloads import round_bf16
from tests.moe_testutil import assert_routing_equal, random_case, rel_l2, run_gpu, run_oracle, same_bits

pytestmark = pytest.mark.gpu

# K = E gives every expert all N rows: remainders of 1, 127, 128, 129, 255 and
# 0 rows past multiples of 256; widths with and without a last 128 columns.
# 2600 rows by 16 column tiles are 320 big tiles on 256 CUs, the last 64 cut;
# 3300 by 20 are 780, the last round kept whole.  200 and 70 experts: the
# plan's prefixes over several waves, some experts empty.
CASES = [
    (257, 128, 2, 2, 128, 0), (383, 256, 3, 3, 128, 0), (384, 384, 2, 2, 256, 0),
    (385, 192, 2, 2, 320, 1), (511, 640, 2, 2, 384, 2), (512, 128, 1, 1, 640, 0),
    (2600, 256, 2, 2, 2048, 0), (3300, 128, 3, 3, 2560, 0), (4100, 320, 2, 2, 896, 1),
    (1300, 256, 200, 8, 128, 0), (1500, 256, 70, 1, 256, 0),
]


@pytest.mark.parametrize("N,D,E,K,F,etype", CASES)
def test_tile_plan_edges(gpu_lib, N, D, E, K, F, etype):
    act = 1 if etype else 0
    x, wr, experts = random_case(N + D + F, N, D, E, F, expert_type=etype)
    if E == 70:
        wr[:, 41:] = wr[:, 40:41]  # equal logits: a token picks 40 before any of these
    x, wr = round_bf16(x), round_bf16(wr)
    experts = [[round_bf16(m) for m in ws] for ws in experts]
    kw = dict(B=1, T=N, K=K, expert_type=etype, activation=act, bf16=True)
    delta, aux, ent, routing, info = run_gpu(x, wr, experts, **kw)
    ref = run_gpu(x, wr, experts, flags=_lib.MXM_FLAG_MFMA_TILE128, **kw)
    assert info["mfma"] and not info["bf16_stream"]
    assert_routing_equal(routing, ref[3])
    assert same_bits(delta, ref[0])
    assert (aux, ent) == (ref[1], ref[2])
    rows = np.sort(np.random.default_rng(3).choice(N, size=min(N, 96), replace=False)).astype(np.int32)
    want = run_oracle(x, wr, experts, K=K, expert_type=etype, activation=act, bf16=True, rows=rows)
    # the bf16 flow's roundings (the repository's bar for every bf16 product)
    assert rel_l2(delta[rows], want["delta"][rows]) <= 2e-2
