"""The combine of narrow rows (one or two waves per token, K up to 64 picks
sorted by lane permutes) at the edges of its spans: the exact-order op bit for
bit against the CPU restatement, whose expert outputs meet in ascending expert
order; a bf16 op's rows of 512, 520, 1024 and 1032 against it too."""
import numpy as np
import pytest

from mixlab_amd.workloads import round_bf16
from tests.moe_testutil import random_case, rel_l2, run_gpu, run_oracle, same_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,E,K", [(4, 3, 3), (252, 70, 64), (256, 70, 65), (260, 20, 9),
                                   (512, 9, 8), (516, 4, 1), (6, 5, 2)])
def test_combine_fp32(gpu_lib, D, E, K):
    N, F = 131, 8
    x, wr, experts = random_case(D + K, N, D, E, F, wscale=0.2)
    delta, *_ = run_gpu(x, wr, experts, B=1, T=N, K=K)
    assert same_bits(delta, run_oracle(x, wr, experts, K=K)["delta"])


@pytest.mark.parametrize("D", [512, 520, 1024, 1032])
def test_combine_bf16(gpu_lib, D):
    N, E, K, F = 1203, 4, 3, 128
    x, wr, experts = random_case(D, N, D, E, F)
    x, wr = round_bf16(x), round_bf16(wr)
    experts = [[round_bf16(w) for w in ws] for ws in experts]
    delta, *_ = run_gpu(x, wr, experts, B=1, T=N, K=K, bf16=True)
    rows = np.arange(0, N, 17, dtype=np.int32)
    want = run_oracle(x, wr, experts, K=K, bf16=True, rows=rows)
    assert rel_l2(delta[rows], want["delta"][rows]) <= 2e-2  # the bar of the bf16 flow
