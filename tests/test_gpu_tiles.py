"""The MFMA grouped GEMM's tile plan (256 x 256 and 128 x 128 tiles of one
launch, pairs of 128 x 128 tiles) at the edges of its tiles: the op without a
family flag against the 128 x 128 family, bit for bit (every output is one sum
over k in ascending order whichever tile it falls in), and against the CPU
restatement on a sample of rows."""
import ctypes

import numpy as np
import pytest

from mixlab_amd import _lib
from mixlab_amd.workloads import round_bf16
from tests.moe_testutil import assert_routing_equal, random_case, rel_l2, run_gpu, run_oracle, same_bits

pytestmark = pytest.mark.gpu

# K = E gives every expert all N rows: remainders of 1, 127, 128, 129, 255 and
# 0 rows past multiples of 256; widths with and without a last 128 columns.  The
# reductions of up to 384 run on the 128 x 128 kernel with and without the flag
# (its own edges, 200 and 70 experts on its LDS prefixes and 98 row tiles in whole
# groups per XCD among them), the longer ones on a plan of quarter tiles.
CASES = [
    (257, 128, 2, 2, 128, 0), (383, 256, 3, 3, 128, 0), (384, 384, 2, 2, 256, 0),
    (385, 192, 2, 2, 320, 1), (511, 640, 2, 2, 384, 2), (512, 128, 1, 1, 640, 0),
    (2600, 256, 2, 2, 2048, 0), (3300, 128, 3, 3, 2560, 0), (4100, 320, 2, 2, 896, 1),
    (1300, 256, 200, 8, 128, 0), (1500, 256, 70, 1, 256, 0), (6200, 128, 2, 2, 256, 0),
]


def plan(counts, ncols, cus):
    """The scheduled kernel's plan: big tiles run, big tiles cut in four, small
    row tiles, tiles that a workgroup runs at most, workgroups of an eighth of the
    device with one big tile more than the others, and whether a round is cut."""
    counts = np.asarray(counts, np.int64)
    big = (counts + 127) // 256
    small = int((counts > big * 256).sum())
    ncb, ncs = ncols // 256, ncols // 128
    grid = min(cus, (int(counts.sum() // 128 + min(len(counts), counts.sum())) * ncs + 7) // 8 * 8)
    B = int(big.sum()) * ncb
    S0 = small * ncs + (ncs & 1) * 2 * int(big.sum())
    rem, run = B % grid, B
    if rem > 0:
        cut = -(-(4 * rem + S0) // grid)
        keep = 3 + -(-max(0, S0 - (grid - rem) * 3) // grid)
        if cut < keep:
            run = B - rem
    return dict(run=run, cut=B - run, small=small, deep=-(-run // grid), odd=(run // 8) % (grid // 8),
                partial=bool((counts[big > 0] % 256 != 0).any()))


# Up projections of more than 384 (D) on the scheduled kernel, by what their
# plan holds: big tiles run and the last round's cut; that round kept, with
# workgroups of one big tile more than the rest and small tiles handed to the
# rest first; several big tiles per workgroup; the last 128 columns of an odd
# number; big tiles of 129 and of 228 rows, remainders of 1 and 127; 70 and 200
# experts (prefixes over several waves, some experts empty); 108 row tiles, of
# which the XCDs take two whole groups of 6 each in turn, then eighths of the rest.
PLAN_CASES = [
    (2600, 512, 2, 2, 2048, 0, dict(run=256, cut=64, small=2)),
    (2600, 512, 2, 2, 1024, 0, dict(run=160, cut=0, small=2, odd=20)),
    (3300, 448, 3, 3, 2560, 0, dict(run=768, cut=12, deep=3, partial=True)),
    (3300, 448, 3, 3, 3200, 2, dict(run=468, cut=0, deep=2, partial=True)),
    (385, 448, 2, 2, 5120, 0, dict(run=160, cut=0, small=0, partial=True)),
    (257, 448, 3, 3, 5632, 0, dict(run=132, cut=0, small=3)),
    (383, 500, 3, 3, 5632, 1, dict(run=132, cut=0, small=3)),
    (9000, 448, 3, 3, 512, 0, dict(run=420, cut=0, small=3, deep=2, odd=20)),
    (9001, 500, 3, 3, 384, 0, dict(run=256, cut=59, small=3)),
    (6000, 512, 70, 1, 512, 0, dict(cut=0, deep=1)),
    (1500, 512, 200, 8, 512, 0, dict(run=0, cut=0, small=200)),
]


@pytest.mark.parametrize("N,D,E,K,F,etype,want_plan", PLAN_CASES,
                         ids=["-".join(map(str, c[:6])) for c in PLAN_CASES])
def test_tile_plan_mixed(gpu_lib, N, D, E, K, F, etype, want_plan):
    family = gpu_lib._Z15mxm_mfma_familyiiiii  # the launcher's choice
    family.restype, family.argtypes = ctypes.c_int, [ctypes.c_int] * 5
    ncols, kd = (1 if etype == 2 else 2) * F, -(-D // 64) * 64
    assert family(N * K, E, ncols, kd, 0) == 0, "not on the scheduled kernel"
    routing = run_case(N, D, E, K, F, etype)
    p = plan(routing["counts"], ncols, 256)
    assert {k: p[k] for k in want_plan} == want_plan, p
    if E == 70:
        assert p["run"] > 64 and (np.asarray(routing["counts"]) == 0).any()


@pytest.mark.parametrize("N,D,E,K,F,etype", CASES)
def test_tile_plan_edges(gpu_lib, N, D, E, K, F, etype):
    run_case(N, D, E, K, F, etype)


def run_case(N, D, E, K, F, etype):
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
    return routing
