"""The exact-order 64 x 64 matrix-core tile at the edges of its 4-wide loads:
reduction lengths and columns of every residue, rows past a segment -- against
the vector-unit tile (MXM_SIMT_MFMA=0) and the CPU restatement bit for bit."""
import numpy as np
import pytest

from tests.moe_testutil import random_case, run_gpu, run_oracle, same_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,D,E,K,F,etype", [
    (130, 16, 2, 2, 64, 0), (70, 65, 3, 2, 67, 0), (97, 31, 2, 1, 129, 2), (64, 15, 1, 1, 63, 1),
    (200, 130, 5, 3, 1, 0), (65, 1, 2, 1, 18, 2), (300, 48, 4, 4, 190, 1)])
def test_simt_tile_edges(gpu_lib, monkeypatch, N, D, E, K, F, etype):
    monkeypatch.setenv("MXM_SIMT_TILE", "64")
    x, wr, experts = random_case(N + D + F, N, D, E, F, expert_type=etype, wscale=0.1)
    # what a tile reads past a segment or a row must not reach its outputs
    x[-1] = np.nan
    act = 1 if etype else 0
    got = []
    for mf in ("1", "0"):
        monkeypatch.setenv("MXM_SIMT_MFMA", mf)
        got.append(run_gpu(x, wr, experts, B=1, T=N, K=K, expert_type=etype, activation=act)[0])
    assert same_bits(got[0][:-1], got[1][:-1]) and np.isnan(got[0][-1]).all()
    x[-1] = 0.0
    delta = run_gpu(x, wr, experts, B=1, T=N, K=K, expert_type=etype, activation=act)[0]
    want = run_oracle(x, wr, experts, K=K, expert_type=etype, activation=act)
    assert same_bits(delta, want["delta"])
    assert same_bits(delta[:-1], got[0][:-1])


@pytest.mark.parametrize("N,D,E,K,F,etype", [
    (9100, 380, 4, 3, 382, 0), (9100, 383, 3, 3, 321, 2), (7000, 257, 5, 4, 640, 1)])
def test_simt_wide_tile(gpu_lib, monkeypatch, N, D, E, K, F, etype):
    """The 128-column tile (large grids): column and reduction remainders, rows
    past a segment, against the vector-unit tile bit for bit."""
    x, wr, experts = random_case(N + D + F, N, D, E, F, expert_type=etype, wscale=0.1)
    x[-1] = np.nan
    got = []
    for mf in ("1", "0"):
        monkeypatch.setenv("MXM_SIMT_MFMA", mf)
        got.append(run_gpu(x, wr, experts, B=1, T=N, K=K, expert_type=etype,
                           activation=1 if etype else 0)[0])
    assert np.isfinite(got[0][:-1]).all() and np.isnan(got[0][-1]).all()
    assert same_bits(got[0][:-1], got[1][:-1])
