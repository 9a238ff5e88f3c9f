"""The fp32 backward (products over pairs of bf16 planes) after a kept forward:
bf16 ops whose width is no multiple of 128 or below the MFMA tiles, and fp32
ops -- bit for bit the backward that runs its own forward, and against the
float64 restatement."""
import numpy as np
import pytest

from mixlab_amd import _lib
from mixlab_amd.workloads import bf16_bits, round_bf16
from oracle.backward import backward64
from tests.moe_testutil import random_case, rel_l2

pytestmark = pytest.mark.gpu

# widths with rows of whole 16-byte pieces and without (D 201, F 333), one to
# three column tiles, a split hidden (geglu), a plain mlp, fp32 rows
CASES = [(300, 200, 4, 2, 136, 0, 0, "bf16"), (257, 201, 3, 2, 333, 1, 1, "bf16"),
         (140, 64, 4, 2, 96, 0, 0, "bf16"), (200, 320, 2, 1, 130, 2, 2, "bf16"),
         (260, 136, 4, 2, 100, 1, 1, "fp32"), (130, 65, 3, 3, 333, 2, 3, "fp32")]


@pytest.mark.parametrize("N,D,E,K,F,etype,act,dtype", CASES)
def test_kept_planes(gpu_lib, N, D, E, K, F, etype, act, dtype):
    from mixlab_amd.op import MoEFeedForward

    bf16 = dtype == "bf16"
    x, wr, experts = random_case(N + D + F, N, D, E, F, expert_type=etype, wscale=0.1)
    if bf16:
        x, wr = round_bf16(x), round_bf16(wr)
        experts = [[round_bf16(w) for w in ws] for ws in experts]
    dD = np.random.default_rng(4).standard_normal((N, D), dtype=np.float32)
    lib = _lib.init()
    up = bf16_bits if bf16 else (lambda a: np.ascontiguousarray(a, np.float32))
    code = _lib.MXM_DTYPE_BF16 if bf16 else _lib.MXM_DTYPE_F32
    xdev, ddev = _lib.DeviceBuffer.from_array(up(x)), _lib.DeviceBuffer.from_array(dD)
    wpe = 2 if etype == 2 else 3
    sizes = (N * D, D * E, E * wpe * D * F)
    got = []
    for flags in (0, _lib.MXM_FLAG_KEEP_FOR_BACKWARD):
        with MoEFeedForward([1, N, D, E, K, etype, F, act], [0.5], compute_dtype=dtype,
                            flags=flags) as op:
            op.set_weights(up(wr), [[up(w) for w in ws] for ws in experts])
            bufs = [_lib.DeviceBuffer(4 * n) for n in sizes]
            ptrs = [b.value for b in bufs]
            delta = _lib.DeviceBuffer(4 * N * D)
            for _ in range(2):
                op.forward(xdev.value, code, N, delta.value)
                if flags:
                    rc = lib.mxm_moe_backward_kept(op.handle, ddev.value, 0.3, -0.2, *ptrs)
                else:
                    rc = lib.mxm_moe_backward(op.handle, xdev.value, code, N, ddev.value, 0.3,
                                              -0.2, *ptrs)
                _lib.check(rc, "backward")
            op.synchronize()
            got.append([b.download(np.float32, (n,)) for b, n in zip(bufs, sizes)])
            top = op.routing()["top_idx"]
    for a, b in zip(*got):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
    dx, dwr, dexp = backward64(x, wr, experts, top, dD, 0.3, -0.2, etype, act, 0.5)
    want = (dx.ravel(), dwr.ravel(), np.concatenate([w.ravel() for ws in dexp for w in ws]))
    # the gate gradients read the forward's bf16 expert outputs and the
    # probabilities are bf16 under bf16 compute (2^-9); fp32: three plane pairs
    # of 2^-16 each over sums of up to D or F terms
    for a, w in zip(got[0], want):
        assert rel_l2(a, w) <= (2e-2 if bf16 else 1e-4)
