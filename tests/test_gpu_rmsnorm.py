"""The block's RMSNorm at the edges of its row kernels (4-element rows held in
registers up to 2048, element rows otherwise): the block bit for bit against
the CPU restatement on the exact-order expert kernels."""
import numpy as np
import pytest

import oracle
from mixlab_amd import _lib, moe
from mixlab_amd.workloads import bf16_bits, round_bf16
from tests.moe_testutil import same_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [4, 66, 252, 260, 1028, 2048, 2052])
@pytest.mark.parametrize("flow", ["fp32", "bf16"])
def test_rmsnorm_rows(gpu_lib, flow, D):
    from mixlab_amd.op import MoEBlock

    bf16 = flow == "bf16"
    r = round_bf16 if bf16 else (lambda a: a)
    rng = np.random.default_rng(D)
    spec = moe.BlockSpec.from_json('{"type":"moe","num_experts":2,"top_k":1}')
    with MoEBlock(spec, 1, 5, D, mlp_mult=0.001, compute_dtype=flow,
                  flags=_lib.MXM_FLAG_FORCE_SIMT) as blk:
        ws = [rng.standard_normal(m.shape, dtype=np.float32) * np.float32(0.05) for m in blk.metas]
        ws[0] = 1.0 + ws[0]
        blk.set_weights(ws)
        x = r(rng.standard_normal((5, D), dtype=np.float32))
        out, _, _ = blk.forward_host(bf16_bits(x) if bf16 else x)
        routing = blk.op.routing()
    experts = [[r(w) for w in ws[2 + 3 * e:5 + 3 * e]] for e in range(2)]
    want = oracle.block_forward(x, r(ws[0]), r(ws[1]), experts, top_k=1, eps=blk.eps,
                                aux_weight=blk.aux_weight, bf16=bf16)
    assert same_bits(routing["gates"], want["gates"])
    assert same_bits(out, want["x_out"])
