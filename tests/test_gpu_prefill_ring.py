"""The prefill's gate/up ring at its edges: experts of 1 to 129 rows (every count of live 16-row token tiles, from which
the ring's depth follows, a full tile and one row past it, idle experts), over hidden sizes of 2, 4 and 6 chunks (fewer
chunks than the ring has stages among them). Every routed pair's and the shared expert's down-input codes and scales
equal the oracle's, and every token's output is within tolerance."""

import numpy as np
import pytest

from oracle.expert import expert_forward
from oracle.inputs import activations
from oracle.moe import moe_layer_routed
from tests.helpers import assert_close, max_rel_err
from tests.test_gpu_prefill import check_down_codes, small_layer
from vesper_amd.config import MoEConfig

pytestmark = pytest.mark.gpu

ROWS = (1, 16, 17, 33, 0, 64, 65, 96, 100, 113, 128, 129, 0)   # of expert e


@pytest.mark.parametrize("hidden,shared", [(256, True), (512, False), (768, True)])
def test_ring_depths_and_short_rows(gpu_ctx, hidden, shared):
    cfg = MoEConfig(hidden=hidden, intermediate=384, experts=len(ROWS), top_k=1, swiglu_limit=10.0,
                    shared="mxfp4" if shared else None, max_tokens=16)
    rng = np.random.default_rng(hidden)
    layer, bank, _, arrays = small_layer(gpu_ctx, rng, cfg)
    try:
        ids = rng.permutation(np.repeat(np.arange(len(ROWS), dtype=np.int32), ROWS)).reshape(-1, 1)
        tokens = ids.shape[0]
        x = activations(rng, tokens, hidden)
        wts = rng.uniform(0.1, 2.0, (tokens, 1)).astype(np.float32)
        got, stages = layer.prefill(x, ids, wts, stages=True)
        ref = moe_layer_routed(x, ids, wts, {e: arrays[e] for e in range(cfg.experts)},
                               arrays[cfg.experts] if shared else None, num_experts=cfg.experts,
                               swiglu_limit=cfg.swiglu_limit)
        sh = expert_forward(x, arrays[cfg.experts], None, cfg.swiglu_limit) if shared else None
        check_down_codes(stages, ids, ref["experts"], shared=sh, what=f"hidden {hidden}")
        assert_close(got, ref["output_bf16"], "prefill")
        for t in range(tokens):
            assert max_rel_err(got[t], ref["output_bf16"][t]) <= 2e-2, t
    finally:
        layer.close()
        bank.free()
