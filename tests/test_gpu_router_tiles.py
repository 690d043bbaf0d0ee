"""The many-token router (8 x 8 tiles, from 25 tokens up to 5120 wide, and wider from 8192 sums) gives the bits of the
few-token one on every (expert, token): the same rows in calls of up to 16 tokens. Expert and token counts that leave partial tiles, one expert, widths below one
thread pass, just past one and with a short last pass, and the scores and selection values of a biased router."""

import ctypes as C

import numpy as np
import pytest

from oracle.formats import bf16_bits
from vesper_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("experts,hidden,tokens", [(1, 4, 25), (13, 516, 31), (8, 1024, 32), (100, 1028, 41),
                                                   (256, 7168, 27), (384, 5120, 129), (1024, 8192, 26)])
def test_tiles_equal_the_few_token_router(gpu_ctx, experts, hidden, tokens):
    rng = np.random.default_rng(experts + hidden + tokens)
    w = gpu_ctx.upload((rng.standard_normal((experts, hidden)) * 0.05).astype(np.float32))
    bias = gpu_ctx.upload(rng.standard_normal(experts).astype(np.float32))
    bits = bf16_bits(rng.standard_normal((tokens, hidden)).astype(np.float32))
    k = min(4, experts)

    def route(rows):
        t = rows.shape[0]
        x = gpu_ctx.upload(rows)
        shapes = {"logits": ((t, experts), np.float32), "scores": ((t, experts), np.float32),
                  "selection": ((t, experts), np.float32), "indices": ((t, k), np.int32), "weights": ((t, k), np.float32)}
        d = {n: gpu_ctx.empty(s, dt) for n, (s, dt) in shapes.items()}
        out = _lib.MxRouterOut(*[d[n].ptr for n in shapes], None, None, None)
        gpu_ctx.lib.router(gpu_ctx._h(), _lib.vp(w), _lib.vp(bias), _lib.vp(x), t, hidden, experts, k,
                           _lib.MX_SCORE["sigmoid"], 2.5, C.byref(out), None)
        got = {n: a.download() for n, a in d.items()}
        for a in [x, *d.values()]:
            a.free()
        return got

    whole = route(bits)
    parts = [route(bits[i:i + 16]) for i in range(0, tokens, 16)]
    for name, got in whole.items():
        np.testing.assert_array_equal(got.view(np.uint32), np.concatenate([p[name] for p in parts]).view(np.uint32),
                                      err_msg=name)
    w.free()
    bias.free()
