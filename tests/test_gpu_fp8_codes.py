"""The codes and scales that a decode-size FP8 projection writes on request, at the token counts where they come from the
GEMV's own quantizer (5 to 32) and from the row quantizer (up to 4): the oracle's bytes, zero blocks and a wide range of scales included,
each output asked for alone and both, and the product the same as without them."""

import ctypes as C

import numpy as np
import pytest

from oracle.formats import bf16_bits, bf16_values
from oracle.projections import fp8_projection, fp8_weights
from tests.test_gpu_row_gemv import projections
from vesper_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("block", [32, 128])
@pytest.mark.parametrize("tokens", [1, 4, 5, 16, 17, 32])
@pytest.mark.parametrize("rows,width", [(64, 128), (192, 1152)])
def test_requested_codes(gpu_ctx, block, tokens, rows, width):
    rng = np.random.default_rng(block + tokens + width)
    w, sw = fp8_weights(rng, rows, width, block)
    x = rng.standard_normal((tokens, width)).astype(np.float32) * np.exp2(rng.integers(-30, 30, (tokens, 1)))
    x[0, :32], x[-1, -128:] = 0.0, 0.0
    x[tokens // 2, 3] = 1e20
    bits = bf16_bits(x.astype(np.float32))
    ref = fp8_projection(bf16_values(bits), w, sw, block)
    ctx = gpu_ctx
    xd = ctx.upload(bits)
    q, y = ctx.empty((tokens, width), np.uint8), ctx.empty((tokens, rows), np.uint16)
    s = ctx.empty(*(((tokens, width // 32), np.uint8) if block == 32 else ((tokens, width // 128), np.float32)))
    ys = []
    with projections(w, sw, block) as proj:
        for want_q, want_s in ((0, 0), (1, 0), (0, 1), (1, 1)):
            q.upload(np.full(q.shape, 0xEE, np.uint8))
            s.upload(np.full(s.shape, 7, s.dtype))
            ctx.lib.fp8_projection(ctx._h(), C.c_void_p(proj.tiled["p"]), rows, width, block, _lib.vp(xd), tokens,
                                   _lib.vp(y), None, _lib.vp(q) if want_q else None, _lib.vp(s) if want_s else None, None)
            ys.append(y.download())
            np.testing.assert_array_equal(q.download(), ref["input_fp8"] if want_q else np.full(q.shape, 0xEE, np.uint8))
            np.testing.assert_array_equal(s.download(), ref["scale"] if want_s else np.full(s.shape, 7, s.dtype))
    for other in ys[1:]:
        np.testing.assert_array_equal(other, ys[0])
    for a in (xd, q, y, s):
        a.free()
