"""FP8 calls whose outputs share bytes with their input, at the token counts where the GEMV can quantize that input
itself: the output has the bits of the call with separate buffers, as the input is read before anything is written.
Projections in place and shifted, the FP32 sums over the input, and the expert's stages over its input and output."""

import ctypes as C

import numpy as np
import pytest

from oracle.formats import bf16_bits
from oracle.inputs import activations, fp8_block32_expert_normal
from oracle.projections import fp8_weights
from tests.test_gpu_row_gemv import projections
from vesper_amd import _lib
from vesper_amd.shared import ResidentSharedExpert

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("block", [32, 128])
@pytest.mark.parametrize("size,tokens", [(1024, 1), (1024, 2), (512, 4), (5120, 1)])
def test_projection_over_its_input(gpu_ctx, block, size, tokens):
    rng = np.random.default_rng(block + size + tokens)
    w, sw = fp8_weights(rng, size, size, block)
    bits = bf16_bits(rng.standard_normal((tokens, size)).astype(np.float32))
    nbytes = tokens * size * 2
    with projections(w, sw, block) as proj:
        lib, ctx, tiled = gpu_ctx.lib, gpu_ctx, C.c_void_p(proj.tiled["p"])
        buf = ctx.malloc(6 * nbytes)

        def call(x, y, trace=None):
            ctx.copy_h2d(buf + x, bits)
            lib.fp8_projection(ctx._h(), tiled, size, size, block, C.c_void_p(buf + x), tokens, C.c_void_p(buf + y),
                               None if trace is None else C.c_void_p(buf + trace), None, None, None)
            ctx.sync()
            return ctx.download(buf + y, (tokens, size), np.uint16)

        want = call(0, nbytes)
        for x, y, trace in ((0, 0, None), (0, nbytes // 2, None), (nbytes, nbytes - 256, None), (0, 2 * nbytes, 0),
                            (nbytes, 4 * nbytes, 0)):
            np.testing.assert_array_equal(call(x, y, trace), want, err_msg=f"x at {x}, y at {y}, trace at {trace}")
        ctx.free(buf)


@pytest.mark.parametrize("tokens", [1, 2, 4])
def test_expert_stages_over_input_and_output(tokens):
    size = 512   # hidden = intermediate: a stage buffer can be x or y
    rng = np.random.default_rng(tokens)
    arrays = fp8_block32_expert_normal(rng, size, size)
    x = activations(rng, tokens, size)
    with ResidentSharedExpert(arrays, swiglu_limit=10.0, hidden=size, intermediate=size) as shared:
        want = shared.forward(x)
        ctx = shared.ctx
        xd, yd = ctx.upload(bf16_bits(x)), ctx.empty((tokens, size), np.uint16)
        trace = ctx.malloc(tokens * size * 20)
        w = [C.c_void_p(shared.tiled[p]) for p in ("w1", "w3", "w2")]

        def call(x_at, y_at, **stages):
            ctx.copy_h2d(x_at, bf16_bits(x))
            names = ("q", "s", "w1", "w3", "down_input", "trace", "down_q", "down_s")
            st = _lib.MxExpertStages(*[stages.get(n) for n in names])
            ctx.lib.fp8_expert_forward(ctx._h(), *w, size, size, C.c_void_p(x_at), tokens, 10.0, None, C.c_void_p(y_at),
                                       C.byref(st), None)
            ctx.sync()
            return ctx.download(y_at, (tokens, size), np.uint16)

        xp, yp = xd.ptr, yd.ptr
        spare = ctx.malloc(tokens * size * 2)
        for what, got in (("y over x", call(xp, xp)), ("down input in y", call(xp, yp, down_input=yp)),
                          ("down input over x", call(xp, yp, down_input=xp)), ("W1 over x", call(xp, yp, w1=xp)),
                          ("W3 over x", call(xp, yp, w3=xp)), ("trace over x", call(trace + 256, yp, trace=trace)),
                          ("W1 and down input in one buffer", call(xp, yp, w1=spare, down_input=spare))):
            np.testing.assert_array_equal(got, want["w2"], err_msg=what)
        for p in (trace, spare):
            ctx.free(p)
        xd.free()
        yd.free()
