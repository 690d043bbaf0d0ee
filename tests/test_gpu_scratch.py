"""The first FP8 call of a context may be under stream capture, where nothing can be allocated: the scratch that a
decode-size call needs is there from the context's creation. The captured calls replay to the eager results."""

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

THREAD_LOCAL = 1   # hipStreamCaptureModeThreadLocal


class Graph:
    """What `calls` launches on `stream`, captured."""

    def __init__(self, ctx, stream, calls):
        self.hip, self.stream = ctx.lib.cdll, C.c_void_p(stream)   # the symbols of its HIP runtime
        graph, self.exec = C.c_void_p(), C.c_void_p()
        self.check(self.hip.hipStreamBeginCapture(self.stream, THREAD_LOCAL))
        try:
            calls()
        finally:
            status = self.hip.hipStreamEndCapture(self.stream, C.byref(graph))
        self.check(status)
        self.check(self.hip.hipGraphInstantiate(C.byref(self.exec), graph, None, None, C.c_size_t(0)))
        self.check(self.hip.hipGraphDestroy(graph))

    @staticmethod
    def check(status):
        assert status == 0, f"HIP error {status}"

    def launch(self):
        self.check(self.hip.hipGraphLaunch(self.exec, self.stream))
        self.check(self.hip.hipStreamSynchronize(self.stream))

    def close(self):
        self.check(self.hip.hipGraphExecDestroy(self.exec))


@pytest.mark.parametrize("block,rows,width,tokens", [(32, 64, 16384, 32), (128, 64, 16384, 5), (128, 2112, 1024, 17)])
def test_captured_first_projection(gpu_ctx, block, rows, width, tokens):
    rng = np.random.default_rng(rows + width + tokens)
    w, sw = fp8_weights(rng, rows, width, block)
    bits = bf16_bits(rng.standard_normal((tokens, width)).astype(np.float32))
    with projections(w, sw, block) as proj, _lib.Context(0) as ctx:
        x, y = ctx.upload(bits), ctx.empty((tokens, rows), np.uint16)
        stream = ctx.stream()

        def call(on, at):
            at.lib.fp8_projection(at._h(), C.c_void_p(proj.tiled["p"]), rows, width, block, _lib.vp(x), tokens, _lib.vp(y),
                                  None, None, None, on)

        call(None, gpu_ctx)
        gpu_ctx.sync()
        want = y.download()
        graph = Graph(ctx, stream, lambda: call(C.c_void_p(stream), ctx))
        for _ in range(3):
            y.upload(np.zeros_like(want))
            ctx.sync()
            graph.launch()
            np.testing.assert_array_equal(y.download(), want)
        graph.close()
        x.free()
        y.free()


def test_captured_first_expert(gpu_ctx):
    size, tokens = 512, 16
    rng = np.random.default_rng(3)
    arrays = fp8_block32_expert_normal(rng, size, size)
    bits = bf16_bits(activations(rng, tokens, size))
    with ResidentSharedExpert(arrays, swiglu_limit=10.0, hidden=size, intermediate=size) as shared, _lib.Context(0) as ctx:
        x, y = ctx.upload(bits), ctx.empty((tokens, size), np.uint16)
        w = [C.c_void_p(shared.tiled[p]) for p in ("w1", "w3", "w2")]
        stream = ctx.stream()

        def call(on, at):
            at.lib.fp8_expert_forward(at._h(), *w, size, size, _lib.vp(x), tokens, 10.0, None, _lib.vp(y), None, on)

        call(None, gpu_ctx)
        gpu_ctx.sync()
        want = y.download()
        graph = Graph(ctx, stream, lambda: call(C.c_void_p(stream), ctx))
        for _ in range(3):
            y.upload(np.zeros_like(want))
            ctx.sync()
            graph.launch()
            np.testing.assert_array_equal(y.download(), want)
        graph.close()
        x.free()
        y.free()
