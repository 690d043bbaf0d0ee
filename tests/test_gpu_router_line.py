"""The router on both sides of each line of its kernel choice -- 24 | 25 tokens, 5120 | wider, few | many sums, and more
tiles than one grid dimension holds -- gives the bits of calls of up to 16 tokens."""

import ctypes as C

import numpy as np
import pytest

from oracle.formats import bf16_bits
from vesper_amd import _lib

pytestmark = pytest.mark.gpu


def project(ctx, w, x, tokens, hidden, experts, logits):
    ctx.lib.gate_project(ctx._h(), C.c_void_p(w), C.c_void_p(x), tokens, hidden, experts, C.c_void_p(logits), None)


@pytest.mark.parametrize("experts,hidden,tokens", [(256, 1024, 24), (256, 5120, 25), (8, 5120, 25), (256, 5124, 31),
                                                   (256, 5124, 32), (3, 8192, 40), (33, 7168, 249)])
def test_rows_do_not_depend_on_the_batch(gpu_ctx, experts, hidden, tokens):
    rng = np.random.default_rng(experts + hidden + tokens)
    w = gpu_ctx.upload((rng.standard_normal((experts, hidden)) * 0.05).astype(np.float32))
    x = gpu_ctx.upload(bf16_bits(rng.standard_normal((tokens, hidden)).astype(np.float32)))
    got, parts = (gpu_ctx.empty((tokens, experts), np.float32) for _ in range(2))
    project(gpu_ctx, w.ptr, x.ptr, tokens, hidden, experts, got.ptr)
    for i in range(0, tokens, 16):
        project(gpu_ctx, w.ptr, x.ptr + 2 * hidden * i, min(16, tokens - i), hidden, experts, parts.ptr + 4 * experts * i)
    np.testing.assert_array_equal(got.download().view(np.uint32), parts.download().view(np.uint32))
    for a in (w, x, got, parts):
        a.free()


def test_more_tiles_than_a_grid_dimension(gpu_ctx):
    """2^20 experts x 1040 tokens of 4 values: 17,039,360 tiles of 8 x 8, of 16,777,215 that one dimension holds."""
    experts, tokens, hidden = 1 << 20, 1040, 4
    rng = np.random.default_rng(1)
    weight = rng.integers(-8, 9, (experts, hidden)).astype(np.float32)
    rows = rng.integers(-8, 9, (tokens, hidden)).astype(np.float32)
    w, x = gpu_ctx.upload(weight), gpu_ctx.upload(bf16_bits(rows))
    logits = gpu_ctx.malloc(experts * tokens * 4)
    try:
        project(gpu_ctx, w.ptr, x.ptr, tokens, hidden, experts, logits)
        for t in (0, 1, 519, tokens - 1):   # small whole numbers: every sum is exact
            got = gpu_ctx.download(logits + 4 * experts * t, (experts,), np.float32)
            np.testing.assert_array_equal(got, weight @ rows[t])
    finally:
        gpu_ctx.free(logits)
        w.free()
        x.free()
