"""The grouped FP8 product at the edges of its token tiles (16 | 17, up to 32 tokens) and of its workgroup shapes: rows of
few and of many tiles, narrow and long K. On representable inputs each group's rows equal the oracle's projection of that
group's activations bit for bit."""

import ctypes as C

import numpy as np
import pytest

from oracle.formats import bf16_bits, bf16_values
from oracle.projections import fp8_projection
from tests.test_gpu_projections import exact_case
from vesper_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tokens", [1, 4, 5, 16, 17, 32])
@pytest.mark.parametrize("groups,rows,width", [(3, 64, 128), (8, 64, 512), (5, 448, 1024), (8, 576, 512), (2, 64, 8320),
                                               (2, 8256, 1152)])
def test_grouped_exact(gpu_ctx, groups, rows, width, tokens):
    n = groups * rows
    w, sw, _ = exact_case(32, 1, n, width, 2, 2, n + width)
    rng = np.random.default_rng(tokens)
    x = rng.integers(-2, 3, (tokens, groups, width)).astype(np.float32)
    x[..., ::32] = 448.0
    bits = bf16_bits(x)
    wd, swd, xd = gpu_ctx.upload(w), gpu_ctx.upload(sw), gpu_ctx.upload(bits)
    blob = gpu_ctx.malloc(int(gpu_ctx.lib.cdll.mx_fp8_tiled_bytes(n, width, 32)))
    q, s = gpu_ctx.empty((tokens, groups, width), np.uint8), gpu_ctx.empty((tokens, groups, width // 32), np.uint8)
    y, trace = gpu_ctx.empty((tokens, groups, rows), np.uint16), gpu_ctx.empty((tokens, groups, rows), np.float32)
    h, lib = gpu_ctx._h(), gpu_ctx.lib
    lib.fp8_tile(h, _lib.vp(wd), _lib.vp(swd), n, width, 32, C.c_void_p(blob), None)
    lib.act_quant32(h, _lib.vp(xd), _lib.vp(q), _lib.vp(s), tokens * groups, width, None)
    lib.fp8_grouped_projection(h, C.c_void_p(blob), groups, rows, width, _lib.vp(q), _lib.vp(s), tokens, _lib.vp(y),
                               _lib.vp(trace), None)
    got, sums = y.download(), trace.download()
    for g in range(groups):
        part = slice(rows * g, rows * (g + 1))
        ref = fp8_projection(bf16_values(bits[:, g]), w[part], sw[rows // 32 * g:rows // 32 * (g + 1)], 32)
        np.testing.assert_array_equal(sums[:, g].view(np.uint32), ref["output_fp32"].view(np.uint32), err_msg=f"group {g}")
        np.testing.assert_array_equal(got[:, g], ref["output_bf16"], err_msg=f"group {g}")
    gpu_ctx.free(blob)
    for a in (wd, swd, xd, q, s, y, trace):
        a.free()
