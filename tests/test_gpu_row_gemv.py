"""The FP8 decode GEMV (up to 32 tokens) at the edges of its workgroup shapes and of its token tiles.

Rows x width below reach every shape rule: few 16-row tiles with 4 and 8 K parts (one chunk in all, fewer chunks than
K parts, 56 chunks and more), the middle range (2 tiles of 4 and 8 K parts, two tiles a wave) and many tiles; token
counts reach the in-kernel quantization, one token tile and two (17 tokens: one in the second tile). On representable
inputs (every partial sum exact in any order) the FP32 sums equal the oracle's bit for bit, and on random inputs a call
that writes no codes (quantized in the kernel, or in the GEMV's load order) equals one that writes them in rows.
"""

import ctypes as C

import numpy as np
import pytest

from oracle.formats import bf16_bits, bf16_values
from oracle.inputs import activations, fp8_block32_expert_normal
from oracle.projections import fp8_projection, fp8_weights
from tests.test_gpu_projections import exact_case, project_both_ways
from vesper_amd import _lib
from vesper_amd.projections import NativeProjections
from vesper_amd.shared import ResidentSharedExpert

pytestmark = pytest.mark.gpu


def projections(w, sw, block):
    return NativeProjections({"layers.0.attn.p.weight": w, "layers.0.attn.p.scale": sw}, block=block,
                             layout={"p": w.shape})


SHAPES = [(*shape, tokens) for shape in ((64, 128), (192, 640), (64, 7168), (4160, 256), (16448, 384))
          for tokens in (1, 2, 4, 5, 8, 16, 17, 32)] + [(4160, 16384, tokens) for tokens in (4, 8, 17)]


@pytest.mark.parametrize("block", [32, 128])
@pytest.mark.parametrize("rows,width,tokens", SHAPES)
def test_shapes_exact_and_alike_with_and_without_codes(gpu_ctx, block, rows, width, tokens):
    seed = block + rows + width + tokens
    w, sw, x = exact_case(block, tokens, rows, width, 1, 2, seed)
    with projections(w, sw, block) as proj:
        bits = bf16_bits(x)
        ref = fp8_projection(bf16_values(bits), w, sw, block)
        for trace, y in project_both_ways(proj, gpu_ctx, "p", bits, rows, width):
            np.testing.assert_array_equal(trace.view(np.uint32), ref["output_fp32"].view(np.uint32))
            np.testing.assert_array_equal(y, ref["output_bf16"])
    rng = np.random.default_rng(seed)
    w, sw = fp8_weights(rng, rows, width, block)
    with projections(w, sw, block) as proj:
        bits = bf16_bits(rng.standard_normal((tokens, width)).astype(np.float32))
        (t_q, y_q), (t_f, y_f) = project_both_ways(proj, gpu_ctx, "p", bits, rows, width)
        np.testing.assert_array_equal(t_f.view(np.uint32), t_q.view(np.uint32))
        np.testing.assert_array_equal(y_f, y_q)


def test_very_wide_projection(gpu_ctx):
    """Block 128, 1024 chunks of 64 rows: K shared between 16 workgroups of 4 parts (16 chunks each)."""
    w, sw, x = exact_case(128, 3, 64, 131072, 1, 1, 5)
    x[:, 1::128] = 0.0
    with projections(w, sw, 128) as proj:
        bits = bf16_bits(x)
        ref = fp8_projection(bf16_values(bits), w, sw, 128)
        for trace, _ in project_both_ways(proj, gpu_ctx, "p", bits, 64, 131072):
            np.testing.assert_allclose(trace, ref["output_fp32"], rtol=0, atol=1e-5 * np.abs(ref["output_fp32"]).max())


@pytest.mark.parametrize("tokens", [1, 3, 4, 5, 16])
@pytest.mark.parametrize("hidden,intermediate", [(128, 128), (512, 384), (2560, 1152)])
def test_shared_expert_alike_with_and_without_stages(hidden, intermediate, tokens):
    """Without requested stages the expert quantizes in its GEMVs (few tokens) or in their load order; the output has
    the bits of the call that writes every stage. A down-input buffer that is only 4-byte aligned is taken too."""
    rng = np.random.default_rng(hidden + intermediate + tokens)
    arrays = fp8_block32_expert_normal(rng, hidden, intermediate)
    x = activations(rng, tokens, hidden)
    with ResidentSharedExpert(arrays, swiglu_limit=10.0, hidden=hidden, intermediate=intermediate) as shared:
        want = shared.forward(x)
        ctx, xd = shared.ctx, shared.work["x"]          # forward left the bits there
        odd = ctx.malloc(tokens * intermediate * 2 + 16)
        for stages in (None, _lib.MxExpertStages(None, None, None, None, odd + 4, None, None, None)):
            yd = ctx.empty((tokens, hidden), np.uint16)
            ctx.lib.fp8_expert_forward(ctx._h(), *[C.c_void_p(shared.tiled[p]) for p in ("w1", "w3", "w2")], hidden,
                                       intermediate, _lib.vp(xd), tokens, 10.0, None, _lib.vp(yd),
                                       None if stages is None else C.byref(stages), None)
            np.testing.assert_array_equal(yd.download(), want["w2"])
            yd.free()
        din = ctx.download(odd + 4, (tokens, intermediate), np.uint16)
        np.testing.assert_array_equal((din.astype(np.uint32) << 16).view(np.float32), want["down_input"])
        ctx.free(odd)
