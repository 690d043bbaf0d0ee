"""The FP8 decode GEMV where K is shared between workgroups (few rows and a long K) and where a K part is longer than the
64 weight scales that a wave keeps. On representable inputs (every partial sum exact in any order) the FP32 sums equal
the oracle's bit for bit, and on random inputs a call that writes no codes equals one that writes them."""

import ctypes as C

import numpy as np
import pytest

from oracle.formats import bf16_bits, bf16_values
from oracle.inputs import activations, fp8_block32_expert_normal
from oracle.projections import fp8_projection, fp8_weights
from tests.test_gpu_projections import exact_case, project_both_ways
from tests.test_gpu_row_gemv import projections
from tests.test_gpu_shared_fp8 import check_fp8_stages
from vesper_amd import _lib
from vesper_amd.shared import ResidentSharedExpert

pytestmark = pytest.mark.gpu


def check_exact(gpu_ctx, block, rows, width, tokens):
    w, sw, x = exact_case(block, tokens, rows, width, 1, 1, rows + width + tokens)
    with projections(w, sw, block) as proj:
        bits = bf16_bits(x)
        ref = fp8_projection(bf16_values(bits), w, sw, block)
        for trace, y in project_both_ways(proj, gpu_ctx, "p", bits, rows, width):
            np.testing.assert_array_equal(trace.view(np.uint32), ref["output_fp32"].view(np.uint32))
            np.testing.assert_array_equal(y, ref["output_bf16"])


# 2, 4, 7 and 16 splits, an uneven last one, rows for half the CUs (2 splits), and one tile more (none)
@pytest.mark.parametrize("block", [32, 128])
@pytest.mark.parametrize("rows,width,tokens", [(64, 8320, 5), (64, 16512, 1), (64, 16512, 2), (320, 30848, 3),
                                               (1024, 16384, 17), (2048, 12288, 8), (2112, 12288, 8), (64, 65536, 32)])
def test_split_exact(gpu_ctx, block, rows, width, tokens):
    check_exact(gpu_ctx, block, rows, width, tokens)


@pytest.mark.parametrize("block,tokens", [(32, 1), (128, 4), (128, 20)])
def test_split_alike_with_and_without_codes(gpu_ctx, block, tokens):
    rng = np.random.default_rng(tokens)
    w, sw = fp8_weights(rng, 128, 33792, block)
    with projections(w, sw, block) as proj:
        bits = bf16_bits(rng.standard_normal((tokens, 33792)).astype(np.float32))
        (t_q, y_q), (t_f, y_f) = project_both_ways(proj, gpu_ctx, "p", bits, 128, 33792)
    np.testing.assert_array_equal(t_f.view(np.uint32), t_q.view(np.uint32))
    np.testing.assert_array_equal(y_f, y_q)


@pytest.mark.parametrize("rows,width,tokens", [(4160, 34304, 5), (2112, 33792, 3)])
def test_weight_scales_past_64_chunks_of_a_part(gpu_ctx, rows, width, tokens):
    """Block 128, two tiles a wave (a ring of 3 chunks) and one (of 4): 4 K parts of 67 and of 66 chunks."""
    check_exact(gpu_ctx, 128, rows, width, tokens)


def test_split_down_product_of_the_expert():
    rng = np.random.default_rng(5)
    arrays = fp8_block32_expert_normal(rng, 128, 16640)
    x = activations(rng, 3, 128)
    with ResidentSharedExpert(arrays, swiglu_limit=10.0, hidden=128, intermediate=16640) as shared:
        got = shared.forward(x)
        check_fp8_stages(got, x, arrays, 10.0)
        ctx, xd = shared.ctx, shared.work["x"]
        yd = ctx.empty((3, 128), np.uint16)
        ctx.lib.fp8_expert_forward(ctx._h(), *[C.c_void_p(shared.tiled[p]) for p in ("w1", "w3", "w2")], 128, 16640,
                                   _lib.vp(xd), 3, 10.0, None, _lib.vp(yd), None, None)
        np.testing.assert_array_equal(yd.download(), got["w2"])
        yd.free()
