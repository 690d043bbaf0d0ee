"""W1 / W3 of the exact gate/up core at the edges of its two forms (up to 4 tokens of a slot: the blocks of a chunk
share one MFMA operand; more: one column per token) and of its stages (4 chunks of 128; a last stage of 1 to 4
chunks): bit for bit the block spec's sums (fp4_gemv_spec, src/vesper/formats.py:97-118), as are the SwiGLU
epilogue and the down input's codes and scales on them, for every token."""

import numpy as np
import pytest

from oracle.expert import expert_forward, swiglu
from oracle.formats import quantize_activation
from oracle.inputs import activations, mxfp4_expert
from vesper_amd.expert import ResidentExpert

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hidden", [128, 384, 512, 640, 1152])
@pytest.mark.parametrize("tokens", [1, 2, 4, 5, 9, 16])
def test_gate_up_forms_and_stage_remainders(hidden, tokens):
    rng = np.random.default_rng(1000 * tokens + hidden)
    intermediate = 128
    arrays = mxfp4_expert(rng, hidden, intermediate)
    x = activations(rng, tokens, hidden) * np.float32(2.0) ** rng.integers(-6, 7, (tokens, hidden)).astype(np.float32)
    route = rng.uniform(0.05, 1.5, tokens).astype(np.float32)
    with ResidentExpert(arrays, swiglu_limit=10.0, hidden=hidden, intermediate=intermediate) as expert:
        got = expert.forward(x, route)
    ref = expert_forward(x, arrays, route, 10.0)
    for name in ("w1", "w3"):
        np.testing.assert_array_equal(got[name], ref[name], err_msg=name)
    down_input, trace = swiglu(got["w1"], got["w3"], 10.0, route)
    np.testing.assert_array_equal(got["down_input"].view(np.uint32), down_input.view(np.uint32))
    np.testing.assert_array_equal(got["trace"].view(np.uint32), trace.view(np.uint32))
    codes, scales = quantize_activation(got["down_input"])
    np.testing.assert_array_equal(got["down_q"], codes)
    np.testing.assert_array_equal(got["down_s"], scales)
