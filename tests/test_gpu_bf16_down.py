"""The BF16-activation expert's down product at the edges of its split (8 waves share I / 128 chunks: fewer chunks than
waves, 9, 16 and 18), within the tolerance bar of the float64 formula, and its rows independent of the batch."""

import numpy as np
import pytest

from oracle.expert import expert_reference_stages
from oracle.formats import bf16_bits
from oracle.inputs import activations, mxfp4_expert
from tests.helpers import assert_close
from vesper_amd.expert import BF16ActivationExpert

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hidden,intermediate", [(128, 128), (256, 384), (640, 1152), (384, 2048), (256, 2304)])
def test_down_split(hidden, intermediate):
    rng = np.random.default_rng(hidden + intermediate)
    arrays = mxfp4_expert(rng, hidden, intermediate, scale_lo=118, scale_hi=120)
    x = activations(rng, 16, hidden)
    with BF16ActivationExpert(arrays, hidden=hidden, intermediate=intermediate) as expert:
        whole = expert.forward(x)["y"]
        ref = expert_reference_stages(x, arrays)["y"]
        assert_close(whole, bf16_bits(ref.astype(np.float32)), "y")
        for t in (0, 5, 15):
            np.testing.assert_array_equal(expert.forward(x[t:t + 1])["y"][0], whole[t])
