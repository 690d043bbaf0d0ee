"""The BF16-activation expert on either side of the token count at which its MFMA operands change places (4 | 5): rows
equal the larger batch's bit for bit, and y and h the float64 formula within the tolerance bar, at chunk counts below, at
and past the wave split and the register ring (1, 2, 9, 33 and 40 gate/up chunks over 8 waves and 4 ring slots); a token
whose down input overflows leaves the other tokens' rows alone."""

import numpy as np
import pytest

from oracle.expert import expert_reference_stages
from oracle.formats import bf16_bits
from oracle.inputs import activations, mxfp4_expert
from tests.helpers import assert_close
from tests.test_gpu_bf16_expert import normwise
from vesper_amd.expert import BF16ActivationExpert

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hidden,intermediate", [(128, 128), (256, 640), (1152, 256), (4224, 128), (5120, 384)])
def test_few_tokens(hidden, intermediate):
    rng = np.random.default_rng(7 * hidden + intermediate)
    arrays = mxfp4_expert(rng, hidden, intermediate, scale_lo=118, scale_hi=120)
    x = activations(rng, 5, hidden)
    with BF16ActivationExpert(arrays, hidden=hidden, intermediate=intermediate) as expert:
        whole, ref = expert.forward(x), expert_reference_stages(x, arrays)
        assert_close(whole["y"], bf16_bits(ref["y"].astype(np.float32)), "y")
        assert normwise(whole["h"], ref["h"]) < 1e-5
        for t in (1, 2, 3, 4):
            got = expert.forward(x[:t])
            assert normwise(got["h"], ref["h"][:t]) < 1e-5
            for name in ("h", "y"):
                np.testing.assert_array_equal(got[name], whole[name][:t], err_msg=name)


def test_an_overflowing_token_stays_alone():
    rng = np.random.default_rng(11)
    arrays = mxfp4_expert(rng, 384, 256, scale_lo=118, scale_hi=120)
    x = activations(rng, 4, 384)
    with BF16ActivationExpert(arrays, hidden=384, intermediate=256) as expert:
        clean = expert.forward(x)["y"]
        x[1, 5] = x[2, 7] = 3e38
        marked = expert.forward(x)["y"]
    np.testing.assert_array_equal(marked[[0, 3]], clean[[0, 3]])
    assert ((marked[[1, 2]] & 0x7F80) == 0x7F80).any(axis=1).all()
