"""The logit bound that selects the softmax form is collected from every
workgroup of the projection: one token with long rotary rows is enough."""
import pytest
import torch

from memory_efficient_attn_layer_amd.attention import FusedAttentionFunction
from memory_efficient_attn_layer_amd.synthetic import Workload, make_inputs
from oracle import block as ob
from tests.parity_util import assert_out_close

pytestmark = pytest.mark.gpu
NAMES = ("x", "wq", "wk", "wv", "wg", "wo", "f1", "f2")


@pytest.mark.parametrize("N,H,t", [(64, 1, 5), (64, 1, 128 * 7 + 3), (64, 1, 128 * 15), (64, 1, 128 * 19 + 100),
                                   (32, 2, 128 * 18 + 1), (128, 1, 128 * 11 + 64), (256, 1, 128 * 13 + 9)])
def test_one_long_row_selects_the_online_softmax(N, H, t):
    # The token's logit with itself is 16 times log2(e) sqrt(N), past 2^127 for
    # the fixed form from N = 64 on (N = 32: 131 in log2 units).
    w = Workload(99, "bound", 1, 128 * 20, 64, H, N)
    inp = make_inputs(w)
    for n in ("f1", "f2"):
        inp[n] = inp[n].clone()
        inp[n][t] *= 4
    with torch.no_grad():
        y = FusedAttentionFunction.apply(*(inp[n].cuda() for n in NAMES), H, N)
    assert_out_close("y", y, ob.block_forward(*(inp[n].float() for n in NAMES), H, N))
