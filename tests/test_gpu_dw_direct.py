"""Weight gradients of wide layers, whose tiles fill the card without splitting
the tokens: bf16 rows straight from the accumulators, partial tiles included."""
import pytest

from memory_efficient_attn_layer_amd.synthetic import Workload
from tests.parity_util import check_block

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,T,C,H,N", [(2, 96, 2048, 16, 128), (1, 70, 1056, 33, 64), (1, 33, 2080, 34, 32)])
def test_block_matches_oracle(B, T, C, H, N):
    check_block(Workload(99, "wide", B, T, C, H, N), seed=C)
