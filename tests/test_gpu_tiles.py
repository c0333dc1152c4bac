"""The tiled output projection, dZ and dx (calls of few tokens) at the edges of
their tiles, and against the row-owning forms that larger calls take."""
import pytest
import torch

from memory_efficient_attn_layer_amd.synthetic import Workload, make_inputs
from tests.parity_util import check_block, gpu_block

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,T,C,H,N", [
    (1, 33, 96, 2, 32),       # 32-token tiles, one row past an edge; heads in pairs within a k-slab
    (5, 13, 160, 2, 64),      # a tile over five sequences; an odd number of 32-wide k-steps
    (130, 1, 64, 1, 128),     # every row another sequence; features past C in the only tile
    (1, 1040, 1024, 8, 128),  # 64-token tiles
    (7, 300, 1024, 32, 32),   # 128-token tiles over sequences of 300
    (2, 65, 832, 8, 64),      # dx feature groups (first 512 features parked in bf16), partial last tile
    (3, 45, 1056, 2, 64),     # the same past C = 1024
], ids=lambda v: str(v))
def test_tiled_forms_match_oracle(B, T, C, H, N):
    check_block(Workload(99, "tiles", B, T, C, H, N), seed=B + T, table_grad=False)


@pytest.mark.parametrize("B,C,H,N", [(260, 256, 2, 64), (130, 800, 8, 64), (130, 1056, 8, 64), (130, 768, 8, 64)],
                         ids=lambda v: str(v))
def test_tiled_and_row_owning_forms_return_the_same_bits(B, C, H, N):
    """A large batch runs the row-owning kernels, one of its sequences alone
    the tiled ones: same products in the same order, same epilogues."""
    w = Workload(99, "tiles", B, 128, C, H, N)
    inp = make_inputs(w, seed=C)
    full = gpu_block(inp, H, N, table_grad=False)
    for b in (0, B - 1):
        one = dict(inp, x=inp["x"][b:b + 1], dy=inp["dy"][b:b + 1])
        got = gpu_block(one, H, N, table_grad=False)
        assert torch.equal(got["y"], full["y"][b:b + 1]) and torch.equal(got["dx"], full["dx"][b:b + 1])
