"""The attention kernels with two wave groups per workgroup (small grids), where
the groups' shares end unevenly: one tile more for one group, tiles past the
diagonal or the sequence end, rows that meet no key in the second group."""
import pytest
import torch

from memory_efficient_attn_layer_amd import stages
from memory_efficient_attn_layer_amd.synthetic import Workload
from tests.parity_util import assert_grad_close, assert_out_close, check_block
from tests.test_gpu_varlen import _gpu_varlen, _inputs, _oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [256, 257, 321, 385, 513])
@pytest.mark.parametrize("H,N", [(2, 32), (1, 64), (1, 128)], ids=lambda v: str(v))
def test_block_matches_oracle(T, H, N):
    check_block(Workload(99, "split", 1, T, 64, H, N), seed=T + N, table_grad=T % 2 == 0)


@pytest.mark.parametrize("scale", [1.0, 6.0], ids=["plain", "wide-logits"])
@pytest.mark.parametrize("H,N", [(2, 32), (1, 64), (1, 128)], ids=lambda v: str(v))
def test_online_softmax_of_two_groups(H, N, scale):
    """The stage entry point has no logit bound, so each group keeps a running
    maximum of its own and the sums meet rescaled."""
    g = torch.Generator("cuda").manual_seed(N)
    for T in (256, 300, 449):
        q, k, v = (torch.randn(1, H, T, N, device="cuda", generator=g).mul(s).bfloat16() for s in (scale, scale, 1.0))
        o, lse = stages.attn_fwd(q, k, v)
        s = (q.float().cpu() @ k.float().cpu().transpose(-1, -2)) / N ** 0.5
        s.masked_fill_(~torch.ones(T, T, dtype=torch.bool).tril(), float("-inf"))
        ref = (torch.softmax(s, -1) @ v.float().cpu()).transpose(1, 2).reshape(1, T, H * N)
        assert_out_close("o", o, ref)
        assert_out_close("lse", lse, torch.logsumexp(s, -1), tol=1e-3)


def test_packed_sequences_of_uneven_lengths():
    lens, C, H, N = [300, 1, 70, 257], 64, 2, 64
    inp = _inputs(lens, C, H, N, t_max=300, seed=3)
    got, ref = _gpu_varlen(inp, lens, H, N, table_grad=False), _oracle(inp, lens, H, N)
    for n in ("y", "dx", "dwq", "dwk", "dwv", "dwg", "dwo"):
        assert_out_close(n, got[n], ref[n], tol=3e-2)


def test_packed_table_gradients():
    lens, C, H, N = [300, 1, 0, 257, 90], 64, 2, 64
    inp = _inputs(lens, C, H, N, t_max=310, seed=5)
    got, ref = _gpu_varlen(inp, lens, H, N), _oracle(inp, lens, H, N)
    for n in ("df1", "df2"):
        assert_grad_close(n, got[n][:300], ref[n][:300])
        assert not bool(got[n][300:].any())


@pytest.mark.parametrize("B,T,H,N", [(17, 300, 5, 64), (16, 256, 8, 64), (17, 383, 5, 128), (8, 512, 8, 128)],
                         ids=["n64-255", "n64-256", "n128-255", "n128-256"])
def test_both_sides_of_the_grid_line(B, T, H, N):
    check_block(Workload(99, "line", B, T, 64, H, N), seed=T, table_grad=False)
