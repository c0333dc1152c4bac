"""The projection with weights past an XCD's L2 (more than 4 MB of q, k, v and g
rows), whose tiles run in bands of eight token tiles: packed sequences and
prompts into a larger cache, with a partial last band."""
import pytest
import torch

from memory_efficient_attn_layer_amd.decode import KVCache, prefill
from memory_efficient_attn_layer_amd.synthetic import Workload, make_inputs
from oracle import block as ob
from tests.parity_util import assert_grad_close, assert_out_close
from tests.test_gpu_varlen import _gpu_varlen, _inputs, _oracle

pytestmark = pytest.mark.gpu

SHAPES = [(1024, 32, 32), (1024, 16, 64), (1024, 8, 128), (1024, 4, 256)]


@pytest.mark.parametrize("C,H,N", SHAPES)
@pytest.mark.parametrize("tables", ["bf16", "fp32"])
def test_packed_sequences(C, H, N, tables):
    lens = [413, 1, 0, 300, 129, 260]  # 1103 tokens: nine token tiles
    assert 8 * C * H * N > 4 << 20
    inp = _inputs(lens, C, H, N, t_max=450, seed=N)
    if tables == "bf16":
        inp["f1"], inp["f2"] = inp["f1"].bfloat16(), inp["f2"].bfloat16()
    got, ref = _gpu_varlen(inp, lens, H, N), _oracle(inp, lens, H, N)
    assert_out_close("y", got["y"], ref["y"])
    for n in ("dx", "dwq", "dwk", "dwv", "dwg", "dwo", "df1", "df2"):
        assert_grad_close(n, got[n], ref[n], scale=ref["dwv"])


@pytest.mark.parametrize("C,H,N", SHAPES)
def test_prompt_into_a_larger_cache(C, H, N):
    B, T, cap = 1, 1100, 1300
    inp = make_inputs(Workload(99, "bands", B, cap, C, H, N), seed=N)
    x = inp["x"][:, :T].contiguous()
    names = ("wq", "wk", "wv", "wg", "wo", "f1", "f2")
    cache = KVCache.empty(B, H, N, cap, "cuda")
    for t in (cache.k, cache.v):
        t.fill_(7.0)
    y = prefill(x.cuda(), *(inp[n].cuda() for n in names), H, N, cache)
    ref = ob.block_intermediates(x.float(), *(inp[n].float() for n in names), H, N)
    assert_out_close("y", y, ref["y"])
    for n, t in (("k", cache.k), ("v", cache.v)):
        assert_out_close(n, t[:, :, :T], ref[n].transpose(1, 2))
        assert bool((t[:, :, T:] == 7.0).all())
