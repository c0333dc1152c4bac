"""The decode step at the edges of its key splits: positions around a
workgroup's turn of keys (512, 256, 128 or 64 keys for heads of 32 to 256
dimensions), the first and the last cache row, batches on both sides of the
16-token product tiles, against the block's math in fp32 on a random cache."""
import pytest
import torch

from memory_efficient_attn_layer_amd.decode import KVCache, decode_step
from memory_efficient_attn_layer_amd.yarn import rotary_tables
from oracle import block as ob
from tests.parity_util import assert_out_close

pytestmark = pytest.mark.gpu

EPS = 1e-6


def _reference(x, ws, f1, f2, pos, k, v, H, N):
    """y (B, C) and the new k, v rows (B, H, N), all fp32 on the CPU."""
    B, C = x.shape
    xn = ob.rms_norm(x.float(), EPS)
    q, kn, vn, g = ((xn @ w.float().t()).reshape(B, 1, H, N) for w in ws[:4])
    rows = [ob.rotary(ob.rms_norm(t, EPS)[b:b + 1], f1[p:p + 1], f2[p:p + 1]) for t in (q, kn) for b, p in enumerate(pos)]
    q, kn = torch.cat(rows[:B])[:, 0], torch.cat(rows[B:])[:, 0]
    o = torch.empty(B, H, N)
    for b, p in enumerate(pos):
        keys = torch.cat((k[b, :, :p].float(), kn[b, :, None]), dim=1)
        vals = torch.cat((v[b, :, :p].float(), vn[b, 0][:, None]), dim=1)
        pr = torch.softmax((keys @ q[b, :, :, None])[..., 0] / N ** 0.5, dim=-1)
        o[b] = (pr[:, None] @ vals)[:, 0]
    y = (o * torch.sigmoid(g[:, 0])).reshape(B, H * N) @ ws[4].float().t()
    return y, kn, vn[:, 0]


@pytest.mark.parametrize("C,H,N,cap,pos", [
    (96, 2, 32, 1100, [0, 1, 511, 512, 513, 1099]),
    (160, 1, 64, 520, [0, 255, 256, 257, 519]),
    (64, 2, 128, 300, [299, 0, 127, 128, 129]),
    (32, 1, 256, 130, [63, 64, 65, 129, 0]),
    (512, 3, 64, 70, [(7 * b) % 70 for b in range(16)]),   # one product tile of 16 tokens
    (512, 3, 64, 70, [(11 * b) % 70 for b in range(17)]),  # 64-token tiles
    (1056, 2, 64, 3000, [2999]),                           # an odd number of 32-wide k-steps, many splits
], ids=lambda v: str(v) if not isinstance(v, list) else f"B{len(v)}")
def test_decode_step_at_split_edges(C, H, N, cap, pos):
    B, g = len(pos), torch.Generator().manual_seed(C + cap)
    bound = 0.5 / C ** 0.5
    ws = [((torch.rand(H * N, C, generator=g) * 2 - 1) * bound).bfloat16() for _ in range(4)]
    ws.append(((torch.rand(C, H * N, generator=g) * 2 - 1) * bound).bfloat16())
    f1, f2 = rotary_tables(cap, N, dtype=torch.float32)
    x = torch.randn(B, C, generator=g).bfloat16()
    k = ob.rms_norm(torch.randn(B, H, cap, N, generator=g), EPS).bfloat16()
    v = (torch.randn(B, H, cap, N, generator=g) * 0.3).bfloat16()
    cache = KVCache(k.clone().cuda(), v.clone().cuda())
    y = decode_step(x.cuda(), *(w.cuda() for w in ws), f1.cuda(), f2.cuda(), H, N, pos, cache)
    ref, kn, vn = _reference(x, ws, f1, f2, pos, k, v, H, N)
    assert_out_close("y", y, ref)
    at = torch.arange(B)
    assert_out_close("k row", cache.k.cpu()[at, :, pos], kn)
    assert_out_close("v row", cache.v.cpu()[at, :, pos], vn)
    keep = torch.ones(B, cap, dtype=torch.bool)
    keep[at, pos] = False
    for got, was in ((cache.k.cpu(), k), (cache.v.cpu(), v)):
        assert torch.equal(got.transpose(1, 2)[keep], was.transpose(1, 2)[keep])
