"""The decode step on values at the ends of their range: infinities in the
cache, products whose squares leave fp32."""
import pytest
import torch

from memory_efficient_attn_layer_amd.decode import KVCache, decode_step
from memory_efficient_attn_layer_amd.yarn import rotary_tables
from oracle import block as ob
from tests.parity_util import assert_out_close
from tests.test_gpu_decode_edges import _reference

pytestmark = pytest.mark.gpu

C, H, CAP = 64, 2, 300


def _inputs(N, B=1):
    g = torch.Generator().manual_seed(N)
    ws = [((torch.rand(H * N, C, generator=g) - 0.5) / C ** 0.5).bfloat16() for _ in range(4)]
    ws.append(((torch.rand(C, H * N, generator=g) - 0.5) / C ** 0.5).bfloat16())
    f1, f2 = rotary_tables(CAP, N, dtype=torch.float32)
    x = torch.randn(B, C, generator=g).bfloat16()
    k = ob.rms_norm(torch.randn(B, H, CAP, N, generator=g), 1e-6).bfloat16()
    v = (torch.randn(B, H, CAP, N, generator=g) * 0.3).bfloat16()
    return ws, f1, f2, x, k, v


def _decode(x, ws, f1, f2, pos, k, v, N, eps=1e-6):
    y = decode_step(x.cuda(), *(w.cuda() for w in ws), f1.cuda(), f2.cuda(), H, N, pos, KVCache(k.cuda(), v.cuda()), eps)
    return y.cpu()


@pytest.mark.parametrize("N,pos", [(32, 257), (64, 259), (128, 131), (256, 67)])
def test_infinite_value_in_the_last_cached_row(N, pos):
    """The slots of a block past the cached rows take no part: an infinity in the
    last row gives infinities of the reference's signs, not NaN."""
    ws, f1, f2, x, k, v = _inputs(N)
    v[0, 1, pos - 1, 3] = float("inf")
    ref, _, _ = _reference(x, ws, f1, f2, [pos], k, v, H, N)
    y = _decode(x, ws, f1, f2, [pos], k, v, N)
    assert bool(ref.isinf().all()) and torch.equal(y.float(), ref)


@pytest.mark.parametrize("N", [32, 64, 128, 256])
@pytest.mark.parametrize("xs,wsc,eps", [(2.0 ** 56, 2.0 ** 20, 1e-6), (2.0 ** -45, 2.0 ** -30, 1e-30)], ids=["large", "small"])
def test_products_whose_squares_leave_fp32(N, xs, wsc, eps):
    """q and k are normalised after the input's scale is taken out, so their
    squares stay in range wherever those of x do."""
    ws, f1, f2, x, k, v = _inputs(N, B=2)
    pos, at = [17, CAP - 1], torch.arange(2)
    ref, kn, _ = _reference(x, ws, f1, f2, pos, k, v, H, N)  # eps is too small to count on either side
    ws[0], ws[1] = ws[0] * wsc, ws[1] * wsc
    kc, vc = k.cuda(), v.cuda()
    y = decode_step((x * xs).cuda(), *(w.cuda() for w in ws), f1.cuda(), f2.cuda(), H, N, pos, KVCache(kc, vc), eps)
    assert_out_close("k row", kc.cpu()[at, :, pos], kn)
    assert_out_close("y", y, ref)
