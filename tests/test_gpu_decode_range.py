"""The decode step on values at the ends of their range: infinities in the
cache, products whose squares leave fp32, softmax weights below the normal
numbers, positions past the capacity."""
import ctypes

import pytest
import torch

from memory_efficient_attn_layer_amd import _lib
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


@pytest.mark.parametrize("N", [32, 64, 128, 256])
@pytest.mark.parametrize("pos", [1, 2], ids=["across-splits", "within-a-wave"])
def test_weights_below_the_normal_numbers_count(N, pos):
    """A key about 2^-135 behind the best one, with values of 2^127. Rounding q
    to bf16 moves its exponent by at most 2^-9 of 135 plus the new key's share,
    under half a unit: a factor of 1.5."""
    ws, f1, f2, x, k, v = _inputs(N)
    ws[2] = torch.zeros_like(ws[2])
    xn = ob.rms_norm(x.double(), 1e-6)
    q, kn, g = (((xn @ ws[i].double().t()).reshape(1, 1, H, N)) for i in (0, 1, 3))
    q, kn = (ob.rotary(ob.rms_norm(t, 1e-6), f1[pos:pos + 1].double(), f2[pos:pos + 1].double())[0, 0] for t in (q, kn))
    unit = 1.4426950408889634 / N ** 0.5  # log2 units of a logit
    far = (q * kn.bfloat16().double()).sum(-1, keepdim=True).mul(unit).clamp(min=0.0) - 135.0
    k[0, :, 0] = (q * far / (unit * q.square().sum(-1, keepdim=True))).bfloat16()
    k[0, :, 1:pos] = 0.0  # a logit of 0
    v[0] = 0.0
    v[0, :, 0] = 2.0 ** 127
    keys = torch.cat((k[0, :, :pos].double(), kn[:, None]), dim=1)
    p = torch.softmax((keys @ q[:, :, None])[..., 0] / N ** 0.5, dim=-1)
    ref = ((p[:, :1] * 2.0 ** 127) * torch.sigmoid(g[0, 0])).reshape(1, H * N) @ ws[4].double().t()
    assert 2.0 ** -136 < float(p[:, 0].min()) and float(p[:, 0].max()) < 2.0 ** -128
    y = _decode(x, ws, f1, f2, [pos], k, v, N).double()
    ratio = float((y * ref).sum() / ref.square().sum())
    assert 1 / 1.5 < ratio < 1.5


def test_position_past_the_capacity():
    """Clamped to the capacity for the cache, to the tables for the rotary row."""
    N, cap, pos = 64, 40, 45
    ws, f1, f2, x, k, v = _inputs(N)
    k, v = k[:, :, :cap].contiguous(), v[:, :, :cap].contiguous()
    lib, dev = _lib.load(), [t.cuda() for t in (x, *ws, f1, f2)]

    def run(t_max, f1, f2, p):
        d = _lib.desc(1, cap, C, H, N, t_max, 1e-6)
        need = lib.mea_decode_workspace_bytes(ctypes.byref(d))
        kc, vc, y = k.cuda(), v.cuda(), torch.empty(1, C, dtype=torch.bfloat16, device="cuda")
        scratch = torch.empty(need, dtype=torch.uint8, device="cuda")
        at = torch.tensor([p], dtype=torch.int32, device="cuda")
        rc = lib.mea_decode(ctypes.byref(d), *(t.data_ptr() for t in dev[:6]), f1.data_ptr(), f2.data_ptr(), at.data_ptr(),
                            kc.data_ptr(), vc.data_ptr(), y.data_ptr(), scratch.data_ptr(), need, _lib.stream_of(y.device))
        assert rc == 0, _lib.strerror(rc)
        return y.cpu(), kc.cpu(), vc.cpu()

    moved = [t[:cap].clone() for t in dev[6:]]
    for t, full in zip(moved, dev[6:]):
        t[cap - 1] = full[pos]
    for got, want in zip(run(CAP, dev[6], dev[7], pos), run(cap, *moved, cap - 1)):
        assert torch.equal(got, want)
