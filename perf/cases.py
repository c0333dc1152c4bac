"""The calls whose speed this repository looks after.

Each case is one call that a program makes of the attention block: a training
step of the layer (forward and every gradient), an inference forward, a
KV-cache prefill, or one decode step. Sizes run from the smallest calls, where
launches and latency count, to the largest ones the benchmark knows; inputs
have the distributions of ``synthetic.make_inputs`` (x and dy standard normal,
weights uniform within 0.5 / sqrt(C)) and are made on the GPU from the seed.

A case is a dict of plain values:

  kind        "train"    forward + backward through the module
              "packed"   the same over packed variable-length sequences
              "forward"  inference forward of the module under no_grad
              "prefill"  a prompt into a KV cache
              "decode"   one new token per sequence against a KV cache
  B, T        sequences and tokens of each (packed: sequences and the longest;
              decode: sequences and the cache's capacity)
  C, H, N     model width, heads, head width
  tables      dtype of the rotary tables, "bf16" or "fp32"
  yarn        YaRN scale (1.0: plain RoPE)
  table_grad  the rotary tables are trained too
  graph       decode through the captured graph instead of eager calls
"""
from __future__ import annotations

import math
from types import SimpleNamespace

import torch

from memory_efficient_attn_layer_amd import CausalSoftmaxAttention, KVCache, fused_attn_varlen
from memory_efficient_attn_layer_amd.decode import DecodeGraph, decode_step, prefill

EPS = 1e-6
DEVICE = "cuda"


def _case(name, kind, B, T, C, H, N, tables="bf16", yarn=1.0, table_grad=False, graph=False):
    c = dict(kind=kind, B=B, T=T, C=C, H=H, N=N, tables=tables, yarn=yarn, table_grad=table_grad, graph=graph)
    if name is not None:
        c["name"] = name
    return c


def listed():
    return [
        # The smallest training step the repository names (workload 0): launches and host work.
        _case("train-smallest", "train", 2, 256, 256, 4, 64),
        # Fine-tuning on a few sequences of an odd length, fp32 tables, wide heads.
        _case("train-ragged", "train", 3, 999, 768, 6, 128, tables="fp32"),
        # Narrow heads with rotary tables that are trained (both table gradients).
        _case("train-narrow-table-grad", "train", 4, 2048, 512, 16, 32, table_grad=True),
        # A training step on a batch of documents packed back to back.
        _case("train-packed", "packed", 24, 2000, 512, 8, 64),
        # One long sequence under YaRN (workload 2's shape, one sequence).
        _case("train-long", "train", 1, 32768, 512, 8, 64, yarn=4.0),
        # 128-wide heads at long sequences (workload 3's shape, a quarter of the batch).
        _case("train-wide", "train", 4, 8192, 1024, 8, 128),
        # The pretraining step (workload 1).
        _case("train-pretrain", "train", 64, 4096, 512, 8, 64),
        # Scoring a batch of short texts: inference forward of the module.
        _case("forward-batch", "forward", 8, 512, 1024, 16, 64),
        # A chat prompt into the cache of a serving layer (workload 4's widths).
        _case("prefill-chat", "prefill", 1, 700, 2048, 16, 128),
        # The longest prompt (workload 4).
        _case("prefill-longest", "prefill", 1, 131072, 2048, 16, 128, yarn=8.0),
        # One user's next token, eager call (workload 4's widths).
        _case("decode-one", "decode", 1, 4096, 2048, 16, 128, tables="fp32"),
        # The next token of a batch of users, each at a position of its own, replayed from a graph.
        _case("decode-batch", "decode", 64, 4096, 512, 8, 64, tables="fp32", graph=True),
    ]


# Model shapes (C, H, N) that the repository's workloads and tests use, or plain multiples of them.
_SHAPES = ((256, 4, 64), (512, 8, 64), (512, 16, 32), (768, 12, 64), (768, 6, 128), (1024, 8, 128), (1024, 16, 64),
           (2048, 16, 128))


def _log_uniform(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)) - 1e-9)))))


def draw(rng):
    """One more case: sizes log-uniform over what the listed cases stand for (mostly odd), every kind."""
    kind = rng.choice(("train", "train", "packed", "forward", "prefill", "decode"))
    C, H, N = rng.choice(_SHAPES)
    tables = rng.choice(("bf16", "fp32"))
    if kind == "decode":
        T = _log_uniform(rng, 128, 65536)
        B = _log_uniform(rng, 1, max(1, min(64, (1 << 28) // (T * H * N))))
        return _case(None, kind, B, T, C, H, N, tables="fp32", graph=rng.random() < 0.5)
    if kind == "packed":
        T = _log_uniform(rng, 64, 8192)
        return _case(None, kind, _log_uniform(rng, 2, max(2, min(64, 65536 // T))), T, C, H, N, tables=tables)
    T = _log_uniform(rng, 32, 32768)
    B = _log_uniform(rng, 1, max(1, min(64, 65536 // T))) if kind != "prefill" else _log_uniform(rng, 1, max(1, min(8, 65536 // T)))
    grad = kind == "train" and rng.random() < 0.2
    return _case(None, kind, B, T, C, H, N, tables=tables, yarn=rng.choice((1.0, 1.0, 4.0)), table_grad=grad)


def _tables(c, dtype):
    """Rotary tables (T, N) in the adjacent-pair layout, RoPE or YaRN over a quarter or an eighth of the length."""
    T, N, s = c["T"], c["N"], c["yarn"]
    i = torch.arange(N // 2, dtype=torch.float64, device=DEVICE)
    theta = 10000.0 ** (-2.0 * i / N)
    m = 1.0
    if s != 1.0:
        r = (T / s) * theta / (2.0 * math.pi)
        gamma = ((r - 1.0) / 31.0).clamp(0.0, 1.0)
        theta = (1.0 - gamma) * theta / s + gamma * theta
        m = 0.1 * math.log(s) + 1.0
    ang = torch.arange(T, dtype=torch.float64, device=DEVICE)[:, None] * theta[None, :]
    cos, sin = m * torch.cos(ang), m * torch.sin(ang)
    f1 = torch.stack((cos, cos), dim=-1).reshape(T, N)
    f2 = torch.stack((-sin, sin), dim=-1).reshape(T, N)
    return f1.to(dtype), f2.to(dtype)


def _lengths(c):
    """Lengths of a packed batch: a spread between a sixteenth of the longest and the longest, the same for every seed."""
    B, T = c["B"], c["T"]
    return [T if b == 0 else max(1, (T + T * ((37 * b) % 61) // 4) // 16) for b in range(B)]


def _inputs(c, seed):
    """Everything random of a case, as bf16 tensors (and the rotary tables)."""
    g = torch.Generator(device=DEVICE).manual_seed(int(seed) * 7919 + 17)
    B, T, C, H, N = (c[k] for k in "BTCHN")
    bound = 0.5 / C ** 0.5

    def normal(*shape):
        return torch.randn(*shape, device=DEVICE, dtype=torch.float32, generator=g).to(torch.bfloat16)

    def weight(rows, cols):
        w = torch.rand(rows, cols, device=DEVICE, dtype=torch.float32, generator=g)
        return ((w * 2.0 - 1.0) * bound).to(torch.bfloat16)

    d = {k: weight(H * N, C) for k in ("wq", "wk", "wv", "wg")}
    d["wo"] = weight(C, H * N)
    d["f1"], d["f2"] = _tables(c, torch.bfloat16 if c["tables"] == "bf16" else torch.float32)
    shape = {"packed": (sum(_lengths(c)), C), "decode": (B, C)}.get(c["kind"], (B, T, C))
    d["x"] = normal(*shape)
    if c["kind"] in ("train", "packed"):
        d["dy"] = normal(*shape)
    if c["kind"] == "decode":
        # Keys as the cache holds them (RMS-normalised and rotated rows: norm sqrt(N)), plain values.
        d["k"] = torch.nn.functional.normalize(normal(B, H, T, N).float(), dim=-1).mul_(N ** 0.5).to(torch.bfloat16)
        d["v"] = normal(B, H, T, N).mul_(0.29)
        # Every sequence somewhere in the second half of the capacity.
        d["pos"] = torch.randint(T // 2, T, (B,), device=DEVICE, generator=g, dtype=torch.int32)
    return d


def prepare(case, seed):
    c, d = case, _inputs(case, seed)
    with torch.device(DEVICE):
        layer = CausalSoftmaxAttention(c["C"], c["H"], c["N"]).to(torch.bfloat16)
    with torch.no_grad():
        for key in "qkvgo":
            getattr(layer, key + "_proj").weight.copy_(d["w" + key])
    yarn = SimpleNamespace(factor1=d["f1"], factor2=d["f2"])
    s = {"case": c, "layer": layer, "yarn": yarn, "x": d["x"], "dy": d.get("dy")}
    weights = [getattr(layer, key + "_proj").weight for key in "qkvgo"]
    if c["kind"] in ("train", "packed"):
        s["x"].requires_grad_(True)
        s["leaves"] = [s["x"], *weights]
        if c["table_grad"]:
            s["leaves"] += [d["f1"].requires_grad_(True), d["f2"].requires_grad_(True)]
    if c["kind"] == "packed":
        s["max_len"] = c["T"]
        ends = [0]
        for n in _lengths(c):
            ends.append(ends[-1] + n)
        s["cu"] = torch.tensor(ends, dtype=torch.int32, device=DEVICE)
    if c["kind"] == "prefill":
        s["cache"] = KVCache.empty(c["B"], c["H"], c["N"], c["T"], DEVICE)
    if c["kind"] == "decode":
        s["cache"], s["pos"] = KVCache(d["k"], d["v"]), d["pos"]
        s["weights"] = [w.detach() for w in weights]
        if c["graph"]:
            s["graph"] = DecodeGraph(*s["weights"], d["f1"], d["f2"], c["H"], c["N"], s["cache"], EPS)
    return s


def run(state):
    s, c = state, state["case"]
    layer, yarn, x = s["layer"], s["yarn"], s["x"]
    if c["kind"] in ("train", "packed"):
        if c["kind"] == "train":
            y = layer(x, yarn)
        else:
            y = fused_attn_varlen(x, layer.q_proj, layer.k_proj, layer.v_proj, layer.g_proj, layer.o_proj, yarn,
                                  c["H"], c["N"], s["cu"], s["max_len"])
        return [y.detach(), *torch.autograd.grad(y, s["leaves"], s["dy"])]
    with torch.no_grad():
        if c["kind"] == "forward":
            return [layer(x, yarn)]
        if c["kind"] == "prefill":
            return [layer.prefill(x, yarn, s["cache"]), s["cache"].k, s["cache"].v]
        if c["graph"]:
            y = s["graph"].step(x, s["pos"])
        else:
            y = decode_step(x, *s["weights"], yarn.factor1, yarn.factor2, c["H"], c["N"], s["pos"], s["cache"], EPS)
        return [y, s["cache"].k, s["cache"].v]


def _pairs(c):
    """Query-key pairs of one head, over all sequences."""
    if c["kind"] == "decode":
        return c["B"] * (0.75 * c["T"] + 1)  # positions are uniform over the second half of the capacity
    lens = _lengths(c) if c["kind"] == "packed" else [c["T"]] * c["B"]
    return sum(n * (n + 1) / 2 for n in lens)


def work(case):
    """Products and bytes one pass cannot do without: each input read once, each output written once."""
    c = case
    C, HN = c["C"], c["H"] * c["N"]
    M = {"packed": sum(_lengths(c)), "decode": c["B"]}.get(c["kind"], c["B"] * c["T"])
    gemm = 2.0 * M * C * HN * 5
    attn = 4.0 * HN * _pairs(c)
    weights = 5.0 * HN * C * 2
    table = 2.0 * c["T"] * c["N"] * (2 if c["tables"] == "bf16" else 4)
    if c["kind"] in ("train", "packed"):
        # Gradients: two products for each of the forward's. x, dy read, y, dx written; weights and their gradients.
        return {"flops": 3.0 * (gemm + attn), "bytes": 4.0 * M * C * 2 + 2 * weights + table * (2 if c["table_grad"] else 1)}
    if c["kind"] == "forward":
        return {"flops": gemm + attn, "bytes": 2.0 * M * C * 2 + weights + table}
    if c["kind"] == "prefill":
        return {"flops": gemm + attn, "bytes": 2.0 * M * C * 2 + 2.0 * M * HN * 2 + weights + table}
    return {"flops": gemm + attn, "bytes": 2.0 * HN * 2 * _pairs(c) + weights + 2.0 * M * C * 2}


def tolerance(case):
    """bf16 operands and activations, fp32 sums: every output and gradient comes out 3e-3 to 6e-3 off the 64-bit
    result (measured over the listed cases), so two correct implementations stay within four times that."""
    return {"rel": 2e-2}


class _Attend(torch.autograd.Function):
    """Causal softmax attention of (G, T, N) fp64 rows, in chunks of queries; nothing of size T x T is kept."""

    @staticmethod
    def chunk(G, T):
        return max(1, min(T, (1 << 28) // max(1, G * T)))

    @staticmethod
    def probs(q, k, a, b):
        s = torch.matmul(q[:, a:b], k[:, :b].transpose(1, 2)) / q.shape[-1] ** 0.5
        rows, cols = torch.arange(a, b, device=q.device), torch.arange(b, device=q.device)
        s.masked_fill_(cols[None, :] > rows[:, None], -math.inf)
        return torch.softmax(s, dim=-1)

    @staticmethod
    def forward(ctx, q, k, v):
        ctx.save_for_backward(q, k, v)
        o, n = torch.empty_like(v), _Attend.chunk(q.shape[0], q.shape[1])
        for a in range(0, q.shape[1], n):
            b = min(q.shape[1], a + n)
            o[:, a:b] = torch.matmul(_Attend.probs(q, k, a, b), v[:, :b])
        return o

    @staticmethod
    def backward(ctx, do):
        q, k, v = ctx.saved_tensors
        do = do.contiguous()
        dq, dk, dv = torch.zeros_like(q), torch.zeros_like(k), torch.zeros_like(v)
        n = _Attend.chunk(q.shape[0], q.shape[1])
        for a in range(0, q.shape[1], n):
            b = min(q.shape[1], a + n)
            p = _Attend.probs(q, k, a, b)
            dv[:, :b] += torch.matmul(p.transpose(1, 2), do[:, a:b])
            ds = torch.matmul(do[:, a:b], v[:, :b].transpose(1, 2))
            ds.sub_((ds * p).sum(-1, keepdim=True)).mul_(p).div_(q.shape[-1] ** 0.5)
            dq[:, a:b] = torch.matmul(ds, k[:, :b])
            dk[:, :b] += torch.matmul(ds.transpose(1, 2), q[:, a:b])
        return dq, dk, dv


def _norm(t):
    return t * torch.rsqrt(t.square().mean(-1, keepdim=True) + EPS)


def _rotate(t, f1, f2):
    """t (T, H, N) at the table rows f1, f2 (T, N)."""
    swapped = t.reshape(*t.shape[:-1], -1, 2).flip(-1).reshape(t.shape)
    return t * f1[:, None, :] + swapped * f2[:, None, :]


def _block(x, d, c):
    """The block over one sequence x (T, C), all in fp64. Returns y, the k and the v rows (H, T, N)."""
    T, H, N = x.shape[0], c["H"], c["N"]
    xn = _norm(x)
    q, k, v, g = ((xn @ d[w].t()).reshape(T, H, N) for w in ("wq", "wk", "wv", "wg"))
    f1, f2 = d["f1"][:T], d["f2"][:T]
    q, k = _rotate(_norm(q), f1, f2), _rotate(_norm(k), f1, f2)
    q, k, v = (t.transpose(0, 1).contiguous() for t in (q, k, v))
    o = _Attend.apply(q, k, v).transpose(0, 1)
    return (o * torch.sigmoid(g)).reshape(T, H * N) @ d["wo"].t(), k, v


def exact(case, seed):
    c = case
    d = {n: t if n == "pos" else t.double() for n, t in _inputs(c, seed).items()}
    if c["kind"] == "decode":
        return _exact_decode(c, d)
    x = d["x"]
    rows = _lengths(c) if c["kind"] == "packed" else [c["T"]] * c["B"]
    xs = x.reshape(-1, c["C"]).split(rows)
    if c["kind"] in ("forward", "prefill"):
        with torch.no_grad():
            got = [_block(t, d, c) for t in xs]
        y = torch.stack([t[0] for t in got])
        return [y] if c["kind"] == "forward" else [y, torch.stack([t[1] for t in got]), torch.stack([t[2] for t in got])]
    names = ["wq", "wk", "wv", "wg", "wo"] + (["f1", "f2"] if c["table_grad"] else [])
    for n in names:
        d[n].requires_grad_(True)
    sums = [torch.zeros_like(d[n]) for n in names]
    ys, dxs = [], []
    for t, dy in zip(xs, d["dy"].reshape(-1, c["C"]).split(rows)):
        t = t.detach().requires_grad_(True)
        y = _block(t, d, c)[0]
        dx, *more = torch.autograd.grad(y, [t] + [d[n] for n in names], dy)
        for s, m in zip(sums, more):
            s += m
        ys.append(y.detach())
        dxs.append(dx)
    return [torch.cat(ys).reshape(x.shape), torch.cat(dxs).reshape(x.shape), *sums]


def _exact_decode(c, d):
    B, H, N = c["B"], c["H"], c["N"]
    xn, pos = _norm(d["x"]), d["pos"].long()
    q, k, v, g = ((xn @ d[w].t()).reshape(B, H, N) for w in ("wq", "wk", "wv", "wg"))
    f1, f2 = d["f1"][pos], d["f2"][pos]
    q, k = _rotate(_norm(q), f1, f2), _rotate(_norm(k), f1, f2)
    at = torch.arange(B, device=q.device)
    d["k"][at, :, pos], d["v"][at, :, pos] = k, v
    o = torch.empty_like(q)
    for b in range(B):
        n = int(pos[b]) + 1
        p = torch.softmax((d["k"][b, :, :n] @ q[b, :, :, None])[..., 0] / N ** 0.5, dim=-1)
        o[b] = (p[:, None, :] @ d["v"][b, :, :n])[:, 0]
    y = (o * torch.sigmoid(g)).reshape(B, H * N) @ d["wo"].t()
    return [y, d["k"], d["v"]]
