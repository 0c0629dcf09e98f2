"""The performance cases of libmoe_hip: what a program that uses it has it do.

A case is a dict with a "kind" (the entry point that it goes through) and its
sizes:
  forward   moe_hip_forward_dev on device rows, one or several layers
  sublayer  moe_hip_ffn_sublayer_dev, x += MoE(rms_norm(x)) in place
  step      moe_hip_decode_block_dev, block after block: one decode step
  backward  moe_hip_backward_dev, every gradient and the load-balancing loss
  host      moe_hip_forward, the drop-in on host matrices (one sequence)
  row       moe_decode_batch, the drop-in of the decode loop (host rows)

Inputs are N(0, 1) rows and N(0, 0.02) weights, as the models of this library
are initialised.  exact() restates each path in float64 torch.
"""
import ctypes as C
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "llm.c_amd"))

import abi_types  # noqa: E402
import moe_hip as mh  # noqa: E402

EPS = 1e-5
AUX = 0.01
STD = 0.02
M64 = (1 << 64) - 1


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # A long prompt batch through one layer of a large model, with a
        # skewed router (the hottest expert takes several times its share).
        dict(name="prefill large skewed", kind="forward", T=16384, d=2048, F=8192, E=64, k=4, layers=1, skew=0.55),
        # Batch 8 x sequence 512 of the 8-block decoder: the FFN half of a block.
        dict(name="decoder sublayer 8x512", kind="sublayer", T=4096, d=512, F=2048, E=8, k=2),
        # Batch 8 x sequence 512 of the small model.
        dict(name="small layer 8x512", kind="forward", T=4096, d=256, F=1024, E=8, k=2, layers=1, skew=0.0),
        # Many small experts, top-8.
        dict(name="fine-grained experts", kind="forward", T=4096, d=1024, F=512, E=256, k=8, layers=1, skew=0.0),
        # Widths, rows and an expert count that no tile divides.
        dict(name="ragged prefill", kind="forward", T=1003, d=320, F=1376, E=12, k=3, layers=1, skew=0.0),
        # A serving step of many sequences (or short prompts packed together):
        # 8 layers, so the weights come from memory as they do in a model.
        dict(name="serving batch 256", kind="forward", T=256, d=512, F=2048, E=16, k=2, layers=8, skew=0.0),
        # One token for each of 64 sequences through the 8-block decoder.
        dict(name="decode step 64", kind="step", B=64, ctx=1024, d=512, nh=8, nkv=2, F=2048, E=16, k=2, blocks=8),
        # One token of a single sequence: latency.
        dict(name="decode step 1", kind="step", B=1, ctx=1024, d=512, nh=8, nkv=2, F=2048, E=16, k=2, blocks=8),
        # Training: gradients of the small model's and the decoder's layer.
        dict(name="backward small 8x512", kind="backward", T=4096, d=256, F=1024, E=8, k=2),
        dict(name="backward decoder 8x512", kind="backward", T=4096, d=512, F=2048, E=8, k=2),
        # A C program's block forward of one 512-token sequence, host matrices.
        dict(name="host drop-in 512", kind="host", T=512, d=512, F=2048, E=8, k=2),
        # A C program's decode loop, one row: the smallest call.
        dict(name="host decode row", kind="row", T=1, d=512, F=2048, E=8, k=2),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["forward", "forward", "forward", "sublayer", "step", "step", "backward", "backward", "host", "row"])
    while True:
        c = dict(kind=kind)
        if kind == "step":
            hd = rng.choice([32, 64])
            nkv = rng.choice([1, 2, 4])
            nh = nkv * rng.choice([2, 4, 8])
            d = rng.choice([256, 512, 512, 1024])
            c.update(B=_log(rng, 1, 128), ctx=_log(rng, 16, 2048), d=d, nh=nh, nkv=nkv, F=128 * rng.randint(4, 24),
                     E=rng.randint(2, 16), blocks=rng.randint(1, 8), hd=hd)
            c["k"] = rng.randint(1, min(4, c["E"]))
            if c["B"] * c["ctx"] * nkv * hd * c["blocks"] * 8 > 2e9:
                continue
        elif kind in ("host", "row"):
            # (the drop-ins take any widths)
            c.update(T=_log(rng, 8, 2048) if kind == "host" else _log(rng, 1, 64), d=_log(rng, 64, 1024),
                     F=_log(rng, 128, 2816), E=rng.randint(2, 16))
            c["k"] = rng.randint(1, min(4, c["E"]))
            if 12 * c["d"] * c["F"] * c["E"] > 3e8:
                continue
        else:
            c.update(T=_log(rng, 64 if kind != "forward" else 1, 8192), d=64 * _log(rng, 2, 32), F=32 * _log(rng, 8, 256),
                     E=_log(rng, 2, 256))
            c["k"] = rng.randint(1, min(8, c["E"]))
            if kind == "forward":
                c.update(layers=1, skew=round(rng.choice([0.0, 0.0, rng.uniform(0.1, 0.6)]), 3))
            flops = 6.0 * c["T"] * c["k"] * c["d"] * c["F"] * (3 if kind == "backward" else 1)
            if flops > 1.2e12 or 12 * c["d"] * c["F"] * c["E"] > (2e9 if kind == "backward" else 6e9):
                continue
            if kind == "backward" and c["k"] > 4:
                continue
        return c


# ---------------------------------------------------------- synthetic weights
def _mix(z):
    """splitmix64's finaliser on int64 tensors (wrapping products)."""
    def shr(a, n):
        return (a >> n) & ((1 << (64 - n)) - 1)

    z = z ^ shr(z, 30)
    z = z * (0xBF58476D1CE4E5B9 - (1 << 64))
    z = z ^ shr(z, 27)
    z = z * (0x94D049BB133111EB - (1 << 64))
    return z ^ shr(z, 31)


def _mix_int(z):
    z ^= z >> 30
    z = z * 0xBF58476D1CE4E5B9 & M64
    z ^= z >> 27
    z = z * 0x94D049BB133111EB & M64
    return z ^ (z >> 31)


def synth(seed, stream, shape, std, device="cuda"):
    """The values that moe_hip_layer_fill_synthetic documents for one stream
    (seeded N(0, std), element i a function of (seed, stream, i)), as float64
    rounded to float32's values."""
    n = int(np.prod(shape))
    key = _mix_int((seed * 0x9E3779B97F4A7C15 + 0x632BE59BD9B4E019) & M64) ^ _mix_int((stream + 0xD1B54A32D192ED03) & M64)
    key -= (1 << 64) if key >> 63 else 0
    gold = 0x9E3779B97F4A7C15 - (1 << 64)
    i = torch.arange(n, dtype=torch.int64, device=device) * 2
    h1, h2 = _mix((i + 1) * gold + key), _mix((i + 2) * gold + key)
    mask = (1 << 53) - 1
    u1 = (((h1 >> 11) & mask) + 1).double() * 2.0 ** -53
    u2 = ((h2 >> 11) & mask).double() * 2.0 ** -53
    z = torch.sqrt(-2.0 * torch.log(u1)) * torch.cos(2.0 * math.pi * u2)
    return (float(np.float32(std)) * z).float().reshape(shape)


def expert(seed, e, d, F):
    return (synth(seed, 16 + 3 * e, (d, F), STD), synth(seed, 17 + 3 * e, (d, F), STD), synth(seed, 18 + 3 * e, (F, d), STD))


def _gen(seed, salt):
    return torch.Generator(device="cuda").manual_seed((int(seed) * 1000003 + salt) & 0x7FFFFFFF)


def _randn(seed, salt, *shape):
    return torch.randn(*shape, device="cuda", dtype=torch.float32, generator=_gen(seed, salt))


def _bias(case, seed):
    """A skewed router's bias: -skew log(rank), the ranks in a seeded order."""
    if not case.get("skew"):
        return None
    g = torch.Generator().manual_seed(int(seed) & 0x7FFFFFFF)
    rank = torch.randperm(case["E"], generator=g).double() + 1
    b = -case["skew"] * torch.log(rank)
    return (b - b.mean()).float()


def _layer_seed(seed, i):
    return (int(seed) * 16 + i) & 0x7FFFFFFF


# ------------------------------------------------------------- prepare and run
def _ptr(t):
    return C.c_void_p(t.data_ptr())


def _empty(*shape, dtype=torch.float32):
    return torch.empty(*shape, dtype=dtype, device="cuda")


_STREAM = []


def _stream():
    """The program's compute stream: the library's calls share one workspace,
    so they are queued on one stream."""
    if not _STREAM:
        _STREAM.append(torch.cuda.Stream())
    return _STREAM[0]


class State:
    """What a program keeps between calls; host weights leave the library's
    residency cache with it."""

    hw = None

    def __del__(self):
        try:
            if self.hw is not None:
                mh.lib().moe_hip_invalidate(C.byref(self.hw.weights))
        except Exception:
            pass


def _rope(max_seq, hd):
    i = np.arange(hd // 2, dtype=np.float64)
    ang = np.arange(max_seq)[:, None] / 10000.0 ** (2 * i / hd)[None, :]
    return np.cos(ang).astype(np.float32), np.sin(ang).astype(np.float32)


def _attn_weights(case, seed, blk):
    d, nh, nkv, hd = case["d"], case["nh"], case["nkv"], _hd(case)
    shapes = ((d, nh * hd), (d, nkv * hd), (d, nkv * hd), (nh * hd, d))
    return [STD * _randn(seed, 100 * blk + 10 + j, *s) for j, s in enumerate(shapes)]


def _caches(case, seed, blk):
    sh = (case["B"], case["ctx"] + 1, case["nkv"] * _hd(case))
    return _randn(seed, 100 * blk + 20, *sh), _randn(seed, 100 * blk + 21, *sh)


def _hd(case):
    return case.get("hd", case["d"] // case["nh"])


def _positions(case, seed):
    """Most sequences at the full context, the others somewhere before it."""
    B, ctx = case["B"], case["ctx"]
    g = torch.Generator().manual_seed(int(seed) & 0x7FFFFFFF)
    pos = torch.full((B,), ctx, dtype=torch.int32)
    early = torch.rand(B, generator=g) < 0.25
    early[0] = False
    return torch.where(early, torch.randint(0, ctx + 1, (B,), generator=g, dtype=torch.int32), pos)


def _host_weights(case, seed):
    d, F, E = case["d"], case["F"], case["E"]
    return (STD * _randn(seed, 1, d, E), STD * _randn(seed, 2, E, d, F), STD * _randn(seed, 3, E, d, F), STD * _randn(seed, 4, E, F, d))


def prepare(case, seed):
    s = State()
    s.case, kind = case, case["kind"]
    d, F, E, k = case["d"], case["F"], case["E"], case["k"]
    if kind in ("host", "row"):
        s.hw = abi_types.HostMoE(*[w.cpu().numpy() for w in _host_weights(case, seed)], k)
        mh.check(mh.lib().moe_hip_invalidate(C.byref(s.hw.weights)))
        s.x = _randn(seed, 5, case["T"], d).cpu().numpy()
        if kind == "row":
            s.res0 = _randn(seed, 6, case["T"], d).cpu().numpy()
            s.res = s.res0.copy()
            s.cfg = s.hw.config(case["T"])
        return s
    n = case.get("layers", case.get("blocks", 1))
    s.layers = []
    for i in range(n):
        layer = mh.Layer(d, F, E, k)
        layer.fill_synthetic(_layer_seed(seed, i), STD, STD)
        b = _bias(case, _layer_seed(seed, i))
        if b is not None:
            layer.set_bias(b.numpy())
        s.layers.append(layer)
    s.stream = _stream()
    if kind == "step":
        B = case["B"]
        hd = _hd(case)
        s.attn, s.kv = [], []
        for i in range(n):
            a = mh.Attn(d, case["nh"], case["nkv"], hd, case["ctx"] + 1)
            a.load(*[w.cpu().numpy() for w in _attn_weights(case, seed, i)], np.ones(d, np.float32))
            a.set_rope(*_rope(case["ctx"] + 1, hd))
            s.attn.append(a)
            s.kv.append(_caches(case, seed, i))
        s.x0 = _randn(seed, 5, B, d)
        s.x = torch.empty_like(s.x0)
        s.rms = torch.ones(d, device="cuda")
        s.pos = _positions(case, seed).cuda()
        s.ids = [_empty(B, k, dtype=torch.int32) for _ in range(n)]
    else:
        T = case["T"]
        s.x0 = _randn(seed, 5, T, d)
        s.probs, s.ids = _empty(T, E), _empty(T, k, dtype=torch.int32)
        if kind == "forward":
            s.out = [_empty(T, d) for _ in range(n)]
        elif kind == "sublayer":
            s.x, s.xn, s.rms = torch.empty_like(s.x0), _empty(T, d), 1.0 + 0.1 * _randn(seed, 7, d)
        else:
            s.dout = _randn(seed, 6, T, d)
            s.grads = [_empty(T, d), _empty(d, E), _empty(E, d, F), _empty(E, d, F), _empty(E, F, d)]
            s.aux = _empty(1)
    torch.cuda.synchronize()
    return s


def run(s):
    case, kind = s.case, s.case["kind"]
    if kind == "host":
        return mh.moe_forward(s.x, s.hw)
    if kind == "row":
        s.res[:] = s.res0
        mh.check(mh.lib().moe_decode_batch(C.byref(s.hw.weights), C.byref(s.cfg), mh.fptr(s.x), case["T"], mh.fptr(s.res)))
        return s.res
    st = C.c_void_p(s.stream.cuda_stream)
    if kind == "forward":
        T = case["T"]
        for i, layer in enumerate(s.layers):
            last = i + 1 == len(s.layers)
            layer.forward_dev(_ptr(s.x0), T, _ptr(s.out[i]), _ptr(s.probs) if last else None, _ptr(s.ids) if last else None, 0, st)
        return {"out": s.out, "probs": s.probs, "ids": s.ids}
    if kind == "sublayer":
        with torch.cuda.stream(s.stream):
            s.x.copy_(s.x0)
        s.layers[0].ffn_sublayer_dev(_ptr(s.x), _ptr(s.rms), EPS, case["T"], _ptr(s.xn), _ptr(s.probs), _ptr(s.ids), st)
        return {"x": s.x, "x_norm": s.xn, "probs": s.probs, "ids": s.ids}
    if kind == "step":
        with torch.cuda.stream(s.stream):
            s.x.copy_(s.x0)
        for a, layer, kv, ids in zip(s.attn, s.layers, s.kv, s.ids):
            a.decode_block_dev(layer, _ptr(s.rms), _ptr(s.x), case["B"], _ptr(s.pos), _ptr(kv[0]), _ptr(kv[1]), EPS, None, _ptr(ids), st)
        return {"x": s.x, "k": [kv[0] for kv in s.kv], "v": [kv[1] for kv in s.kv], "ids": s.ids}
    s.layers[0].backward_dev(_ptr(s.x0), case["T"], _ptr(s.dout), AUX, *[_ptr(g) for g in s.grads], _ptr(s.aux), 0, st)
    return dict(zip(("dx", "dw_router", "dw_gate", "dw_up", "dw_down"), s.grads), aux=s.aux)


# ----------------------------------------------------------------------- work
def work(case):
    """Bytes: activations in and out once, and every weight that the rows can
    reach once (T k assignments reach at most min(E, T k) experts; fewer at
    random, E (1 - (1 - k/E)^T))."""
    kind, d, F, E, k = case["kind"], case["d"], case["F"], case["E"], case["k"]
    T = case["B"] if kind == "step" else case["T"]
    used = E * (1.0 - (1.0 - k / E) ** T)
    n = case.get("layers", case.get("blocks", 1))
    w = 4.0 * (3 * d * F * used + d * E)
    flops = 6.0 * T * k * d * F + 2.0 * T * d * E
    rows = 4.0 * (2 * T * d + T * E + T * k)
    if kind == "backward":
        # (recompute, the three input products and the three weight products)
        return {"bytes": w + 4.0 * (3 * E * d * F + d * E + 3 * T * d), "flops": 3.0 * flops}
    if kind in ("host", "row"):
        return {"bytes": w + rows, "flops": flops}
    if kind == "step":
        qd, kd = case["nh"] * _hd(case), case["nkv"] * _hd(case)
        proj = 2.0 * d * qd + 2.0 * d * kd
        kv = 2.0 * T * (case["ctx"] + 1) * kd * 0.875
        return {"bytes": n * (w + 4.0 * (proj + kv + 4 * T * d)), "flops": n * (flops + 2.0 * T * proj + 4.0 * T * (case["ctx"] + 1) * qd * 0.875)}
    return {"bytes": n * w + rows + 4.0 * (n - 1) * T * d + (8.0 * T * d if kind == "sublayer" else 0.0), "flops": n * flops}


def tolerance(case):
    """All float32 sums of up to 8192 products: other summation orders differ
    by a few 1e-7 to 2e-6 of the result.  Expert ids are whole numbers: a
    decode step's later blocks route rows that carry earlier rounding, where a
    tie may fall the other way."""
    return {"rel": 1e-5, "max": 3e-4, "differ": 0.002 if case["kind"] == "step" else 0.0}


# ---------------------------------------------------------------------- exact
def _exp_router(v):
    """The router softmax's exponential as the reference defines it: blocks of
    8 experts take a degree-6 polynomial of 2^f, the E % 8 left over exp."""
    z = v.clamp(-88.0, 88.0) * 1.4426950408
    n = torch.floor(z)
    f = z - n
    p = torch.full_like(f, 0.0001540353)
    for c in (0.0013333558, 0.0096181292, 0.0555041086, 0.2402265069, 0.6931471806, 1.0):
        p = p * f + c
    y = p * torch.exp2(n)
    tail = v.shape[1] // 8 * 8
    y[:, tail:] = torch.exp(v[:, tail:])
    return y


def _route(x, wr, bias, k):
    z = x @ wr
    if bias is not None:
        z = z + bias.to(x)
    y = _exp_router(z - z.max(1, keepdim=True).values)
    p = y / y.sum(1, keepdim=True)
    sel, ids = torch.topk(p, k, dim=1)
    return p, ids, sel, sel / sel.sum(1, keepdim=True)


def _experts(x, ids, gw, weights, E):
    out = torch.zeros_like(x)
    for e in range(E):
        t, s = (ids == e).nonzero(as_tuple=True)
        if t.numel() == 0:
            continue
        wg, wu, wd = (w.double() for w in weights(e))
        g = x[t] @ wg
        h = torch.nn.functional.silu(g) * (x[t] @ wu)
        out.index_add_(0, t, gw[t, s].unsqueeze(1) * (h @ wd))
    return out


def _norm(x, w):
    return x * torch.rsqrt(x.square().mean(1, keepdim=True) + float(np.float32(EPS))) * w


def exact(case, seed):
    kind, d, F, E, k = case["kind"], case["d"], case["F"], case["E"], case["k"]
    if kind in ("host", "row"):
        wr, wg, wu, wd = _host_weights(case, seed)
        x = _randn(seed, 5, case["T"], d).double()
        p, ids, _, gw = _route(x, wr.double(), None, k)
        out = _experts(x, ids, gw, lambda e: (wg[e], wu[e], wd[e]), E)
        return (out, p, None) if kind == "host" else out + _randn(seed, 6, case["T"], d).double()
    if kind == "step":
        return _exact_step(case, seed)
    T = case["T"]
    x = _randn(seed, 5, T, d).double()
    if kind == "backward":
        return _exact_backward(case, seed, x, _randn(seed, 6, T, d).double())
    xn = _norm(x, (1.0 + 0.1 * _randn(seed, 7, d)).double()) if kind == "sublayer" else x
    outs = []
    for i in range(case.get("layers", 1)):
        ls = _layer_seed(seed, i)
        p, ids, _, gw = _route(xn, synth(ls, 1, (d, E), STD).double(), _bias(case, ls), k)
        outs.append(_experts(xn, ids, gw, lambda e: expert(ls, e, d, F), E))
    if kind == "sublayer":
        return {"x": x + outs[0], "x_norm": xn, "probs": p, "ids": None}
    return {"out": outs, "probs": p, "ids": None}


def _exact_step(case, seed):
    B, d, nh, nkv, hd, F, E, k = (case["B"], case["d"], case["nh"], case["nkv"], _hd(case), case["F"], case["E"], case["k"])
    x = _randn(seed, 5, B, d).double()
    pos = _positions(case, seed).cuda().long()
    cos, sin = (torch.from_numpy(t).cuda().double()[pos].unsqueeze(1) for t in _rope(case["ctx"] + 1, hd))
    rows = torch.arange(B, device="cuda")
    seen = torch.arange(case["ctx"] + 1, device="cuda").unsqueeze(0) <= pos.unsqueeze(1)
    ks, vs = [], []

    def rope(v, heads):
        v = v.reshape(B, heads, hd // 2, 2)
        a, b = v[..., 0], v[..., 1]
        return torch.stack((a * cos - b * sin, a * sin + b * cos), -1).reshape(B, heads, hd)

    for i in range(case["blocks"]):
        wq, wk, wv, wo = (w.double() for w in _attn_weights(case, seed, i))
        kc, vc = (c.double() for c in _caches(case, seed, i))
        xn = _norm(x, 1.0)
        q = rope(xn @ wq, nh)
        kc[rows, pos] = rope(xn @ wk, nkv).reshape(B, -1)
        vc[rows, pos] = xn @ wv
        o = torch.empty(B, nh, hd, dtype=torch.float64, device="cuda")
        for h in range(nh):
            lo = (h // (nh // nkv)) * hd
            a = (kc[..., lo:lo + hd] * q[:, h].unsqueeze(1)).sum(-1) / math.sqrt(hd)
            a = torch.softmax(a.masked_fill(~seen, -math.inf), 1)
            o[:, h] = (a.unsqueeze(-1) * vc[..., lo:lo + hd]).sum(1)
        x = x + o.reshape(B, -1) @ wo
        ls = _layer_seed(seed, i)
        xn = _norm(x, 1.0)
        p, ids, _, gw = _route(xn, synth(ls, 1, (d, E), STD).double(), None, k)
        x = x + _experts(xn, ids, gw, lambda e: expert(ls, e, d, F), E)
        ks.append(kc.float())
        vs.append(vc.float())
    return {"x": x, "k": ks, "v": vs, "ids": [None] * case["blocks"]}


def _exact_backward(case, seed, x, dout):
    T, d, F, E, k = case["T"], case["d"], case["F"], case["E"], case["k"]
    ls = _layer_seed(seed, 0)
    wr = synth(ls, 1, (d, E), STD).double()
    p, ids, sel, gw = _route(x, wr, None, k)
    dx, dgw = torch.zeros_like(x), torch.zeros_like(gw)
    dwg, dwu, dwd = [], [], []
    for e in range(E):
        wg, wu, wd = (w.double() for w in expert(ls, e, d, F))
        t, s = (ids == e).nonzero(as_tuple=True)
        xe, dy = x[t], dout[t]
        g, u = xe @ wg, xe @ wu
        sg = torch.sigmoid(g)
        h = g * sg * u
        dgw[t, s] = (dy * (h @ wd)).sum(1)
        dy = dy * gw[t, s].unsqueeze(1)
        dh = dy @ wd.T
        dg, du = dh * u * (sg + g * sg * (1.0 - sg)), dh * g * sg
        dx.index_add_(0, t, dg @ wg.T + du @ wu.T)
        dwg.append((xe.T @ dg).float())
        dwu.append((xe.T @ du).float())
        dwd.append((h.T @ dy).float())
    frac = torch.bincount(ids.reshape(-1), minlength=E).double() / (T * k)
    dp = (AUX * E / T * frac).expand(T, E).clone()
    dsel = (dgw - (dgw * gw).sum(1, keepdim=True)) / sel.sum(1, keepdim=True)
    dp.scatter_add_(1, ids, dsel)
    dz = p * (dp - (p * dp).sum(1, keepdim=True))
    return {"dx": dx + dz @ wr.T, "dw_router": x.T @ dz, "dw_gate": torch.stack(dwg), "dw_up": torch.stack(dwu),
            "dw_down": torch.stack(dwd), "aux": (E * (frac * p.mean(0)).sum()).reshape(1)}
