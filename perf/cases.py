"""The workloads this framework's speed is followed on, through its public entry points.

Kinds of case:

* ``decode``: one generation step of a batch over KV caches (``NSADecodeCache.step``);
* ``prefill``: the whole attention layer's forward over a prompt (``nsa_attention``, no gradients);
* ``train``: the same layer forward and backward;
* ``aligned``: ``nsa_fused_forward`` with the caller's block lists on the aligned grid, forward and backward;
* ``selection``: the selection branch alone, forward and backward (``selection_attn_triton``);
* ``layer``: the model's ``NSAAttention`` module, forward and backward, with its parameters' gradients;
* ``phi``: the compression MLP over the spans of a layer's keys, forward and backward.

``geom`` texts are "l,d,l',n,w,init,local": compression span and stride, selection block, blocks a query selects,
window, whether block 0 is forced and how many most recent blocks are.
"""

import math
import os
import sys

import torch
import torch.nn.functional as F

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "openbox-llm_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

DEV = "cuda"
PLAIN = "32,16,64,16,512,0,0"
DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}


def listed():
    return [
        # one conversation being generated at 32K tokens: latency alone counts
        dict(name="decode_1x32k", kind="decode", dtype="bf16", B=1, T=32768, Hq=64, Hkv=4, D=128, geom=PLAIN,
             ragged=False),
        # a server's batch in generation, its sequences of unlike lengths up to 32K
        dict(name="decode_32x32k", kind="decode", dtype="bf16", B=32, T=32768, Hq=64, Hkv=4, D=128, geom=PLAIN,
             ragged=True),
        # long-document generation: a few sequences at 128K, 32 blocks each
        dict(name="decode_4x128k", kind="decode", dtype="bf16", B=4, T=131072, Hq=32, Hkv=2, D=128,
             geom="32,16,64,32,512,0,0", ragged=False),
        # an ordinary chat prompt, of no round length
        dict(name="prefill_1x1301", kind="prefill", dtype="bf16", B=1, T=1301, Hq=64, Hkv=4, D=128,
             geom="32,16,64,16,512,1,2"),
        # long-context prefill: 128K tokens, some key blocks that stand out
        dict(name="prefill_1x128k", kind="prefill", dtype="bf16", B=1, T=131072, Hq=32, Hkv=2, D=128,
             geom="32,16,64,32,512,0,0"),
        # the headline: long-context training of one layer at 32K
        dict(name="train_1x32k", kind="train", dtype="bf16", B=1, T=32768, Hq=64, Hkv=4, D=128, geom=PLAIN),
        # a numerics check or a small float32 experiment: launches count
        dict(name="train_f32_1x1k", kind="train", dtype="f32", B=1, T=1024, Hq=4, Hkv=1, D=64,
             geom="32,16,64,16,512,1,2"),
        # the aligned grid with the caller's block lists, groups of four heads, a length of no whole blocks
        dict(name="aligned_1x6011", kind="aligned", dtype="bf16", B=1, T=6011, Hq=16, Hkv=4, D=64,
             geom="64,64,64,16,512,0,0"),
        # selection attention as a part of another layer: 4 sequences of 8K
        dict(name="selection_4x8k", kind="selection", dtype="bf16", B=4, T=8192, Hq=16, Hkv=1, D=64, geom=PLAIN),
        # one attention layer of the 12-layer d768 decoder in mixed-precision training, groups of six heads
        dict(name="layer_8x4k", kind="layer", dtype="bf16", B=8, T=4096, Hq=12, Hkv=2, D=64, geom=PLAIN, rope=True),
        # a layer of the small default model (d512, blocks of 16, 256 tokens) in float32
        dict(name="layer_f32_8x256", kind="layer", dtype="f32", B=8, T=256, Hq=8, Hkv=2, D=64,
             geom="16,16,16,4,32,0,0", rope=False),
        # the paper's compressor over one layer's keys
        dict(name="phi_1x32k", kind="phi", dtype="bf16", B=1, T=32768, Hq=4, Hkv=4, D=128, geom=PLAIN, hidden=128),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    heads = [(64, 4, 128), (32, 2, 128), (16, 1, 128), (16, 1, 64), (16, 4, 64), (12, 2, 64), (8, 2, 64)]
    geoms = [PLAIN, "32,16,64,16,512,1,2", "32,16,64,32,512,0,0", "64,64,64,16,512,0,0"]
    kind = rng.choice(["decode", "decode", "prefill", "train", "train", "aligned", "selection", "layer", "phi"])
    Hq, Hkv, D = rng.choice(heads)
    c = dict(kind=kind, dtype="bf16", B=1, T=0, Hq=Hq, Hkv=Hkv, D=D, geom=rng.choice(geoms))
    if kind == "decode":
        c["B"] = _log_int(rng, 1, 32)
        c["T"] = _log_int(rng, 1000, min(131072, (1 << 29) // (c["B"] * Hkv * D)))
        c["ragged"] = rng.random() < 0.5
    elif kind == "prefill":
        c["T"] = _log_int(rng, 300, 131072 * 2 // max(2, Hkv))
    elif kind == "train":
        if rng.random() < 0.3:
            c["dtype"] = "f32"
            c["T"] = _log_int(rng, 300, 65536 // Hq)
        else:
            c["B"] = rng.choice([1, 1, 2])
            c["T"] = _log_int(rng, 300, 32768 // c["B"])
    elif kind == "aligned":
        ls = rng.choice([16, 32, 64])
        c["geom"] = "%d,%d,%d,%d,%d,0,0" % (ls, ls, ls, rng.choice([4, 8, 16]), rng.choice([128, 512]))
        c["T"] = _log_int(rng, 300, 8192)
    elif kind == "selection":
        c["B"] = rng.choice([1, 2, 4])
        c["T"] = _log_int(rng, 500, 8192)
        c["geom"] = "32,16,64,%d,512,0,0" % rng.choice([8, 16])
    elif kind == "layer":
        c["Hq"], c["Hkv"], c["D"] = rng.choice([(12, 2, 64), (16, 1, 64), (16, 4, 64)])
        c["B"] = rng.choice([1, 2, 4, 8])
        c["T"] = _log_int(rng, 500, 32768 // c["B"])
        c["rope"] = rng.random() < 0.7
    else:
        c["T"] = _log_int(rng, 2000, 32768)
        c["hidden"] = rng.choice([32, 64, 128])
        c["geom"] = PLAIN
        c["Hq"] = Hkv
    return c


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _geom(c):
    l, d, ls, n, w, fi, nl = (int(x) for x in c["geom"].split(","))
    return l, d, ls, n, w, bool(fi), nl


class _Rand:
    """Seeded values on the GPU in the case's dtype."""

    def __init__(self, c, seed):
        self.g = torch.Generator(device=DEV).manual_seed(seed * 7919 + 17)
        self.dtype = DTYPES[c["dtype"]]

    def n(self, *shape, dtype=None):
        return torch.randn(*shape, generator=self.g, device=DEV).to(dtype or self.dtype)

    def heads(self, *shape):
        """N(0,1) values with a scale of 0.5 to 2 per head (dimension 1)."""
        s = torch.rand(shape[1], generator=self.g, device=DEV) * 1.5 + 0.5
        x = torch.randn(*shape, generator=self.g, device=DEV)
        return x.mul_(s.view(1, -1, *([1] * (len(shape) - 2)))).to(self.dtype)


def _block_lists(c, r):
    """Causal block lists of the caller: complete blocks in random order, -1 where a query has fewer."""
    ls, n = _geom(c)[2:4]
    nb = c["T"] // ls
    t = torch.arange(c["T"], device=DEV)
    ok = (torch.arange(nb, device=DEV)[None, :] + 1) * ls <= t[:, None] + 1
    sc = torch.rand(c["B"], c["Hkv"], c["T"], nb, generator=r.g, device=DEV).masked_fill_(~ok, -1.0)
    k = min(n, nb)
    v, i = sc.topk(k, dim=-1)
    idx = torch.full((c["B"], c["Hkv"], c["T"], n), -1, device=DEV, dtype=torch.int32)
    idx[..., :k] = torch.where(v >= 0, i, torch.full_like(i, -1)).to(torch.int32)
    return idx


def _attention_inputs(c, seed):
    """q, kc, vc, ks, vs, kw, vw, gate logits and dO of a layer's core."""
    r = _Rand(c, seed)
    B, T, Hq, Hkv, D = (c[k] for k in ("B", "T", "Hq", "Hkv", "D"))
    ins = [r.heads(B, Hq, T, D)] + [r.heads(B, Hkv, T, D) for _ in range(6)]
    if c["kind"] == "prefill" and T >= 16384:
        # every hundredth 64-token block of keys stands out, as headings and names do
        nb = T // 64
        pick = torch.randperm(nb, generator=r.g, device=DEV)[:max(1, nb // 100)]
        tok = (pick[:, None] * 64 + torch.arange(64, device=DEV)[None, :]).reshape(-1)
        for i in (1, 3, 5):
            ins[i][:, :, tok] += 3.0
    ins.append(r.n(B, Hq, T, 3))
    return ins, r.n(B, Hq, T, D), r


def _decode_inputs(c, seed):
    """Prompt keys / values of the six caches, the lengths, and the new token's rows."""
    r = _Rand(c, seed)
    B, T, Hq, Hkv, D = (c[k] for k in ("B", "T", "Hq", "Hkv", "D"))
    prompt = [r.n(B, Hkv, T, D) for _ in range(6)]
    lens = [T - 1] * B
    if c["ragged"]:
        g = torch.Generator().manual_seed(seed + 5)
        lens = torch.randint(max(1, T // 16), T, (B,), generator=g).tolist()
    return prompt, lens, r.n(B, Hq, D), r.n(B, Hq, 3), [r.n(B, Hkv, D) for _ in range(6)]


def _layer_inputs(c, seed):
    """Parameters of the attention module by name, its input and the output's gradient."""
    r = _Rand(c, seed)
    l = _geom(c)[0]
    d, kv = c["Hq"] * c["D"], c["Hkv"] * c["D"]
    f = torch.float32
    p = {"q_proj.weight": r.n(d, d, dtype=f) / math.sqrt(d)}
    for br in ("cmp", "slc", "win"):
        p["k_%s.weight" % br] = r.n(kv, d, dtype=f) / math.sqrt(d)
        p["v_%s.weight" % br] = r.n(kv, d, dtype=f) / math.sqrt(d)
    for cp in ("comp_k", "comp_v"):
        p[cp + ".intra_pos"] = r.n(l, c["D"], dtype=f) * 0.1
        p[cp + ".pool_logits"] = r.n(l, dtype=f) * 0.1
        p[cp + ".proj.weight"] = r.n(c["D"], c["D"], dtype=f) / math.sqrt(c["D"])
    p["gate.weight"] = r.n(3 * c["Hq"], d, dtype=f) / math.sqrt(d)
    p["gate.bias"] = r.n(3 * c["Hq"], dtype=f) * 0.1
    p["out_proj.weight"] = r.n(d, d, dtype=f) / math.sqrt(d)
    return p, r.n(c["B"], c["T"], d, dtype=f), r.n(c["B"], c["T"], d)


def _phi_inputs(c, seed):
    r = _Rand(c, seed)
    l, d = _geom(c)[:2]
    D, H, f = c["D"], c["hidden"], torch.float32
    n = (c["T"] - l) // d + 1
    p = {"intra_pos": r.n(l, D, dtype=f) * 0.1, "fc1.weight": r.n(H, l * D, dtype=f) / math.sqrt(l * D),
         "fc1.bias": r.n(H, dtype=f) * 0.1, "fc2.weight": r.n(D, H, dtype=f) / math.sqrt(H),
         "fc2.bias": r.n(D, dtype=f) * 0.1}
    return p, r.n(c["B"], c["Hkv"], c["T"], D), r.n(c["B"], c["Hkv"], n, D)


# ---------------------------------------------------------------------------
# the passes
# ---------------------------------------------------------------------------

def prepare(case, seed):
    import nsa_decode
    import nsa_fused_kernel
    import nsa_model
    import nsa_selection_backward
    c = dict(case)
    kind = c["kind"]
    l, d, ls, n, w, fi, nl = _geom(c)
    geom = nsa_fused_kernel.NSAGeometry(l, d, ls, n, w, fi, nl)
    if kind == "decode":
        prompt, lens, q, gate, rows = _decode_inputs(c, seed)
        cache = nsa_decode.NSADecodeCache(c["B"], c["Hkv"], c["D"], c["T"], geom, dtype=DTYPES[c["dtype"]])
        cache.prefill(*prompt, lens=lens)
        return dict(c, cache=cache, lens=cache.lens, q=q, gate=gate, rows=rows)
    if kind in ("layer", "phi"):
        p, x, dy = (_layer_inputs if kind == "layer" else _phi_inputs)(c, seed)
        if kind == "layer":
            rope = nsa_model.Rotary(c["D"]) if c["rope"] else None
            m = nsa_model.NSAAttention(c["Hq"] * c["D"], c["Hq"], c["Hkv"], l, n, w, "fused", cmp_stride=d,
                                       sel_block=ls, force_init=fi, n_local=nl, rope=rope).to(DEV)
        else:
            m = nsa_model.MLPCompressor(l, c["D"], c["hidden"]).to(DEV)
        m.load_state_dict(p)
        return dict(c, m=m, g=geom, x=x.requires_grad_(), dy=dy, leaves=[x] + list(m.parameters()))
    ins, do, r = _attention_inputs(c, seed)
    s = dict(c, g=geom, ins=ins, do=do, attention=nsa_fused_kernel.nsa_attention, fused=nsa_fused_kernel.nsa_fused_forward,
             selection=nsa_selection_backward.selection_attn_triton)
    if kind in ("aligned", "selection"):
        s["idx"] = _block_lists(c, r)
    if kind == "selection":
        s["ins"] = [ins[0], ins[3], ins[4]]
    if kind != "prefill":
        for x in s["ins"]:
            x.requires_grad_()
    return s


def _backward(s, out, leaves, do):
    for x in leaves:
        x.grad = None
    out.backward(do)
    return [x.grad for x in leaves]


def run(s):
    kind = s["kind"]
    if kind == "decode":
        # the prompt's lengths again: every pass generates the same next token
        s["cache"].lens = s["lens"]
        out, idx = s["cache"].step(s["q"], s["gate"], s["rows"])
        return dict(out=out, idx=idx, lens=s["cache"].lens, caches=[*s["cache"].caches(), s["cache"].k_cmp,
                                                                   s["cache"].v_cmp])
    if kind == "prefill":
        with torch.no_grad():
            out, idx = s["attention"](*s["ins"], s["g"])
        return dict(out=out, idx=idx)
    if kind == "train":
        out, idx = s["attention"](*s["ins"], s["g"])
        return dict(out=out.detach(), idx=idx, grads=_backward(s, out, s["ins"], s["do"]))
    if kind == "aligned":
        out = s["fused"](*s["ins"], s["idx"], s["g"].sel_block, s["g"].window)
        return dict(out=out.detach(), grads=_backward(s, out, s["ins"], s["do"]))
    if kind == "selection":
        out = s["selection"](*s["ins"], s["idx"], s["g"].sel_block)
        return dict(out=out.detach(), grads=_backward(s, out, s["ins"], s["do"]))
    if kind == "layer":
        if s["dtype"] == "bf16":
            with torch.autocast("cuda", dtype=torch.bfloat16):
                out = s["m"](s["x"])
        else:
            out = s["m"](s["x"])
    else:
        out = s["m"].pool_sequence(s["x"], s["g"].cmp_stride)
    grads = _backward(s, out, s["leaves"], s["dy"])
    if kind == "layer":
        del grads[_SHIFT]
    return dict(out=out.detach(), grads=grads)


# The position code of the pooled keys moves all keys alike, which no softmax sees: its gradient is 0 but for
# rounding, so it is not among a layer's outputs (x, then the parameters in the module's order).
_SHIFT = 8


# ---------------------------------------------------------------------------
# work and tolerance
# ---------------------------------------------------------------------------

def _keys(T, cap):
    """Sum over queries t < T of min(t + 1, cap)."""
    m = min(T, cap)
    return m * (m + 1) // 2 + (T - m) * cap


def _visible(c):
    """Visible (query, key) pairs of the three branches per KV head: window, compression, selection."""
    l, d, ls, n, w = _geom(c)[:5]
    T = c["T"]
    nc = (T - l) // d + 1 if T >= l else 0
    cmp = sum(min(nc, (t - l + 1) // d + 1) for t in range(l - 1, T)) if T < 4096 else T * nc // 2
    return _keys(T, w), cmp, _keys(T, n * ls)


def work(case):
    c = dict(case)
    l, d, ls, n, w = _geom(c)[:5]
    B, T, Hq, Hkv, D = (c[k] for k in ("B", "T", "Hq", "Hkv", "D"))
    e = 2 if c["dtype"] == "bf16" else 4
    rows, keys = B * Hq * T, B * Hkv * T
    kind = c["kind"]
    if kind == "decode":
        t = T * 17 // 32 if c["ragged"] else T
        per = (t - l) // d + 1 + min(t, w) + min(t, n * ls)
        return {"bytes": 2 * B * Hkv * per * D * e + 2 * B * Hq * D * e + 12 * B * Hkv * D * e,
                "flops": 4 * B * Hq * per * D}
    if kind == "phi":
        nc, H = (T - l) // d + 1, c["hidden"]
        m = B * Hkv * nc
        return {"bytes": 2 * keys * D * e + 2 * m * D * e + 3 * (H * l * D + H * D) * 4,
                "flops": 6 * m * (l * D * H + H * D)}
    win, cmp, sel = _visible(c)
    if kind == "selection":
        win = cmp = 0
    per = B * Hq * (win + cmp + sel) * D
    if kind == "prefill":
        return {"bytes": 2 * rows * D * e + 6 * keys * D * e + 3 * rows * e + B * Hkv * T * n * 4, "flops": 4 * per}
    if kind == "selection":
        return {"bytes": 4 * rows * D * e + 4 * keys * D * e + B * Hkv * T * n * 4, "flops": 14 * per}
    if kind == "layer":
        dm = Hq * D
        wide = dm + 6 * Hkv * D + 3 * Hq + dm
        return {"bytes": B * T * dm * (4 + 4 + 2 * e) + 2 * wide * dm * 4, "flops": 14 * per + 6 * B * T * wide * dm}
    return {"bytes": 4 * rows * D * e + 12 * keys * D * e + 6 * rows * e + B * Hkv * T * n * 4, "flops": 14 * per}


def tolerance(case):
    # Against 64 bits: float32 1.2e-6 (sums of up to thousands of terms, and the exponential), bf16 3e-3 (operands and
    # results rounded at 2^-9), a layer in mixed precision 4.5e-3 (its projections too): about four times that, and
    # for float32 room for another order of the sums.  Whole numbers are block choices: a few queries in a thousand
    # have two blocks that tie to rounding.
    if case["dtype"] == "f32":
        return {"rel": 1e-5, "differ": 1e-3}
    return {"rel": 1.6e-2 if case["kind"] == "layer" else 1e-2, "differ": 2e-3}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------

def _through(x, dtype):
    """x as a tensor of `dtype` holds it, the gradient passed through."""
    return x + (x.detach().to(dtype).double() - x.detach())


def _pool64(x, l, d):
    """Means over the spans [i d, i d + l) of dimension -2."""
    return x.unfold(-2, l, d).mean(-1)


def _softmax64(s, keep):
    p = torch.softmax(s.masked_fill(~keep, -1e300), dim=-1)
    return p * keep.any(-1, keepdim=True)


def _overlap64(nc, ns, l, d, ls):
    i = torch.arange(nc, device=DEV, dtype=torch.float64)[:, None] * d
    j = torch.arange(ns, device=DEV, dtype=torch.float64)[None, :] * ls
    return (torch.minimum(i + l, j + ls) - torch.maximum(i, j)).clamp(min=0) / d


def _choose64(p, t, ns, c):
    """Block lists [R, S] of the queries at positions t, of ns blocks, from the compression probabilities p [R, nc]
    summed over the group."""
    l, d, ls, n, w, fi, nl = _geom(c)
    imp = p @ _overlap64(p.shape[-1], ns, l, d, ls)
    j = torch.arange(ns, device=DEV)
    imp = imp.masked_fill((j[None, :] + 1) * ls - 1 > t[:, None], torch.finfo(torch.float32).min)
    cur = t // ls
    if fi:
        imp[:, 0] = float("inf")
    for m in range(nl):
        ok = (cur - m >= 0) & (cur - m < ns)
        imp[torch.arange(len(t), device=DEV)[ok], (cur - m)[ok]] = float("inf")
    return torch.sort(imp, dim=-1, descending=True, stable=True).indices[:, :min(n, ns)]


def _rows64(q, kc, vc, ks, vs, kw, vw, gate, idx, t0, c, branches="csw"):
    """Outputs [G, R, D] of queries t0 .. t0 + R - 1 of one KV head: q [G, R, D], gate [G, R, 3], keys [*, D], idx
    [R, S] or None."""
    l, d, ls, n, w = _geom(c)[:5]
    R, scale = q.shape[1], q.shape[-1] ** -0.5
    t = torch.arange(t0, t0 + R, device=DEV)
    t1 = t0 + R
    g = torch.sigmoid(gate) if gate is not None else None
    out = 0
    if "c" in branches and kc.shape[0] > 0:
        nc = max(1, min(kc.shape[0], (t1 - l) // d + 1 if t1 >= l else 1))
        vis = (torch.arange(nc, device=DEV) * d + l - 1)[None, :] <= t[:, None]
        p = _softmax64(q @ kc[:nc].T * scale, vis)
        out = out + g[..., 0:1] * (p @ vc[:nc])
        if idx is None:
            # a prompt's candidates are its complete blocks; a decode step's reach to the end of the new token's
            ns = int(t[-1]) // ls + 1 if c["kind"] == "decode" else c["T"] // ls
            idx = _choose64(p.detach().sum(0), t, ns, c)
    if "s" in branches and idx is not None and idx.shape[-1] > 0:
        nb = -(-t1 // ls)
        hit = torch.zeros(R, nb + 1, device=DEV, dtype=torch.bool)
        i = idx.long()
        hit.scatter_(1, torch.where((i >= 0) & (i < nb), i, torch.full_like(i, nb)), True)
        keep = hit[:, :nb].repeat_interleave(ls, dim=1)[:, :t1] & (torch.arange(t1, device=DEV)[None, :] <= t[:, None])
        o = _softmax64(q @ ks[:t1].T * scale, keep) @ vs[:t1]
        out = out + (o if g is None else g[..., 1:2] * o)
    if "w" in branches:
        a = max(0, t0 - w + 1)
        pos = torch.arange(a, t1, device=DEV)[None, :]
        keep = (pos <= t[:, None]) & (t[:, None] - pos < w)
        out = out + g[..., 2:3] * (_softmax64(q @ kw[a:t1].T * scale, keep) @ vw[a:t1])
    return out


def _core64(q, kc, vc, ks, vs, kw, vw, gate, idx, do, c, branches="csw"):
    """Output and (with do) gradients of the three-branch core; kc / vc pooled, all float64, idx int or None."""
    B, Hq, T, D = q.shape
    Hkv = ks.shape[1]
    G = Hq // Hkv
    out = torch.empty_like(q)
    ins = [q, kc, vc, ks, vs, kw, vw, gate]
    grads = [None if x is None else torch.zeros_like(x) for x in ins] if do is not None else None
    for b in range(B):
        for h in range(Hkv):
            hs = slice(h * G, (h + 1) * G)
            kv = [None if x is None else x[b, h].detach().clone().requires_grad_(do is not None) for x in ins[1:7]]
            t0 = 0
            while t0 < T:
                R = max(1, min(T - t0, 2048, int(3e7 / (G * min(T, t0 + 1024)))))
                qr = q[b, hs, t0:t0 + R].detach().clone().requires_grad_(do is not None)
                gr = None if gate is None else gate[b, hs, t0:t0 + R].detach().clone().requires_grad_(do is not None)
                with torch.set_grad_enabled(do is not None):
                    o = _rows64(qr, *kv, gr, None if idx is None else idx[b, h, t0:t0 + R], t0, c, branches)
                out[b, hs, t0:t0 + R] = o.detach()
                if do is not None:
                    o.backward(do[b, hs, t0:t0 + R])
                    grads[0][b, hs, t0:t0 + R] = qr.grad
                    if gr is not None:
                        grads[7][b, hs, t0:t0 + R] = gr.grad
                t0 += R
            if do is not None:
                for i, x in enumerate(kv):
                    if x is not None and x.grad is not None:
                        grads[1 + i][b, h] = x.grad
    return out, grads


def _exact_decode(c, seed):
    prompt, lens, q, gate, rows = _decode_inputs(c, seed)
    l, d = _geom(c)[:2]
    G, dt = c["Hq"] // c["Hkv"], DTYPES[c["dtype"]]
    out = torch.empty(c["B"], c["Hq"], c["D"], device=DEV, dtype=torch.float64)
    for b in range(c["B"]):
        L = lens[b] + 1
        for h in range(c["Hkv"]):
            hs = slice(h * G, (h + 1) * G)
            k = [torch.cat([x[b, h, :L - 1], y[b, h][None]]).double() for x, y in zip(prompt, rows)]
            pooled = [_pool64(x, l, d).to(dt).double() for x in k[:2]]
            out[b, hs] = _rows64(q[b, hs].double()[:, None], *pooled, *k[2:], gate[b, hs].double()[:, None], None,
                                 L - 1, c)[:, 0]
    return dict(out=out, idx=None, lens=None, caches=[None] * 8)


def _exact_layer(c, seed):
    p, x, dy = _layer_inputs(c, seed)
    l, d = _geom(c)[:2]
    dt = DTYPES[c["dtype"]]
    B, T, Hq, Hkv, D = (c[k] for k in ("B", "T", "Hq", "Hkv", "D"))
    p = {k: v.double().requires_grad_() for k, v in p.items()}
    x = x.double().requires_grad_()

    def r(v):
        return _through(v, dt)

    def lin(v, w):
        return r(r(v) @ r(w).T)

    cos = sin = None
    if c["rope"]:
        inv = 10000.0 ** (-torch.arange(0, D, 2, dtype=torch.float64, device=DEV) / D)
        ang = torch.arange(T, device=DEV, dtype=torch.float32)[:, None] * inv.float()[None, :]
        cos, sin = ang.cos().to(dt).double(), ang.sin().to(dt).double()

    def heads(y, n, rot, hd=D):
        y = y.view(B, T, n, hd).transpose(1, 2)
        if rot and c["rope"]:
            a, b = y[..., :hd // 2], y[..., hd // 2:]
            y = r(torch.cat([a * cos - b * sin, b * cos + a * sin], -1))
        return y

    q = heads(lin(x, p["q_proj.weight"]), Hq, True)
    ks = [heads(lin(x, p["k_%s.weight" % br]), Hkv, True) for br in ("cmp", "slc", "win")]
    vs = [heads(lin(x, p["v_%s.weight" % br]), Hkv, False) for br in ("cmp", "slc", "win")]
    gate = heads(r(lin(x, p["gate.weight"]) + p["gate.bias"]), Hq, False, 3)

    def pooled(v, cp):
        w = torch.softmax(p[cp + ".pool_logits"], 0)
        m = v.unfold(2, l, d) @ w + w @ p[cp + ".intra_pos"]
        return lin(m, p[cp + ".proj.weight"])

    chain = [q, pooled(ks[0], "comp_k"), pooled(vs[0], "comp_v"), ks[1], vs[1], ks[2], vs[2], gate]
    wo = r(p["out_proj.weight"])
    do = dy.double() @ wo.detach()
    o, grads = _core64(*[v.detach() for v in chain], None, do.view(B, T, Hq, D).transpose(1, 2).contiguous(), c)
    flat = r(o).transpose(1, 2).reshape(B, T, Hq * D)
    out = flat @ wo.T
    out.backward(dy.double())
    torch.autograd.backward(chain, grads)
    import nsa_model  # the module's parameter order only
    names = [k for k, _ in nsa_model.NSAAttention(Hq * D, Hq, Hkv, l).named_parameters()]
    grads = [x.grad] + [p[k].grad for k in names]
    del grads[_SHIFT]
    return dict(out=out.detach(), grads=grads)


def _exact_phi(c, seed):
    p, x, dy = _phi_inputs(c, seed)
    l, d = _geom(c)[:2]
    dt = DTYPES[c["dtype"]]
    p = {k: v.double().requires_grad_() for k, v in p.items()}
    x = x.double().requires_grad_()
    w1, w2 = _through(p["fc1.weight"], dt), _through(p["fc2.weight"], dt)
    z = (x.unfold(2, l, d).transpose(-1, -2) + p["intra_pos"]).flatten(-2)
    out = F.silu(z @ w1.T + p["fc1.bias"]) @ w2.T + p["fc2.bias"]
    out.backward(dy.double())
    return dict(out=out.detach(), grads=[x.grad] + [p[k].grad for k in (
        "intra_pos", "fc1.weight", "fc1.bias", "fc2.weight", "fc2.bias")])


def exact(case, seed):
    c = dict(case)
    kind = c["kind"]
    if kind == "decode":
        return _exact_decode(c, seed)
    if kind == "layer":
        return _exact_layer(c, seed)
    if kind == "phi":
        return _exact_phi(c, seed)
    l, d = _geom(c)[:2]
    ins, do, r = _attention_inputs(c, seed)
    idx = _block_lists(c, r) if kind in ("aligned", "selection") else None
    do = None if kind == "prefill" else do.double()
    dt = DTYPES[c["dtype"]]
    x = [v.double() for v in ins]
    if kind == "selection":
        out, g = _core64(x[0], None, None, x[3], x[4], None, None, None, idx, do, c, "s")
        return dict(out=out, grads=[g[0], g[3], g[4]])
    # pooled tokens are tensors of the input's type
    kc, vc = x[1].requires_grad_(do is not None), x[2].requires_grad_(do is not None)
    kp, vp = _pool64(kc, l, d), _pool64(vc, l, d)
    out, g = _core64(x[0], kp.detach().to(dt).double(), vp.detach().to(dt).double(), *x[3:], idx, do, c)
    if do is None:
        return dict(out=out, idx=None)
    torch.autograd.backward([kp, vp], [g[1], g[2]])
    grads = [g[0], kc.grad, vc.grad, *g[3:]]
    return dict(out=out, grads=grads) if kind == "aligned" else dict(out=out, idx=None, grads=grads)
