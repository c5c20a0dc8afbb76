"""The performance cases of the GeneT5 mixture-of-experts framework.

Each case is one call that a program using this package makes: the MoE feed-forward
layer in inference (small queries, one 4,550-token window, a packed batch of windows,
fp32 activations), the fused pre-norm residual block, a training micro-step (forward
and backward with dropout), the self-attention core on packed and on short ragged
sequences, the attention module, and a whole encoder call.

A case is a dict of plain values:
  kind    "moe", "block", "train", "attn", "attn_module" or "encoder"
  moe / block / train:  n (tokens), d, F, E, k, and
      dtype ("bf16" | "f32", moe only), skew (Zipf router bias, moe only),
      drop (dropout probability, train only)
  attn:         lens (sequence lengths as text, comma separated), H, Hkv, alibi,
                scale (standard deviation of the queries and keys)
  attn_module:  B, L, H, Hkv, alibi (embed_dim = 64 H)
  encoder:      B, L, layers (d 768, 12 heads, vocabulary 4,096)

Inputs are drawn on the GPU from the seed: activations N(0, 1), weights N(0, 0.02),
as the package's synthetic configurations have them.
"""
from __future__ import annotations

import math

import torch

from genet5_amd import attention, synth
from genet5_amd.harness import encoder as harness_encoder
from genet5_amd.moe import MoEFeedForward

DEV = "cuda:0"
EPS = 1e-6
VOCAB = 4096

# The layer of every GeneT5 configuration, and two smaller layers for narrower models.
GENET5 = dict(d=768, F=3072, E=16, k=2)
NARROW = (dict(d=512, F=2048, E=8, k=2), dict(d=256, F=1024, E=8, k=2))


def listed():
    return [
        # an interactive query of one short fragment: latency and the experts' weights
        dict(name="moe_query_48", kind="moe", n=48, **GENET5, dtype="bf16", skew=False),
        # one exon-sized sequence of odd length
        dict(name="moe_gene_777", kind="moe", n=777, **GENET5, dtype="bf16", skew=False),
        # configuration 1: 2,048 tokens with fp32 activations and router
        dict(name="moe_f32_2048", kind="moe", n=2048, **GENET5, dtype="f32", skew=False),
        # one whole window (a data-parallel shard of the packed batch)
        dict(name="moe_window_4550", kind="moe", n=4550, **GENET5, dtype="bf16", skew=False),
        # configuration 3: eight packed windows, skewed routing
        dict(name="moe_packed_36400", kind="moe", n=36400, **GENET5, dtype="bf16", skew=True),
        # the MoE half of an encoder block on a packed batch (configuration 4's rows)
        dict(name="block_packed_45500", kind="block", n=45500, **GENET5),
        # a small training batch: one gradient-accumulation micro-step
        dict(name="train_gene_1100", kind="train", n=1100, **GENET5, drop=0.1),
        # the training batch: eight packed windows
        dict(name="train_packed_36400", kind="train", n=36400, **GENET5, drop=0.1),
        # attention of configuration 5: eight windows, ALiBi
        dict(name="attn_windows_8x4550", kind="attn", lens=",".join(["4550"] * 8), H=12, Hkv=12,
             alibi=True, scale=1.0),
        # GeneT5's own attention (no positional bias) over ragged short sequences, grouped
        # key/value heads, sharper scores
        dict(name="attn_ragged_gqa", kind="attn",
             lens="1499,37,811,256,640,95,1203,512,333,1024,18,777", H=12, Hkv=4, alibi=False,
             scale=2.0),
        # the attention module on one short sequence
        dict(name="attn_module_1x512", kind="attn_module", B=1, L=512, H=12, Hkv=12, alibi=True),
        # a denoising call of the encoder on two 512 + 512 token sequences
        dict(name="encoder_2x1024", kind="encoder", B=2, L=1024, layers=12),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    layer = dict(GENET5 if rng.random() < 0.75 else rng.choice(NARROW))
    u = rng.random()
    if u < 0.35:
        return dict(kind="moe", n=_log_int(rng, 16, 40000), **layer,
                    dtype="f32" if rng.random() < 0.2 else "bf16", skew=rng.random() < 0.3)
    if u < 0.52:
        return dict(kind="block", n=_log_int(rng, 64, 45500), **layer)
    if u < 0.68:
        return dict(kind="train", n=_log_int(rng, 256, 30000), **layer,
                    drop=rng.choice([0.0, 0.1]))
    if u < 0.85:
        top = _log_int(rng, 128, 4550)
        lens = [rng.randint(max(1, top // 3), top) for _ in range(rng.randint(1, 8))]
        hkv = rng.choice([12, 12, 4])
        return dict(kind="attn", lens=",".join(map(str, lens)), H=12, Hkv=hkv,
                    alibi=rng.random() < 0.6, scale=rng.choice([0.55, 1.0, 2.0]))
    if u < 0.94:
        return dict(kind="attn_module", B=rng.randint(1, 4), L=_log_int(rng, 64, 2275), H=12,
                    Hkv=rng.choice([12, 4]), alibi=rng.random() < 0.7)
    return dict(kind="encoder", B=rng.randint(1, 2), L=_log_int(rng, 128, 1100), layers=12)


# ---- inputs ---------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _randn(g, *shape, std=1.0, dtype=torch.bfloat16):
    t = torch.randn(*shape, generator=g, device=DEV, dtype=torch.float32)
    return (t * std).to(dtype) if std != 1.0 else t.to(dtype)


def _module(cls, g, dtype, *args, **kw):
    """An nn.Module on the GPU with N(0, 0.02) weights in `dtype`."""
    with torch.device(DEV):
        m = cls(*args, **kw)
    m = m.to(dtype)
    with torch.no_grad():
        for p in m.parameters():
            if p.dim() >= 2:
                p.copy_(_randn(g, *p.shape, std=0.02, dtype=dtype))
            else:
                p.fill_(1.0)
    return m


def _lens(case):
    return [int(v) for v in case["lens"].split(",")]


def _attn_inputs(case, seed):
    g = _gen(seed)
    lens = _lens(case)
    T, H, Hkv = sum(lens), case["H"], case["Hkv"]
    q = _randn(g, T, H, 64, std=case["scale"])
    k = _randn(g, T, Hkv, 64, std=case["scale"])
    v = _randn(g, T, Hkv, 64)
    cu = torch.tensor([0] + lens, device=DEV).cumsum(0).to(torch.int32)
    sl = torch.tensor(attention.alibi_slopes(H), device=DEV) if case["alibi"] else None
    return q, k, v, cu, sl


def prepare(case, seed):
    kind = case["kind"]
    g = _gen(seed)
    st = dict(kind=kind)
    if kind in ("moe", "block", "train"):
        dtype = torch.float32 if case.get("dtype") == "f32" else torch.bfloat16
        skew = case.get("skew", False)
        m = _module(MoEFeedForward, g, dtype, case["d"], case["F"], case.get("drop", 0.0), "silu",
                    case["E"], case["k"], skew)
        if skew:
            m.router_bias = torch.from_numpy(synth.zipf_router_bias(case["E"])).to(DEV)
        m.train(kind == "train")
        st["module"] = m
        st["x"] = _randn(g, case["n"], case["d"], dtype=dtype)
        if kind == "block":
            st["x_add"] = _randn(g, case["n"], case["d"], dtype=dtype)
            st["norm"] = (1.0 + 0.1 * _randn(g, case["d"], dtype=torch.float32))
        if kind == "train":
            st["x"].requires_grad_(True)
            st["dy"] = _randn(g, case["n"], case["d"], dtype=dtype)
            st["seed"] = int(seed)
    elif kind == "attn":
        st["q"], st["k"], st["v"], st["cu"], st["slopes"] = _attn_inputs(case, seed)
        st["max"] = max(_lens(case))
    elif kind == "attn_module":
        cfg = attention.FlashAttentionConfig(embed_dim=64 * case["H"], num_heads=case["H"],
                                             num_kv_heads=case["Hkv"], alibi=case["alibi"])
        st["module"] = _module(attention.FlashAttention, g, torch.bfloat16, cfg).eval()
        st["x"] = _randn(g, case["B"], case["L"], 64 * case["H"])
    else:
        st["module"] = _module(harness_encoder.GeneT5MoE, g, torch.bfloat16, VOCAB, 768,
                               case["layers"]).eval()
        with torch.no_grad():
            # experts upcycled from one dense feed-forward and a little trained apart
            for layer in st["module"].layers:
                for w in (layer.ff.w_gate, layer.ff.w_up, layer.ff.w_down):
                    w.copy_(w[:1] + 0.1 * w)
        st["ids"] = torch.randint(1, VOCAB - 1, (case["B"], case["L"]), generator=g, device=DEV)
    return st


def run(st):
    kind = st["kind"]
    if kind == "train":
        # the step's dropout mask comes from torch's CPU generator; a reproducible
        # training program seeds it
        torch.default_generator.manual_seed(st["seed"])
        m, x = st["module"], st["x"]
        y = m(x)
        gx, gr, gg, gu, gd = torch.autograd.grad(
            y, (x, m.router.weight, m.w_gate, m.w_up, m.w_down), st["dy"])
        return dict(y=y.detach(), dx=gx, router=gr, w_gate=gg, w_up=gu, w_down=gd)
    with torch.no_grad():
        if kind == "moe":
            return st["module"](st["x"])
        if kind == "block":
            return st["module"].residual_block(st["x"], st["norm"], EPS, x_add=st["x_add"])
        if kind == "attn":
            return attention.flash_attn_varlen_func(
                st["q"], st["k"], st["v"], st["cu"], st["cu"], st["max"], st["max"],
                softmax_scale=0.125, alibi_slopes=st["slopes"])
        if kind == "attn_module":
            return st["module"](st["x"])[0]
        return st["module"](st["ids"])["logits"]


# ---- what a pass cannot do without ------------------------------------------------------

def _moe_work(n, d, F, E, k, act_bytes=2):
    """Forward: (bytes of the weights of the experts that n tokens reach plus the rows in
    and out, flops of the routed rows and the router)."""
    used = E * (1.0 - (1.0 - k / E) ** n)
    return (used * 3 * d * F * 2 + E * d * act_bytes + 2 * n * d * act_bytes,
            6.0 * d * F * n * k + 2.0 * n * E * d)


def _attn_work(lens, H, Hkv):
    # every query against every key of its sequence (ALiBi's far keys included)
    return (sum(lens) * 64 * 2.0 * (2 * H + 2 * Hkv),
            4.0 * 64 * H * sum(float(n) * n for n in lens))


def work(case):
    kind = case["kind"]
    if kind in ("moe", "block", "train"):
        n, d, F, E, k = (case[c] for c in ("n", "d", "F", "E", "k"))
        b, f = _moe_work(n, d, F, E, k, 4 if case.get("dtype") == "f32" else 2)
        if kind == "block":
            b += n * d * 2  # the added branch; the norm's weight is negligible
        if kind == "train":
            # dy in, dx out, every expert's weight gradients out; two more products for
            # each of the forward's
            b += 2 * n * d * 2 + E * 3 * d * F * 2
            f *= 3
        return dict(bytes=b, flops=f)
    if kind == "attn":
        b, f = _attn_work(_lens(case), case["H"], case["Hkv"])
        return dict(bytes=b, flops=f)
    if kind == "attn_module":
        T, D, kv = case["B"] * case["L"], 64 * case["H"], 64 * case["Hkv"]
        _, f = _attn_work([case["L"]] * case["B"], case["H"], case["Hkv"])
        w = D * (2 * D + 2 * kv)
        return dict(bytes=2.0 * (2 * T * D + w), flops=f + 2.0 * T * w)
    T, D = case["B"] * case["L"], 768
    mb, mf = _moe_work(T, D, 3072, 16, 2)
    _, af = _attn_work([case["L"]] * case["B"], 12, 12)
    return dict(bytes=case["layers"] * (mb + 8.0 * D * D) + 2.0 * VOCAB * (T + D),
                flops=case["layers"] * (mf + af + 8.0 * T * D * D) + 2.0 * T * D * VOCAB)


def tolerance(case):
    # About four times the distance from the 64-bit result that the path shows: bf16
    # storage of h and of the expert outputs (moe), of dY, dh and dGU (train), of the
    # probabilities (attn).
    kind = case["kind"]
    if kind == "moe":
        return dict(rel=1.2e-2)
    if kind == "block":
        return dict(rel=2e-2)
    if kind == "train":
        return dict(rel=2e-2)
    if kind in ("attn", "attn_module"):
        return dict(rel=1e-2 if kind == "attn" else 1.3e-2)
    # twelve layers of 16-bit activations; a token whose second and third expert are
    # nearly tied may change experts in any of them
    return dict(rel=1e-1)


# ---- the same results in 64 bits --------------------------------------------------------

_M32 = 0xFFFFFFFF


def _fmix32(h):
    h = h ^ (h >> 16)
    h = (h * 0x85EBCA6B) & _M32
    h = h ^ (h >> 13)
    h = (h * 0xC2B2AE35) & _M32
    return h ^ (h >> 16)


def _dropout_scale(rows, F, p, seed):
    """Multiplier (0 or 1 / kept share) of hidden columns [0, F) for assignment rows: the
    counter-based mask that the layer documents."""
    thr = int(round(p * 65536))
    key = _fmix32((_fmix32(rows ^ (seed & _M32)) + (seed >> 32)) & _M32)
    col = torch.arange(F // 2, device=rows.device, dtype=torch.int64)
    bits = _fmix32((key[:, None] + col[None, :] * 0x9E3779B9) & _M32)
    both = torch.stack((bits & 0xFFFF, bits >> 16), dim=-1).reshape(rows.numel(), F)
    return (both >= thr).double() * (65536.0 / (65536 - thr))


def _route64(x, wr, bias, k):
    logits = x @ wr.t().contiguous()
    if bias is not None:
        logits = logits + bias
    top, idx = logits.topk(k, dim=1)
    return idx, torch.softmax(top, dim=1)


def _moe64(x, wr, bias, wg, wu, wd, k):
    idx, gate = _route64(x, wr, bias, k)
    y = torch.zeros_like(x)
    for e in range(wr.shape[0]):
        tok, slot = (idx == e).nonzero(as_tuple=True)
        if tok.numel() == 0:
            continue
        xe = x[tok]
        a = xe @ wg[e].double().t().contiguous()
        h = a * torch.sigmoid(a) * (xe @ wu[e].double().t().contiguous())
        y.index_add_(0, tok, gate[tok, slot, None] * (h @ wd[e].double().t().contiguous()))
    return y


def _bf16(w):
    return w.detach().to(torch.bfloat16)  # the expert products' declared weight type


def _moe_args(m):
    bias = None if m.router_bias is None else m.router_bias.double()
    return (m.router.weight.detach().double(), bias, _bf16(m.w_gate), _bf16(m.w_up),
            _bf16(m.w_down), m.top_k)


def _train64(st, case):
    """Forward and the hand-written backward of y = sum_s gate_s E_s(x)."""
    m = st["module"]
    x, dy = st["x"].detach().double(), st["dy"].double()
    wr, bias, wg, wu, wd, k = _moe_args(m)
    E, F, p = m.num_experts, m.ff_dim, case["drop"]
    seed = 0
    if p > 0:
        g = torch.Generator().manual_seed(st["seed"])
        seed = int(torch.randint(0, 2 ** 62, (1,), generator=g).item())
    idx, gate = _route64(x, wr, bias, k)
    y, dx = torch.zeros_like(x), torch.zeros_like(x)
    dgate = torch.zeros_like(gate)
    d_wg, d_wu, d_wd = (torch.zeros(w.shape, dtype=torch.float64, device=DEV)
                        for w in (wg, wu, wd))
    for e in range(E):
        tok, slot = (idx == e).nonzero(as_tuple=True)
        if tok.numel() == 0:
            continue
        ge, ue, de = wg[e].double(), wu[e].double(), wd[e].double()
        xe, ye = x[tok], dy[tok]
        a, u = xe @ ge.t().contiguous(), xe @ ue.t().contiguous()
        s = torch.sigmoid(a)
        mul = _dropout_scale(tok * k + slot, F, p, seed) if p > 0 else 1.0
        h = a * s * u * mul
        out = h @ de.t().contiguous()
        w = gate[tok, slot, None]
        y.index_add_(0, tok, w * out)
        dgate[tok, slot] = (out * ye).sum(1)
        dout = w * ye
        d_wd[e] = dout.t().contiguous() @ h
        dh = (dout @ de) * mul
        da, du = dh * u * s * (1 + a * (1 - s)), dh * a * s
        d_wg[e] = da.t().contiguous() @ xe
        d_wu[e] = du.t().contiguous() @ xe
        dx.index_add_(0, tok, da @ ge + du @ ue)
    dtop = gate * (dgate - (gate * dgate).sum(1, keepdim=True))
    dlog = torch.zeros(x.shape[0], E, dtype=torch.float64, device=DEV).scatter_(1, idx, dtop)
    dx += dlog @ wr
    return dict(y=y, dx=dx, router=dlog.t().contiguous() @ x, w_gate=d_wg, w_up=d_wu, w_down=d_wd)


def _attn64(q, k, v, lens, slopes):
    q, k, v = q.double(), k.double(), v.double()
    rep = q.shape[1] // k.shape[1]
    out = torch.empty_like(q)
    a = 0
    for n in lens:
        pos = torch.arange(n, device=DEV, dtype=torch.float64)
        dist = (pos[None, :] - pos[:, None]).abs()
        for h in range(q.shape[1]):
            s = q[a:a + n, h] @ k[a:a + n, h // rep].t().contiguous() * 0.125
            if slopes is not None:
                s = s - slopes[h].double() * dist
            out[a:a + n, h] = torch.softmax(s, dim=1) @ v[a:a + n, h // rep].contiguous()
        a += n
    return out


def _norm64(x, w):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + EPS) * w


def _encoder64(st, case):
    m = st["module"]
    B, L = st["ids"].shape
    h = m.embed.weight.double()[st["ids"].reshape(-1)]
    slopes = torch.tensor(attention.alibi_slopes(12), device=DEV)
    lin = lambda a, w: a @ w.detach().double().t().contiguous()
    for layer in m.layers:
        t = _norm64(h, layer.norm1.weight.double())
        at = layer.self_attn
        q, k, v = (lin(t, p.weight).view(B * L, 12, 64) for p in (at.q, at.k, at.v))
        h = h + lin(_attn64(q, k, v, [L] * B, slopes).reshape(B * L, 768), at.o.weight)
        h = h + _moe64(_norm64(h, layer.norm2.weight.double()), *_moe_args(layer.ff))
    return lin(_norm64(h, m.final_norm.weight.double()), m.lm_head.weight).view(B, L, VOCAB)


def exact(case, seed):
    st = prepare(case, seed)
    kind = case["kind"]
    with torch.no_grad():
        if kind == "moe":
            return _moe64(st["x"].double(), *_moe_args(st["module"]))
        if kind == "block":
            h = st["x"].double() + st["x_add"].double()
            return h + _moe64(_norm64(h, st["norm"].double()), *_moe_args(st["module"]))
        if kind == "train":
            return _train64(st, case)
        if kind == "attn":
            return _attn64(st["q"], st["k"], st["v"], _lens(case), st["slopes"])
        if kind == "attn_module":
            m, B, L, H = st["module"], case["B"], case["L"], case["H"]
            x = st["x"].double().view(B * L, -1)
            lin = lambda a, w: a @ w.detach().double().t().contiguous()
            q = lin(x, m.q.weight).view(B * L, H, 64)
            k = lin(x, m.k.weight).view(B * L, case["Hkv"], 64)
            v = lin(x, m.v.weight).view(B * L, case["Hkv"], 64)
            sl = m.alibi_slopes(torch.device(DEV))
            return lin(_attn64(q, k, v, [L] * B, sl).reshape(B * L, 64 * H),
                       m.o.weight).view(B, L, -1)
        return _encoder64(st, case)
