"""The work that a program built on this library has it do, as timed cases.

Every case is one call (or the calls of one decode step) through the public
Python binding of the C ABI, at the sizes a GLM-shaped model brings (hidden
6144, 256 experts of inner size 2048, 8 per token, dense inner size 12288,
attention of 64 heads over a 512-wide compressed cache) or at smaller generic
ones. Kinds:

  expert     one MXFP4 expert's SwiGLU FFN on one position (wl_expert_ffn)
  moe        one or more MoE layers: decode at one token (wl_run_moe_residual,
             wl_run_chain for several layers), prefill at more
             (wl_run_moe_batched)
  dense      a dense SwiGLU layer, decode (wl_run_moe_residual) and prefill
             (wl_run_moe_batched)
  attention  one decode position through MLA attention layers, the first of
             them with its own key indexer (wl_run_attention)

Weights are drawn with torch and quantised here (MXFP4: E2M1 values, one
power-of-two scale per 32), so exact() rebuilds the same model in 64 bits
without the library.
"""
import torch

from windlass_amd import moe

DEV = "cuda"
GLM = dict(hidden=6144, inter=2048, experts=256, topk=8)
GLM_ATTN = dict(hidden=6144, n_heads=64, q_lora_rank=2048, kv_lora_rank=512, qk_nope=192, qk_rope=64, v_head=256,
                index_n_heads=32, index_head_dim=128, index_topk=2048)
DENSE_INTER = 12288
EPS, ROPE_THETA, SCALING = 1e-5, 1e6, 2.5
LORA_EPS = 1e-6  # the LoRA norms' and the index keys' epsilon


def _moe(name, tokens, layers=1, shared="bf16", **shape):
    c = dict(GLM, **shape)
    return dict(name=name, kind="moe", tokens=tokens, layers=layers, shared=shared, **c)


def listed():
    return [
        # one expert on one position: the smallest call, the one that programs
        # placing experts themselves make (reference-layout block)
        dict(name="expert_1", kind="expert", hidden=6144, inter=2048),
        # one token through one MoE layer: every step of every decode
        _moe("moe_decode", 1),
        # one token through consecutive MoE layers, as a decode loop runs them
        _moe("moe_chain_4", 1, layers=4),
        # a handful of tokens: a short prompt, a few sequences decoded together,
        # drafted tokens being verified
        _moe("moe_prefill_7", 7),
        # a small batch: many sequences decoded together
        _moe("moe_prefill_64", 64),
        # a prompt of ordinary length through a smaller model with an MXFP4
        # shared expert; no size is a multiple of a tile
        _moe("moe_prefill_333_small", 333, shared="mxfp4", hidden=2944, inter=1408, experts=160, topk=6),
        # a prompt of ordinary length, and the longest chunk a call runs at once
        _moe("moe_prefill_1000", 1000),
        _moe("moe_prefill_4096", 4096),
        # the dense layers a model starts with, at decode and at prefill
        dict(name="dense_decode", kind="dense", tokens=1, hidden=6144, inter=DENSE_INTER),
        dict(name="dense_prefill_200", kind="dense", tokens=200, hidden=6144, inter=DENSE_INTER),
        # attention of one decoded token: a layer with its own indexer and a
        # layer that takes over its selection, in a chat-length context; an
        # indexer layer in a long one
        dict(name="attention_4k", kind="attention", keys=4096, layers=2, **GLM_ATTN),
        dict(name="attention_16k", kind="attention", keys=16384, layers=1, **GLM_ATTN),
    ]


def _log(rng, lo, hi):
    """An integer of [lo, hi], uniform over the logarithm."""
    return min(hi, max(lo, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    r = rng.random()
    if r < 0.05:
        return dict(kind="expert", hidden=128 * rng.randint(16, 48), inter=128 * rng.randint(4, 16))
    if r < 0.65:
        c = dict(GLM)
        if rng.random() < 0.4:
            c = dict(hidden=128 * rng.randint(16, 48), inter=128 * rng.randint(4, 16), experts=16 * rng.randint(4, 16),
                     topk=rng.randint(2, 8))
        tokens = 1 if rng.random() < 0.2 else _log(rng, 2, 4096)
        layers = rng.randint(1, 4) if tokens == 1 else 1
        return dict(kind="moe", tokens=tokens, layers=layers, shared=rng.choice(["bf16", "bf16", "mxfp4"]), **c)
    if r < 0.8:
        tokens = 1 if rng.random() < 0.3 else _log(rng, 2, 512)
        return dict(kind="dense", tokens=tokens, hidden=128 * rng.randint(16, 48), inter=8 * rng.randint(256, 1536))
    keys = _log(rng, 64, 16384)
    return dict(kind="attention", keys=keys, layers=2 if keys <= 4096 else 1, **GLM_ATTN)


# ---- inputs -----------------------------------------------------------------
def _gen(seed, *tags):
    g = torch.Generator(device=DEV)
    s = seed
    for t in tags:
        s = (s * 1000003 + t + 1) & 0x7FFFFFFFFFFF
    g.manual_seed(s)
    return g


def _randn(g, *shape, std=1.0):
    return torch.randn(*shape, generator=g, device=DEV).mul_(std)


def _bf16(g, *shape, std):
    return _randn(g, *shape, std=std).to(torch.bfloat16)


def _norm_weight(g, n):
    return (1.0 + _randn(g, n, std=0.1)).to(torch.bfloat16)


def _mxfp4(g, rows, cols):
    """A weight matrix of unit-variance outputs in MXFP4: packed nibbles
    [rows, cols/2] (low nibble = even column) and E8M0 scales [rows, cols/32]."""
    w = _randn(g, rows * cols // 32, 32, std=cols ** -0.5)
    e = torch.frexp(w.abs().amax(1)).exponent.sub_(3)  # the block's largest value falls in [4, 8)
    a = torch.ldexp(w, -e[:, None])
    sign = (a < 0).to(torch.uint8).mul_(8)
    a = a.abs_().clamp_(max=6.0)
    step = 0.5 + 0.5 * (a >= 2) + (a >= 4)
    v = torch.round(a / step).mul_(step)
    code = torch.where(v < 2, v * 2, torch.where(v < 4, v + 2, v * 0.5 + 4)).to(torch.uint8).add_(sign)
    code = code.view(rows, cols // 2, 2)
    return (code[..., 0] | (code[..., 1] << 4)).contiguous(), (e + 127).to(torch.uint8).view(rows, cols // 32)


def _expert_parts(c, seed, layer, expert):
    g, H, I = _gen(seed, 1, layer, expert), c["hidden"], c["inter"]
    return [t for r, k in ((I, H), (I, H), (H, I)) for t in _mxfp4(g, r, k)]


def _expert_block(c, seed, layer, expert):
    """One packed block: gate weights and scales, up, down."""
    return torch.cat([p.reshape(-1) for p in _expert_parts(c, seed, layer, expert)])


SHARED = 1 << 20  # the shared expert's index among the experts' seeds


def _moe_layer(c, seed, layer):
    """The tensors of one MoE layer but its routed experts."""
    g, H, I, E = _gen(seed, 2, layer), c["hidden"], c["inter"], c["experts"]
    popular = torch.randperm(E, generator=g, device=DEV).add_(1).float().pow_(-1.1).mul_(0.25)
    w = dict(router=_bf16(g, E, H, std=0.02), bias=_randn(g, E, std=0.01) + popular, ln=_norm_weight(g, H))
    if c["shared"] == "bf16":
        w.update(gate=_bf16(g, I, H, std=H ** -0.5), up=_bf16(g, I, H, std=H ** -0.5), down=_bf16(g, H, I, std=I ** -0.5))
    return w


def _norm(x, w, eps):
    x = x.double()
    return w.double() * x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _choice(c, w, hidden):
    xn = _norm(hidden, w["ln"], EPS)
    score = torch.sigmoid(xn @ w["router"].double().T)
    return xn, score, score + w["bias"].double()


def _hidden(c, w, seed):
    """Hidden states [tokens, H]. A token whose last chosen and first rejected
    expert score alike to rounding is drawn again: either choice is right."""
    g = _gen(seed, 3)
    h = _randn(g, c["tokens"], c["hidden"])
    for _ in range(20):
        top = _choice(c, w, h)[2].topk(c["topk"] + 1).values
        near = (top[:, -2] - top[:, -1] < 1e-5).nonzero()[:, 0]
        if not len(near):
            break
        h[near] = _randn(g, len(near), c["hidden"])
    return h


def _dense_layer(c, seed):
    g, H, I = _gen(seed, 4), c["hidden"], c["inter"]
    return dict(ln=_norm_weight(g, H), gate=_bf16(g, I, H, std=H ** -0.5), up=_bf16(g, I, H, std=H ** -0.5),
                down=_bf16(g, H, I, std=I ** -0.5))


def _attention_layer(c, seed, layer):
    g, H, HN, Q, L = _gen(seed, 5, layer), c["hidden"], c["n_heads"], c["q_lora_rank"], c["kv_lora_rank"]
    NP, RP, VD, IH, ID = c["qk_nope"], c["qk_rope"], c["v_head"], c["index_n_heads"], c["index_head_dim"]
    w = dict(input_ln=_norm_weight(g, H), q_a_proj=_bf16(g, Q, H, std=H ** -0.5), q_a_ln=_norm_weight(g, Q),
             q_b_proj=_bf16(g, HN * (NP + RP), Q, std=Q ** -0.5), kv_a_proj=_bf16(g, L + RP, H, std=H ** -0.5),
             kv_a_ln=_norm_weight(g, L), kv_b_proj=_bf16(g, HN * (NP + VD), L, std=L ** -0.5),
             o_proj=_bf16(g, H, HN * VD, std=0.5 * (HN * VD) ** -0.5))
    if layer == 0:
        w.update(idx_wq_b=_bf16(g, IH * ID, Q, std=Q ** -0.5), idx_wk=_bf16(g, ID, H, std=H ** -0.5),
                 idx_k_norm_w=_norm_weight(g, ID), idx_k_norm_b=_bf16(g, ID, std=0.1),
                 idx_weights_proj=_randn(g, IH, H, std=H ** -0.5))
    return w


def _attention_rows(c, seed, layer):
    """The hidden states that filled a layer's cache; the last row is the new position's."""
    return _randn(_gen(seed, 6, layer), c["keys"], c["hidden"])


class _State:
    """What a program holds: the context, the tensors it was given, and the buffers of a call."""

    def __init__(self, case):
        self.case = case
        self.keep = []

    def own(self, *tensors):
        self.keep.extend(tensors)
        return [t.data_ptr() for t in tensors]


def _stream():
    return torch.cuda.current_stream().cuda_stream


def prepare(case, seed):
    s, c = _State(case), case
    if c["kind"] == "expert":
        s.ctx = moe.Context(moe.make_config(hidden=c["hidden"], moe_inter=c["inter"], n_routed_experts=16,
                                            n_experts_per_tok=1))
        s.block = _expert_block(c, seed, 0, 0)
        s.x = _randn(_gen(seed, 3), c["hidden"])
        s.y = torch.empty_like(s.x)
    elif c["kind"] == "moe":
        H, I, E, L = c["hidden"], c["inter"], c["experts"], c["layers"]
        cfg = moe.make_config(hidden=H, moe_inter=I, n_routed_experts=E, n_experts_per_tok=c["topk"], n_layers=L,
                              routed_scaling=SCALING, rms_eps=EPS)
        s.ctx = moe.Context(cfg)
        s.ctx.set_taps(False)  # as a serving loop runs it: the shared expert's test output off
        pool = torch.empty(L * E, moe.native_block_bytes(cfg), dtype=torch.uint8, device=DEV)
        s.own(pool)
        for layer in range(L):
            for e in range(E):
                block = _expert_block(c, seed, layer, e)
                moe.expert_to_native(cfg, block.data_ptr(), pool[layer * E + e].data_ptr(), _stream())
                s.ctx.slot_bind(layer, e, pool[layer * E + e].data_ptr())
            w = _moe_layer(c, seed, layer)
            if c["shared"] == "bf16":
                shared = torch.cat([w[k].reshape(-1) for k in ("gate", "up", "down")])
            else:
                shared = _expert_block(c, seed, layer, SHARED)
            s.ctx.set_layer(layer, *s.own(w["router"], w["bias"], w["ln"]), shared.data_ptr(),
                            moe.SHARED_BF16 if c["shared"] == "bf16" else moe.SHARED_MXFP4)
            if layer == 0:
                s.x = _hidden(c, w, seed)
        s.y, s.tmp = torch.empty_like(s.x), torch.empty_like(s.x)
    elif c["kind"] == "dense":
        s.ctx = moe.Context(moe.make_config(hidden=c["hidden"], moe_inter=1024, n_routed_experts=16,
                                            n_experts_per_tok=1, rms_eps=EPS))
        w = _dense_layer(c, seed)
        s.ctx.set_layer_dense(0, *s.own(w["ln"], w["gate"], w["up"], w["down"]), c["inter"])
        s.x = _randn(_gen(seed, 3), c["tokens"], c["hidden"])
        s.y = torch.empty_like(s.x)
    else:
        a = {k: c[k] for k in GLM_ATTN}
        s.attn = moe.Attention(moe.make_attn_config(n_layers=c["layers"], max_seq=c["keys"], rms_eps=EPS,
                                                    rope_theta=ROPE_THETA, dense_inter=DENSE_INTER, **a))
        rows = []
        for layer in range(c["layers"]):
            w = _attention_layer(c, seed, layer)
            s.own(*w.values())
            s.attn.set_layer(layer, {k: t.data_ptr() for k, t in w.items()})
            rows.append(_attention_rows(c, seed, layer))
        s.x, s.y = rows[0][-1].clone(), torch.empty(c["hidden"], device=DEV)
        for pos in range(c["keys"] - 1):  # the context so far (its rows are overwritten, and not used again)
            for layer in range(c["layers"]):
                s.attn.run_attention(layer, pos, rows[layer][pos].data_ptr(), _stream())
        torch.cuda.synchronize()
    torch.cuda.synchronize()
    return s


def run(s):
    c, st = s.case, _stream()
    x, y = s.x.data_ptr(), s.y.data_ptr()
    if c["kind"] == "expert":
        s.ctx.expert_ffn(s.block.data_ptr(), x, y, None, st)
    elif c["kind"] == "attention":
        s.y.copy_(s.x)  # the position's embedding becomes the residual stream, updated in place
        for layer in range(c["layers"]):
            s.attn.run_attention(layer, c["keys"] - 1, y, st)
    elif c.get("layers", 1) > 1:
        s.y.copy_(s.x)
        s.ctx.run_chain(0, c["layers"], y, s.tmp.data_ptr(), st)
    elif c["tokens"] == 1:
        s.ctx.run_moe_residual(0, x, x, y, st)
    else:
        s.ctx.run_moe_batched(0, c["tokens"], x, x, y, st)
    return s.y


# ---- what a pass cannot do without -------------------------------------------
def _routed(c):
    """Expected number of distinct experts that `tokens` tokens choose, were the choice even."""
    return c["experts"] * (1.0 - (1.0 - c["topk"] / c["experts"]) ** c["tokens"])


def work(case):
    c = case
    H = c["hidden"]
    if c["kind"] == "expert":
        n = 3 * H * c["inter"]
        return {"bytes": n * 17 // 32 + 8 * H, "flops": 2 * n}
    if c["kind"] == "moe":
        n, T = 3 * H * c["inter"], c["tokens"]
        shared = 2 * n if c["shared"] == "bf16" else n * 17 // 32
        nbytes = int(_routed(c) * n * 17 / 32) + shared + c["experts"] * (2 * H + 4) + 2 * H + 8 * H * T
        flops = 2 * T * (n * (c["topk"] + 1) + c["experts"] * H)
        return {"bytes": c["layers"] * nbytes, "flops": c["layers"] * flops}
    if c["kind"] == "dense":
        n, T = 3 * H * c["inter"], c["tokens"]
        return {"bytes": 2 * n + 2 * H + 8 * H * T, "flops": 2 * T * n}
    HN, Q, L, NP, RP, VD = (c[k] for k in ("n_heads", "q_lora_rank", "kv_lora_rank", "qk_nope", "qk_rope", "v_head"))
    IH, ID, T = c["index_n_heads"], c["index_head_dim"], c["keys"]
    kept = min(T, c["index_topk"])
    weights = Q * H + HN * (NP + RP) * Q + (L + RP) * H + HN * (NP + VD) * L + H * HN * VD
    index = IH * ID * Q + ID * H
    nbytes = c["layers"] * (2 * weights + 4 * kept * (L + RP)) + 2 * index + 4 * IH * H + 4 * T * ID + 8 * H
    flops = c["layers"] * 2 * (weights + HN * kept * (2 * L + RP)) + 2 * (index + IH * H + IH * ID * T)
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """Weights in 4 or 16 bits, everything else in 32, sums too. Measured against
    exact(): prefill 2e-7 to 8e-7 (three contractions one after another, the
    longest sums), everything else under 3e-7."""
    return {"rel": 4e-6 if case["kind"] == "moe" and case["tokens"] > 1 else 1.2e-6}


# ---- the same in 64 bits ------------------------------------------------------
def _wide(parts):
    """An MXFP4 matrix's values in 64 bits."""
    w, sc = parts
    m = torch.tensor([0, .5, 1, 1.5, 2, 3, 4, 6], dtype=torch.float64, device=DEV)
    m = torch.cat([m, -m])
    v = torch.stack([m[(w & 15).int()], m[(w >> 4).int()]], -1).view(w.shape[0], -1, 32)
    return torch.ldexp(v, sc.int()[..., None] - 127).view(w.shape[0], -1)


def _ffn(x, gate, up, down):
    g = x @ gate.T
    return (g * torch.sigmoid(g) * (x @ up.T)) @ down.T


def _exact_moe(c, seed):
    h = None
    for layer in range(c["layers"]):
        w = _moe_layer(c, seed, layer)
        if h is None:
            h = _hidden(c, w, seed).double()
        xn, score, choice = _choice(c, w, h)
        idx = choice.topk(c["topk"]).indices
        wt = score.gather(1, idx)
        wt = wt / (wt.sum(1, keepdim=True) + 1e-20) * SCALING
        if c["shared"] == "bf16":
            out = h + _ffn(xn, w["gate"].double(), w["up"].double(), w["down"].double())
        else:
            p = _expert_parts(c, seed, layer, SHARED)
            out = h + _ffn(xn, _wide(p[0:2]), _wide(p[2:4]), _wide(p[4:6]))
        for e in idx.unique().tolist():
            tok, slot = (idx == e).nonzero(as_tuple=True)
            p = _expert_parts(c, seed, layer, e)
            y = _ffn(xn[tok], _wide(p[0:2]), _wide(p[2:4]), _wide(p[4:6]))
            out.index_add_(0, tok, y * wt[tok, slot][:, None])
        h = out
    return h


def _rope(x, pos):
    """Rotates adjacent pairs of the last dimension; the result holds the halves apart."""
    n = x.shape[-1]
    inv = ROPE_THETA ** (-torch.arange(0, n, 2, dtype=torch.float64, device=DEV) / n)
    ang = pos[..., None].double() * inv
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.cat([a * ang.cos() - b * ang.sin(), b * ang.cos() + a * ang.sin()], -1)


def _exact_attention(c, seed):
    HN, L, NP, RP, VD = (c[k] for k in ("n_heads", "kv_lora_rank", "qk_nope", "qk_rope", "v_head"))
    IH, ID, T = c["index_n_heads"], c["index_head_dim"], c["keys"]
    pos = torch.arange(T, device=DEV)
    last = pos[-1:]
    h, sel = _attention_rows(c, seed, 0)[-1].double(), None
    for layer in range(c["layers"]):
        w = {k: v.double() for k, v in _attention_layer(c, seed, layer).items()}
        rows = _attention_rows(c, seed, layer).double()
        rows[-1] = h
        x = _norm(rows, w["input_ln"], EPS)
        ckv = x @ w["kv_a_proj"].T
        kc, kr = _norm(ckv[:, :L], w["kv_a_ln"], LORA_EPS), _rope(ckv[:, L:], pos)
        qr = _norm(x[-1] @ w["q_a_proj"].T, w["q_a_ln"], LORA_EPS)
        if layer == 0:
            k = x @ w["idx_wk"].T
            mu = k.mean(-1, keepdim=True)
            k = (k - mu) / torch.sqrt(((k - mu) ** 2).mean(-1, keepdim=True) + LORA_EPS) * w["idx_k_norm_w"] + w["idx_k_norm_b"]
            k = torch.cat([_rope(k[:, :RP], pos), k[:, RP:]], -1)
            q = (qr @ w["idx_wq_b"].T).view(IH, ID)
            q = torch.cat([_rope(q[:, :RP], last.expand(IH)), q[:, RP:]], -1)
            per_head = (w["idx_weights_proj"] @ x[-1]) * IH ** -0.5
            sel = (per_head[:, None] * torch.relu(q @ k.T * ID ** -0.5)).sum(0).topk(min(T, c["index_topk"])).indices
        q = (qr @ w["q_b_proj"].T).view(HN, NP + RP)
        kvb = w["kv_b_proj"].view(HN, NP + VD, L)
        q_abs = torch.bmm(q[:, None, :NP], kvb[:, :NP].contiguous())[:, 0]
        p = (q_abs @ kc[sel].T + _rope(q[:, NP:], last.expand(HN)) @ kr[sel].T) * (NP + RP) ** -0.5
        ctx = torch.softmax(p, -1) @ kc[sel]
        o = (kvb[:, NP:] * ctx[:, None, :]).sum(-1)
        h = h + w["o_proj"] @ o.reshape(-1)
    return h


def exact(case, seed):
    c = case
    if c["kind"] == "attention":
        return _exact_attention(c, seed)
    if c["kind"] == "moe":
        return _exact_moe(c, seed)
    if c["kind"] == "expert":
        p = _expert_parts(c, seed, 0, 0)
        x = _randn(_gen(seed, 3), c["hidden"]).double()
        return _ffn(x[None], _wide(p[0:2]), _wide(p[2:4]), _wide(p[4:6]))[0]
    w = _dense_layer(c, seed)
    x = _randn(_gen(seed, 3), c["tokens"], c["hidden"])
    return x.double() + _ffn(_norm(x, w["ln"], EPS), w["gate"].double(), w["up"].double(), w["down"].double())
