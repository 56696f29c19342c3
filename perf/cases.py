"""The work a speculative-decoding server has this framework do, as measurable cases.

Every case goes through the package's public entry points on tensors that are already on the
GPU, the way an engine's step calls them: paged attention (verify, decode and prefill chunks),
the KV write, the accept / sample kernels, the KV tier's swap codec, a decoder layer's MLP, and
whole forwards of the target and the draft as a captured graph replays them.  Sizes are those of
the benchmark and the tests (8B target: 32/8 heads of 128, hidden 4096, FFN 14336; 1B draft:
heads of 64, hidden 2048, FFN 8192; vocabulary 128256; 16-token blocks) and, in `draw`, the
ranges around them.

listed() / draw(rng)      cases: dicts of plain values
prepare(case, seed)       inputs, caches, weights and plans a program holds before the call
run(state)                one pass; returns every output and the state it updates
work(case)                bytes and flops the pass cannot do without
tolerance(case)           how far another correct implementation may be off
exact(case, seed)         the outputs in 64 bits, from torch alone
"""
import dataclasses
import math

import numpy as np
import torch

import iitj_llm_coopt_amd as M
from iitj_llm_coopt_amd import fused, spec_engine

DEV = "cuda"
HQ, HKV, BS = 32, 8, 16          # query heads, KV heads, tokens per block, of every model here
MODELS = {"target": spec_engine.TARGET_LLAMA31_8B, "draft": spec_engine.DRAFT_LLAMA32_1B}
WIDTHS = {"target": (4096, 14336), "draft": (2048, 8192)}   # hidden, FFN


def listed():
    return [
        # One user, one token: a short chat decoding without speculation.  The smallest call.
        dict(name="attn_decode_b1", kind="attn", kv="auto", D=128, layout="head", B=1, q=1,
             ragged_q=False, lo=717, hi=717),
        # Verify 5 rows of 32 sequences over 8k-token INT8 contexts (the roofline call).
        dict(name="attn_verify_int8_8k", kind="attn", kv="int8", D=128, layout="head", B=32, q=5,
             ragged_q=False, lo=8192, hi=8192),
        # Verify over a bf16 cache, contexts of 512 to 4096 tokens: an ordinary mixed load.
        dict(name="attn_verify_bf16_ragged", kind="attn", kv="auto", D=128, layout="head", B=32,
             q=5, ragged_q=False, lo=512, hi=4096),
        # Few users with long documents: 4 sequences of 8k to 16k tokens, INT8.
        dict(name="attn_verify_int8_long", kind="attn", kv="int8", D=128, layout="head", B=4, q=5,
             ragged_q=False, lo=8000, hi=16000),
        # An engine step that admits prompts beside running sequences: one whole prompt, one
        # continued chunk and 16 verify items in one batch.
        dict(name="attn_mixed_prefill", kind="mixed", kv="auto", D=128, layout="head", rows1=1500,
             ctx1=0, rows2=500, ctx2=1000, B=16, q=5, lo=300, hi=2100),
        # Acceptance of 4 drafts for 8 sequences, fp32 logits over the whole vocabulary.
        dict(name="accept_b8_fp32", kind="accept", B=8, gamma=4, V=128256, bf16=False, probs=False,
             ragged=False, T=1.0),
        # The draft's proposals: one draw per sequence with its probabilities, bf16 logits.
        dict(name="sample_b32_bf16", kind="sample", N=32, V=128256, bf16=True, T=1.0),
        # A verify step's KV write: 256 sequences append 5 tokens each, quantised on write.
        dict(name="kv_write_int8", kind="kv_write", kv="int8", D=128, layout="head", T=1280,
             blocks=4096),
        # Evict a 4096-token sequence's KV of 32 layers to INT8 and bring it back.
        dict(name="tier_swap_int8", kind="swap", bits=8, D=128, layers=32, tokens=4096),
        # A target layer's norm + MLP at verify rows (32 sequences x 5).
        dict(name="mlp_verify", kind="mlp", model="target", rows=160, packed=False),
        # One draft proposal of 32 sequences: 4 layers and the logits, replayed as a graph.
        dict(name="draft_forward", kind="forward", model="draft", layers=4, B=32, S=1, ctx=1100),
        # One target verify of 32 sequences x 5 rows: 4 layers and the logits, as a graph.
        dict(name="target_forward", kind="forward", model="target", layers=4, B=32, S=5, ctx=1100),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["attn", "attn", "attn", "mixed", "accept", "sample", "kv_write", "swap", "mlp",
                       "forward"])
    kv = rng.choice(["auto", "int8"])
    D = rng.choice([64, 128, 128])
    layout = rng.choice(["head", "head", "token"])
    if kind == "attn":
        B = _log(rng, 1, 64)
        hi = min(_log(rng, 64, 16384), 262144 // B)
        lo = rng.choice([hi, rng.randint(min(16, hi), hi)])
        return dict(kind=kind, kv=kv, D=D, layout=layout, B=B, q=rng.randint(1, 9),
                    ragged_q=rng.random() < 0.3, lo=lo, hi=hi)
    if kind == "mixed":
        return dict(kind=kind, kv=kv, D=D, layout=layout, rows1=_log(rng, 17, 2048), ctx1=0,
                    rows2=_log(rng, 17, 1024), ctx2=rng.randint(1, 2048), B=rng.randint(0, 32),
                    q=rng.randint(1, 5), lo=rng.randint(16, 500), hi=rng.randint(500, 4096))
    if kind == "accept":
        return dict(kind=kind, B=_log(rng, 1, 64), gamma=rng.randint(1, 8),
                    V=rng.choice([32000, 50257, 128256, 151936]), bf16=rng.random() < 0.5,
                    probs=rng.random() < 0.25, ragged=rng.random() < 0.3,
                    T=rng.choice([1.0, 1.0, 0.7]))
    if kind == "sample":
        return dict(kind=kind, N=_log(rng, 1, 128), V=rng.choice([32000, 50257, 128256, 151936]),
                    bf16=rng.random() < 0.5, T=rng.choice([1.0, 1.0, 0.7]))
    if kind == "kv_write":
        return dict(kind=kind, kv=kv, D=D, layout=layout, T=_log(rng, 1, 16384), blocks=4096)
    if kind == "swap":
        return dict(kind=kind, bits=rng.choice([8, 8, 4, 16]), D=D, layers=rng.randint(1, 32),
                    tokens=_log(rng, 16, 4096))
    if kind == "mlp":
        model = rng.choice(["target", "draft"])
        return dict(kind=kind, model=model, rows=_log(rng, 1, 256), packed=model == "draft")
    S = rng.choice([1, 2, 3, 5, 9])
    return dict(kind="forward", model=rng.choice(["target", "draft"]), layers=rng.randint(1, 3),
                B=min(_log(rng, 1, 64), 256 // S), S=S, ctx=_log(rng, 32, 2048))


# ---- inputs (torch alone: prepare() and exact() make the same ones) --------------------------

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _spread(lo, hi, n):
    """n lengths spread evenly over [lo, hi]: the same total for every seed."""
    return [lo + (hi - lo) * (2 * i + 1) // (2 * n) for i in range(n)]


def _shuffled(values, seed):
    order = np.random.default_rng(int(seed)).permutation(len(values))
    return [values[i] for i in order]


def _quantised(x):
    """(codes, fp16 scales) of symmetric absmax INT8 vectors, as an INT8 cache holds them."""
    s = x.abs().amax(-1).clamp_min(1e-8) / 127
    return torch.round(x / s.unsqueeze(-1)).clamp_(-127, 127).to(torch.int8), s.to(torch.float16)


def _pool(g, blocks, D, kv, layout):
    """One layer's caches of `blocks` blocks full of N(0, 1) keys and values (INT8: with 1 % of
    x20 outliers), [blocks, BS, HKV, D] views of head-major or token-major storage."""
    store = (blocks, HKV, BS, D) if layout == "head" else (blocks, BS, HKV, D)
    view = (lambda t: t.transpose(1, 2)) if layout == "head" else (lambda t: t)
    out, scales = [], []
    for _ in range(2):
        if kv == "auto":
            t = torch.empty(store, dtype=torch.bfloat16, device=DEV)
            s = None
        else:
            t = torch.empty(store, dtype=torch.int8, device=DEV)
            s = torch.empty(store[:3], dtype=torch.float16, device=DEV)
        for a in range(0, blocks, 4096):        # in pieces: the fp32 values stay small
            x = torch.randn((min(blocks, a + 4096) - a, *store[1:]), generator=g, device=DEV)
            if kv == "auto":
                t[a:a + 4096] = x.to(torch.bfloat16)
            else:
                x = torch.where(torch.rand(x.shape, generator=g, device=DEV) < 0.01, x * 20, x)
                t[a:a + 4096], s[a:a + 4096] = _quantised(x)
        out.append(view(t))
        scales.append(None if s is None else view(s))
    return out[0], out[1], scales[0], scales[1]


def _items(case, seed):
    """(query rows, keys) of every sequence of an attention case; keys include the new rows."""
    q = case["q"]
    if case["kind"] == "attn":
        rows = [1 + i % q if case["ragged_q"] else q for i in range(case["B"])]
        items = [(n, n + c) for n, c in zip(rows, _spread(case["lo"], case["hi"], case["B"]))]
        return _shuffled(items, seed)
    items = [(case["rows1"], case["rows1"] + case["ctx1"]), (case["rows2"], case["rows2"] + case["ctx2"])]
    return items + _shuffled([(q, q + c) for c in _spread(case["lo"], case["hi"], case["B"])], seed)


def _attn_inputs(case, seed):
    items = _items(case, seed)
    widths = [-(-k // BS) for _, k in items]
    blocks = sum(widths) + 1
    perm = np.random.default_rng(int(seed) + 1).permutation(blocks).astype(np.int32)
    table = np.zeros((len(items), max(widths)), np.int32)
    o = 0
    for b, w in enumerate(widths):
        table[b, :w] = perm[o:o + w]
        o += w
    g = _gen(seed)
    kc, vc, ks, vs = _pool(g, blocks, case["D"], case["kv"], case["layout"])
    T = sum(n for n, _ in items)
    q = torch.randn(T, HQ, case["D"], generator=g, device=DEV).to(torch.bfloat16)
    return items, torch.from_numpy(table).to(DEV), kc, vc, ks, vs, q


def _accept_inputs(case, seed):
    g = _gen(seed)
    B, gm, V = case["B"], case["gamma"], case["V"]
    dt = torch.bfloat16 if case["bf16"] else torch.float32
    tl = torch.randn(B, gm + 1, V, generator=g, device=DEV) * 2
    dl = (tl[:, :gm] + torch.randn(B, gm, V, generator=g, device=DEV) * 0.5).to(dt).contiguous()
    tl = tl.to(dt)
    # draft tokens drawn from the draft's own softmax, as its proposals are
    c = torch.softmax(dl.double() / case["T"], -1).cumsum(-1)
    u = torch.rand(B, gm, 1, generator=g, device=DEV).double()
    tok = torch.searchsorted(c, u * c[..., -1:], right=True).squeeze(-1).clamp_(max=V - 1)
    ua = torch.rand(B, gm, generator=g, device=DEV)
    ur = torch.rand(B, generator=g, device=DEV)
    gam = [i % (gm + 1) for i in range(B)] if case["ragged"] else [gm] * B
    draft = torch.softmax(dl.float() / case["T"], -1) if case["probs"] else dl
    return tl, draft, tok.to(torch.int32), ua, ur, torch.tensor(gam, dtype=torch.int32, device=DEV)


def _sample_inputs(case, seed):
    g = _gen(seed)
    x = torch.randn(case["N"], case["V"], generator=g, device=DEV) * 2
    return (x.to(torch.bfloat16) if case["bf16"] else x), torch.rand(case["N"], generator=g, device=DEV)


def _kv_write_inputs(case, seed):
    g = _gen(seed)
    kv = torch.randn(2, case["T"], HKV, case["D"], generator=g, device=DEV)
    kv = torch.where(torch.rand(kv.shape, generator=g, device=DEV) < 0.01, kv * 20, kv)
    # sequences append 5 tokens each, every one in a block of its own
    n = -(-case["T"] // 5)
    first = torch.randperm(case["blocks"], generator=g, device=DEV)[:n] * BS
    first += torch.randint(0, BS - 4, (n,), generator=g, device=DEV)
    slots = (first[:, None] + torch.arange(5, device=DEV)).reshape(-1)[: case["T"]].contiguous()
    kv = kv.to(torch.bfloat16)
    return kv[0], kv[1], slots


def _swap_inputs(case, seed):
    nb = -(-case["tokens"] // BS)
    g = _gen(seed)
    buf = torch.empty(2 * case["layers"], 2 * nb, HKV, BS, case["D"], dtype=torch.bfloat16, device=DEV)
    for i in range(buf.shape[0]):
        x = torch.randn(buf.shape[1:], generator=g, device=DEV)
        buf[i] = torch.where(torch.rand(x.shape, generator=g, device=DEV) < 0.01, x * 20, x)
    ids = torch.randperm(2 * nb, generator=g, device=DEV)
    return buf, ids[:nb].contiguous(), ids[nb:].contiguous()


def _mlp_inputs(case, seed):
    H, F = WIDTHS[case["model"]]
    g = _gen(seed)

    def w(*size, std=0.02):
        return (torch.randn(*size, generator=g, device=DEV) * std).to(torch.bfloat16)

    return dict(gate_up=w(2 * F, H), down=w(H, F), o=w(case["rows"], H, std=1.0),
                x=w(case["rows"], H, std=1.0), ln1=1 + w(H, std=0.1), ln2=1 + w(H, std=0.1))


def _forward_shape(case):
    return dataclasses.replace(MODELS[case["model"]], layers=case["layers"])


def _forward_inputs(case, seed):
    """Token ids of the step's rows and every layer's cached keys and values [2, B, ctx, HKV, D]
    (draft: bf16; target: INT8 codes and scales)."""
    s = _forward_shape(case)
    g = _gen(int(seed) + 7)
    ids = torch.randint(0, s.vocab, (case["B"] * case["S"],), generator=g, device=DEV)
    layers = []
    for _ in range(s.layers):
        x = torch.randn(2, case["B"], case["ctx"], HKV, s.head_dim, generator=g, device=DEV)
        layers.append(_quantised(x) if case["model"] == "target" else (x.to(torch.bfloat16), None))
    return s, ids, layers


# ---- states -------------------------------------------------------------------------------------

def prepare(case, seed):
    st = dict(case=case)
    kind = case["kind"]
    if kind in ("attn", "mixed"):
        items, st["table"], st["k"], st["v"], st["ks"], st["vs"], st["q"] = _attn_inputs(case, seed)
        rows = np.array([n for n, _ in items])
        st["cu"] = torch.from_numpy(np.concatenate([[0], rows.cumsum()]).astype(np.int32)).to(DEV)
        st["lens"] = torch.tensor([k for _, k in items], dtype=torch.int32, device=DEV)
        st["max_q"], st["max_k"] = int(rows.max()), max(k for _, k in items)
    elif kind == "accept":
        st["args"] = _accept_inputs(case, seed)
    elif kind == "sample":
        st["x"], st["u"] = _sample_inputs(case, seed)
    elif kind == "kv_write":
        st["k"], st["v"], st["slots"] = _kv_write_inputs(case, seed)
        if case["layout"] == "head":
            st["caches"] = M.allocate_kv_cache(case["blocks"], BS, HKV, case["D"], case["kv"], device=DEV)
        else:
            shape = (case["blocks"], BS, HKV, case["D"])
            dt = torch.bfloat16 if case["kv"] == "auto" else torch.int8
            sc = [torch.zeros(shape[:3], dtype=torch.float16, device=DEV) if case["kv"] == "int8" else None
                  for _ in range(2)]
            st["caches"] = (torch.zeros(shape, dtype=dt, device=DEV), torch.zeros(shape, dtype=dt, device=DEV), *sc)
    elif kind == "swap":
        st["buf"], st["out_ids"], st["in_ids"] = _swap_inputs(case, seed)
        st["caches"] = [t.transpose(1, 2) for t in st["buf"]]
    elif kind == "mlp":
        st.update(_mlp_inputs(case, seed))
        if case["packed"]:
            st["gate_up"] = fused.pack_gate_up_weight(st["gate_up"])
        st["down"] = fused.pack_linear_weight(st["down"])
        st["res"] = torch.empty_like(st["x"])
    else:
        _prepare_forward(st, case, seed)
    return st


def _prepare_forward(st, case, seed):
    s, ids, layers = _forward_inputs(case, seed)
    B, S, ctx = case["B"], case["S"], case["ctx"]
    draft = case["model"] == "draft"
    model = spec_engine.RandomLlama(s, DEV, seed=int(seed), max_pos=4096,
                                    packed=("qkv", "o", "gate_up", "down", "lm_head") if draft else None)
    kv = spec_engine.PagedKV(s, B, ctx + S, "auto" if draft else "int8", DEV, BS, int(seed))
    t = torch.arange(ctx, device=DEV)
    blk, off = kv.block_table[:, t // BS].long(), (t % BS).expand(B, ctx)
    for (kc, vc, ks, vs), (x, sc) in zip(kv.layers, layers):
        kc[blk, off], vc[blk, off] = x[0], x[1]
        if sc is not None:
            ks[blk, off], vs[blk, off] = sc[0], sc[1]
    ops = spec_engine.HipOps(DEV)
    start = torch.full((B,), ctx, dtype=torch.int64, device=DEV)
    n_real = torch.full((B,), S, dtype=torch.int64, device=DEV)
    cu = torch.arange(B + 1, dtype=torch.int32, device=DEV) * S
    logits = torch.empty(B * S, s.vocab, dtype=torch.bfloat16, device=DEV)

    @torch.inference_mode()
    def step():
        pos, slots, lens = ops.row_slots(kv, start, S, n_real)
        return model.forward(ops, kv, ids, pos.reshape(-1), slots, (cu, lens, S, ctx + S),
                             logits_out=logits)

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step()
    st.update(model=model, kv=kv, ops=ops, graph=graph, logits=logits, keep=(ids, start, n_real, cu))


# ---- one pass -----------------------------------------------------------------------------------

def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind in ("attn", "mixed"):
        return M.flash_attn_varlen_func(
            q=st["q"], k=st["k"], v=st["v"], cu_seqlens_q=st["cu"], max_seqlen_q=st["max_q"],
            seqused_k=st["lens"], max_seqlen_k=st["max_k"], causal=True, block_table=st["table"],
            k_scale=st["ks"], v_scale=st["vs"])
    if kind == "accept":
        tl, draft, tok, ua, ur, gam = st["args"]
        r = M.accept(tl, draft, tok, case["T"], ua, ur, draft_is_probs=case["probs"],
                     gamma_per_seq=gam if case["ragged"] else None)
        return r.accepted_len, r.tokens, r.margin
    if kind == "sample":
        return M.sample(st["x"], case["T"], uniforms=st["u"])
    if kind == "kv_write":
        kc, vc, ks, vs = st["caches"]
        M.reshape_and_cache_flash(st["k"], st["v"], kc, vc, st["slots"], case["kv"], ks, vs)
        return st["caches"]
    if kind == "swap":
        q, s = M.swap_out_caches(st["caches"], st["out_ids"], case["bits"])
        M.swap_in_caches(q, s, case["bits"], st["in_ids"], st["caches"])
        return q, s, st["buf"]
    if kind == "mlp":
        res = st["res"].copy_(st["x"])       # the residual stream, updated in place below
        h = fused.rms_norm(st["o"], st["ln1"], 1e-5, residual=res)
        d = fused.linear(fused.linear_silu(h, st["gate_up"]), st["down"], defer_reduce=True)
        return fused.rms_norm(d, st["ln2"], 1e-5, residual=res), res
    st["graph"].replay()
    return st["logits"], st["kv"].layers


# ---- what a pass cannot do without --------------------------------------------------------------

def _kv_token_bytes(kv, D):
    return HKV * (4 * D if kv == "auto" else 2 * D + 4)


def work(case):
    kind = case["kind"]
    if kind in ("attn", "mixed"):
        items, D = _items(case, 0), case["D"]
        nbytes = sum(k for _, k in items) * _kv_token_bytes(case["kv"], D)
        nbytes += 2 * sum(n for n, _ in items) * HQ * D * 2
        pairs = sum(n * k - n * (n - 1) // 2 for n, k in items)   # (row, visible key)
        return dict(bytes=nbytes, flops=4 * pairs * HQ * D)
    if kind == "accept":
        rows = sum(2 * (i % (case["gamma"] + 1) if case["ragged"] else case["gamma"]) + 1
                   for i in range(case["B"]))
        drafts = (rows - case["B"]) // 2
        elt = 2 if case["bf16"] else 4
        return dict(bytes=case["V"] * ((rows - drafts) * elt + drafts * (4 if case["probs"] else elt)),
                    flops=0)
    if kind == "sample":
        return dict(bytes=case["N"] * case["V"] * ((2 if case["bf16"] else 4) + 4), flops=0)
    if kind == "kv_write":
        return dict(bytes=case["T"] * (HKV * case["D"] * 4 + _kv_token_bytes(case["kv"], case["D"]) + 8),
                    flops=0)
    if kind == "swap":
        vecs = 2 * case["layers"] * -(-case["tokens"] // BS) * BS * HKV
        D = case["D"]
        packed = {16: 2 * D, 8: D + 2, 4: D // 2 + 2}[case["bits"]]
        return dict(bytes=2 * vecs * (2 * D + packed), flops=0)
    if kind == "mlp":
        H, F = WIDTHS[case["model"]]
        return dict(bytes=3 * H * F * 2 + 4 * case["rows"] * H * 2, flops=6 * case["rows"] * H * F)
    s = _forward_shape(case)
    T, D = case["B"] * case["S"], s.head_dim
    per_layer = (HQ + 2 * HKV) * D * s.hidden + HQ * D * s.hidden + 3 * s.ffn * s.hidden
    weights = s.layers * per_layer + s.vocab * s.hidden
    kv = s.layers * case["B"] * (case["ctx"] + case["S"]) * \
        _kv_token_bytes("auto" if case["model"] == "draft" else "int8", D)
    attn = s.layers * 4 * T * (case["ctx"] + case["S"]) * HQ * D
    return dict(bytes=2 * weights + kv + 2 * T * s.vocab, flops=2 * T * weights + attn)


def tolerance(case):
    return {
        # bf16 outputs; probabilities enter the second product in 16 bits
        "attn": dict(rel=1e-2, max=0.1), "mixed": dict(rel=1e-2, max=0.1),
        # tokens and lengths equal but for ties; margin is a distance of the size of one
        # token's probability, formed from 32-bit probabilities
        "accept": dict(rel=1e-3, max=0.04, differ=0.01),
        "sample": dict(rel=1e-5, max=1e-4, differ=0.01),
        "kv_write": "exact", "swap": "exact",
        "mlp": dict(rel=1e-2, max=0.1),
        # every layer's bf16 roundings travel on; the INT8 codes of the new rows may differ by one
        "forward": dict(rel=3e-2, max=0.3, differ=0.01),
    }[case["kind"]]


# ---- 64-bit results -----------------------------------------------------------------------------

def _attend(q, k, v, scale):
    """q [n, Hq, D], k / v [L, Hkv, D], causal aligned at the end; one KV head at a time."""
    n, L = q.shape[0], k.shape[0]
    G = q.shape[1] // k.shape[1]
    hidden = torch.arange(L, device=DEV)[None, :] > (L - n + torch.arange(n, device=DEV))[:, None]
    out = torch.empty_like(q)
    for h in range(k.shape[1]):
        qh = q[:, h * G:(h + 1) * G].transpose(0, 1).reshape(G * n, -1)
        s = (qh @ k[:, h].t().contiguous()) * scale
        s.masked_fill_(hidden.repeat(G, 1), float("-inf"))
        out[:, h * G:(h + 1) * G] = (torch.softmax(s, -1) @ v[:, h].contiguous()).view(G, n, -1).transpose(0, 1)
    return out


def _values(codes, scales):
    """What an INT8 cache stands for: bf16(code * scale), in 64 bits."""
    return (codes.float() * scales.float().unsqueeze(-1)).to(torch.bfloat16).double()


def _rows_exact(x):
    x = x.double()
    e = torch.exp(x - x.amax(-1, keepdim=True))
    return e / e.sum(-1, keepdim=True)


def _margin_exact(case, seed):
    """The distance of each sequence's deciding uniforms to their boundaries."""
    tl, draft, tok, ua, ur, gam = _accept_inputs(case, seed)
    out = torch.empty(case["B"], dtype=torch.float64, device=DEV)
    for b in range(case["B"]):
        g = int(gam[b])
        p = _rows_exact(tl[b].double() / case["T"])
        q = draft[b].double() if case["probs"] else _rows_exact(draft[b].double() / case["T"])
        k, near = g, 1.0
        for i in range(g):
            t, u = int(tok[b, i]), float(ua[b, i])
            ratio = min(1.0, float(p[i, t] / q[i, t]))
            near = min(near, abs(u - ratio))
            if u >= ratio:
                k = i
                break
        c = (p[g] if k == g else (p[k] - q[k]).clamp_min(0)).cumsum(0)
        tau = ur[b].double() * c[-1]
        j = int(torch.searchsorted(c, tau.reshape(1), right=True).clamp(max=case["V"] - 1))
        below = c[j - 1] if j else torch.zeros_like(tau)
        out[b] = min(near, float(torch.minimum(tau - below, c[j] - tau) / c[-1]))
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind in ("attn", "mixed"):
        items, table, kc, vc, ks, vs, q = _attn_inputs(case, seed)
        out, o = torch.empty(q.shape, dtype=torch.float64, device=DEV), 0
        for b, (n, L) in enumerate(items):
            t = torch.arange(L, device=DEV)
            at = (table[b, t // BS].long(), t % BS)
            k, v = (c[at].double() if s is None else _values(c[at], s[at]) for c, s in ((kc, ks), (vc, vs)))
            out[o:o + n] = _attend(q[o:o + n].double(), k, v, case["D"] ** -0.5)
            o += n
        return out
    if kind == "accept":
        return None, None, _margin_exact(case, seed)
    if kind == "sample":
        x, _ = _sample_inputs(case, seed)
        return None, _rows_exact(x.double() / case["T"])
    if kind == "kv_write":
        k, v, slots = _kv_write_inputs(case, seed)
        out, shape = [], (case["blocks"] * BS, HKV, case["D"])
        real = slots >= 0
        for x in (k, v):
            c = torch.zeros(shape, dtype=torch.float64, device=DEV)
            c[slots[real]] = x[real].double()
            out.append(c)
        if case["kv"] == "auto":
            return [c.view(case["blocks"], BS, HKV, -1) for c in out] + [None, None]
        return [None, None] + [(c.abs().amax(-1) / 127).view(case["blocks"], BS, HKV) for c in out]
    if kind == "swap":
        if case["bits"] == 16:
            return None
        buf, out_ids, _ = _swap_inputs(case, seed)
        x = buf.transpose(2, 3)[:, out_ids].double()
        return None, x.abs().amax(-1) / (127 if case["bits"] == 8 else 7), None
    if kind == "mlp":
        w = {k: t.double() for k, t in _mlp_inputs(case, seed).items()}
        F = w["down"].shape[1]
        r = w["x"] + w["o"]
        h = _norm(r, w["ln1"]) @ w["gate_up"].t()
        r = r + (torch.nn.functional.silu(h[:, :F]) * h[:, F:]) @ w["down"].t()
        return _norm(r, w["ln2"]), r
    return _exact_forward(case, seed), [[None] * 4] * case["layers"]


def _norm(x, w, eps=1e-5):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w


def _exact_forward(case, seed):
    s, ids, cached = _forward_inputs(case, seed)
    B, S, ctx, D = case["B"], case["S"], case["ctx"], s.head_dim
    g = _gen(seed)

    def w(*size):       # the random weights in the order a RandomLlama draws them
        return (torch.randn(*size, generator=g, device=DEV) * 0.02).to(torch.bfloat16).double()

    embed = w(s.vocab, s.hidden)
    head = embed if s.tie_embeddings else w(s.vocab, s.hidden)
    x = embed[ids]
    del embed
    inv = 1.0 / (s.rope_theta ** (torch.arange(0, D, 2, dtype=torch.float32) / D))
    ang = torch.outer(torch.arange(ctx, ctx + S, dtype=torch.float32), inv)
    cos, sin = (t.to(DEV, torch.bfloat16).double().repeat(B, 1)[:, None, :] for t in (ang.cos(), ang.sin()))

    def rope(t):
        a, b = t[..., : D // 2], t[..., D // 2:]
        return torch.cat((a * cos - b * sin, b * cos + a * sin), -1)

    one = torch.ones(s.hidden, dtype=torch.float64, device=DEV)
    for kv, sc in cached:
        qkv_w, o_w = w((HQ + 2 * HKV) * D, s.hidden), w(s.hidden, HQ * D)
        gu_w, down_w = w(2 * s.ffn, s.hidden), w(s.hidden, s.ffn)
        q, k, v = (_norm(x, one) @ qkv_w.t()).split([HQ * D, HKV * D, HKV * D], -1)
        q, k, v = rope(q.view(B * S, HQ, D)), rope(k.view(B * S, HKV, D)), v.view(B * S, HKV, D)
        old = kv.double() if sc is None else _values(kv, sc)
        a = torch.cat([_attend(q[b * S:(b + 1) * S], torch.cat((old[0, b], k[b * S:(b + 1) * S])),
                               torch.cat((old[1, b], v[b * S:(b + 1) * S])), D ** -0.5) for b in range(B)])
        x = x + a.reshape(B * S, -1) @ o_w.t()
        h = _norm(x, one) @ gu_w.t()
        x = x + (torch.nn.functional.silu(h[:, : s.ffn]) * h[:, s.ffn:]) @ down_w.t()
    return _norm(x, one) @ head.t()
