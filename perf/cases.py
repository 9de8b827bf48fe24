"""The work a program asks of this framework, as cases to be timed and compared.

Every case is one call (or one call and a read of its result) through the public binding,
``ane-training_amd/stories_lm.py``: a decode step, a short greedy run, a prompt, a scored
batch, all the logits of a prompt, or the classifier GEMM on the caller's device buffers.
Sizes come from this repository's models (Stories-110M, the scaled 2048-wide model, the
grouped-query shapes of the tests), with layer stacks cut to a few layers where the whole
model would only repeat them, and a small vocabulary where the layers are what is meant.

Weights are seeded N(0, 0.02) in fp16, norm gains 1 + N(0, 0.1); tokens are uniform.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "ane-training_amd"))
import stories_lm as S  # noqa: E402

# Model shapes of the repository: configurations, benchmark and tests.
STORIES = dict(dim=768, hidden=2048, heads=12, kv_heads=12, layers=12)
SCALED = dict(dim=2048, hidden=5632, heads=16, kv_heads=16, layers=4)
SCALED_GQA = dict(dim=2048, hidden=5632, heads=16, kv_heads=8, layers=4)
GQA_1024 = dict(dim=1024, hidden=1024, heads=16, kv_heads=8, layers=8)
SMALL_GQA = dict(dim=256, hidden=512, heads=4, kv_heads=2, layers=2)


# ---- the cases ------------------------------------------------------------------

def listed():
    return [
        # One token of an interactive session near its start: the smallest call, all latency.
        dict(name="token", kind="step", **STORIES, vocab=32000, batch=1, ctx=40, kv32=False),
        # A short greedy continuation on the device, fp32 cache (the headline path).
        dict(name="greedy", kind="greedy", **STORIES, vocab=32000, batch=1, ctx=100, steps=17, kv32=True),
        # One token of a long session: attention over a deep cache.
        dict(name="token_long", kind="step", **STORIES, vocab=32000, batch=1, ctx=1900, kv32=False),
        # A few sequences of one user, fp32 cache, ragged positions.
        dict(name="batch_3", kind="step", **STORIES, vocab=32000, batch=3, ctx=333, kv32=True),
        # A lightly loaded server, grouped-query model, ragged longer contexts.
        dict(name="batch_12", kind="step", **GQA_1024, vocab=1000, batch=12, ctx=777, kv32=False),
        # A fully loaded server: 64 sequences after 192-token prompts, the layers.
        dict(name="batch_64", kind="step", **STORIES, vocab=512, batch=64, ctx=255, kv32=False),
        # The layers of the scaled model for 32 sequences of 512-640 positions.
        dict(name="scaled_32", kind="step", **SCALED, vocab=512, batch=32, ctx=639, kv32=False),
        # A short prompt: first token latency.
        dict(name="prompt_41", kind="last", **STORIES, vocab=32000, nseq=1, seq=41, kv32=False),
        # One 256-token window with every logit on the host.
        dict(name="logits_256", kind="logits", **STORIES, vocab=32000, nseq=1, seq=256, kv32=False),
        # A long prompt through layers of the scaled model with grouped queries.
        dict(name="prompt_1900", kind="last", **SCALED_GQA, vocab=32000, nseq=1, seq=1900, kv32=False),
        # The training-shape forward with its loss: 8 sequences of 256 tokens.
        dict(name="score_8x256", kind="score", **STORIES, vocab=32000, nseq=8, seq=256, kv32=False),
        # The head alone: classifier GEMM and greedy pick on the caller's device buffers.
        dict(name="head_48", kind="head", rows=48, cols=32000, width=768),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "step", "step", "greedy", "last", "last", "score", "logits", "head"])
    if kind == "head":
        k = rng.choice([256, 512, 768, 1024, 2048])
        m = _log_int(rng, 1, 64)
        n = rng.choice([32000, _log_int(rng, 500, 32000)])
        return dict(kind=kind, rows=m, cols=n, width=k)
    shape = rng.choice([STORIES, STORIES, SCALED, SCALED_GQA, GQA_1024, SMALL_GQA])
    kv32 = rng.random() < 0.25
    if kind == "step":
        batch = _log_int(rng, 1, 64)
        ctx = min(_log_int(rng, 8, 2047), 20480 // batch)
        vocab = rng.choice([500, 1000, 32000]) if batch <= 8 else rng.choice([500, 1000])
        return dict(kind=kind, **shape, vocab=vocab, batch=batch, ctx=ctx, kv32=kv32)
    if kind == "greedy":
        return dict(kind=kind, **shape, vocab=rng.choice([1000, 32000]), batch=1,
                    ctx=_log_int(rng, 4, 400), steps=rng.choice([5, 17, 17, 33]), kv32=True)
    # prompts: whole sequences of one length, up to about 2000 rows
    seq = _log_int(rng, 5, 256 if kind == "logits" else 1900)
    nseq = 1 if kind == "logits" else max(1, min(_log_int(rng, 1, 32), 1900 // seq))
    vocab = rng.choice([1000, 32000])
    return dict(kind=kind, **shape, vocab=vocab, nseq=nseq, seq=seq, kv32=kv32)


# ---- inputs ------------------------------------------------------------------------

def _sizes(c):
    """Element counts of the weight tensors in llama2.c order, the classifier last."""
    D, F, L, V = c["dim"], c["hidden"], c["layers"], c["vocab"]
    nkv = c["kv_heads"] * (D // c["heads"])
    return [V * D, L * D, L * D * D, L * nkv * D, L * nkv * D, L * D * D, L * D, L * F * D, L * D * F,
            L * F * D, D, V * D]


def _weights(c, seed):
    """All weights, fp16, one flat tensor on the device."""
    g = torch.Generator(device="cuda").manual_seed(1000003 * (int(seed) % 1000003) + 17)
    sz = _sizes(c)
    w = torch.empty(sum(sz), dtype=torch.float16, device="cuda").normal_(0.0, 0.02, generator=g)
    at = np.concatenate([[0], np.cumsum(sz)])
    for t in (1, 6, 10):   # norm gains
        w[at[t]:at[t + 1]] = 1.0 + 0.1 * torch.randn(sz[t], generator=g, device="cuda")
    return w, at


def _positions(c):
    """Ragged positions of a batch's rows: the last at ctx, the others up to a third less."""
    b = np.arange(c["batch"])
    return (c["ctx"] - (b * 37) % (c["ctx"] // 3 + 1)).astype(np.int32)


def _tokens(c, seed, rows, length):
    return np.random.default_rng(int(seed) + 5).integers(0, c["vocab"], (rows, length)).astype(np.int32)


def _model(c, seed, max_batch, max_seq):
    w, _ = _weights(c, seed)
    host = w.cpu().numpy().view(np.uint16)
    cfg = S.make_config(c["dim"], c["hidden"], c["layers"], c["heads"], c["kv_heads"], c["vocab"], max_seq)
    m = S.Model.create(cfg, host, True, max_batch, max_seq)
    if c["kv32"]:
        m.set_option(S.LM_OPT_KV_F32, 1)
    return m


def prepare(case, seed):
    c = case
    if S.init() != 0:
        raise RuntimeError("no gfx950 device")
    if c["kind"] == "head":
        g = torch.Generator(device="cuda").manual_seed(int(seed) + 3)
        M, N, K = c["rows"], c["cols"], c["width"]
        return dict(c=c, a=torch.empty(M, K, dtype=torch.float16, device="cuda").normal_(0, 1, generator=g),
                    w=torch.empty(N, K, dtype=torch.float16, device="cuda").normal_(0, 0.02, generator=g),
                    out=torch.empty(M, N, dtype=torch.float32, device="cuda"),
                    ids=torch.empty(M, dtype=torch.int32, device="cuda"))
    if c["kind"] in ("step", "greedy"):
        steps = c.get("steps", 1)
        toks = _tokens(c, seed, c["batch"], c["ctx"] + 1)
        m = _model(c, seed, c["batch"], max(256, c["ctx"] + steps + 1))
        # what lies behind the step, in the cache: a session's first window goes through
        # the decode chain, as the generation session does it; a server's prompts as prompts
        if c["kind"] == "greedy":
            for p in range(c["ctx"]):
                m.forward(int(toks[0, p]), p)
        else:
            m.prefill_batch(toks[:, :c["ctx"]], mode=S.LM_LOGITS_LAST, want_logits=False)
        pos = _positions(c)
        return dict(c=c, m=m, pos=pos, tok=toks[np.arange(c["batch"]), pos].copy())
    m = _model(c, seed, c["nseq"], max(256, c["seq"]))
    return dict(c=c, m=m, toks=_tokens(c, seed, c["nseq"], c["seq"]))


# ---- one pass -----------------------------------------------------------------------

def run(state):
    c = state["c"]
    kind = c["kind"]
    if kind == "head":
        rc = S.gemm_argmax_noalloc(c["rows"], c["cols"], c["width"], state["a"].data_ptr(),
                                   state["w"].data_ptr(), state["out"].data_ptr(), state["ids"].data_ptr(),
                                   torch.cuda.current_stream().cuda_stream)
        if rc:
            raise S.LMError(rc, "gemm_argmax_noalloc")
        return state["out"], state["ids"]
    m = state["m"]
    if kind == "step":
        if c["batch"] == 1:
            return m.forward(int(state["tok"][0]), int(state["pos"][0]))
        return m.forward_batch(state["tok"], state["pos"])[0]
    if kind == "greedy":
        ids = m.generate_greedy(state["tok"], state["pos"], c["steps"])
        return ids, m.read_logits(0, c["batch"])
    if kind == "last":
        return m.prefill_batch(state["toks"], mode=S.LM_LOGITS_LAST)
    if kind == "logits":
        return m.prefill(state["toks"][0])
    return m.prefill_loss(state["toks"])[0]


# ---- what one pass cannot do without -------------------------------------------------

def work(case):
    c = case
    if c["kind"] == "head":
        M, N, K = c["rows"], c["cols"], c["width"]
        return {"bytes": 2 * (M * K + N * K) + 4 * M * N + 4 * M, "flops": 2 * M * N * K}
    D, F, L, V = c["dim"], c["hidden"], c["layers"], c["vocab"]
    nkv = c["kv_heads"] * (D // c["heads"])
    per_layer = D * (2 * D + 2 * nkv + 3 * F)   # weights of a layer
    kv = 4 if c["kv32"] else 2
    wbytes = 2 * L * per_layer + 4 * D * (2 * L + 1)
    if c["kind"] in ("step", "greedy"):
        B = c["batch"]
        pos = [int(p) for p in _positions(c)]
        nb = nf = 0
        for t in range(c.get("steps", 1)):
            ctx = sum(p + t + 1 for p in pos)
            nb += wbytes + 2 * V * D + 2 * L * ctx * nkv * kv + 2 * B * D
            nf += 2 * B * (L * per_layer + V * D) + 4 * L * ctx * D
        return {"bytes": nb + 4 * B * V, "flops": nf}
    n, s = c["nseq"], c["seq"]
    rows, pairs = n * s, n * s * (s + 1) / 2
    if c["kind"] == "last":
        # the last layer owes only keys and values to every row, the rest to the last rows
        f = 2 * rows * ((L - 1) * per_layer + 2 * nkv * D) + 4 * (L - 1) * pairs * D
        f += 2 * n * (per_layer - 2 * nkv * D + V * D) + 4 * n * s * D
        out = 4 * n * V
    else:
        f = 2 * rows * (L * per_layer + V * D) + 4 * L * pairs * D
        out = 4 * rows * V if c["kind"] == "logits" else 4 * n
    return {"bytes": wbytes + 2 * V * D + 2 * rows * D + 2 * L * rows * nkv * kv + out, "flops": f}


# Relative errors measured against `exact` (2-norm) and stated at about four times that.
def tolerance(case):
    k = case["kind"]
    if k == "head":     # fp16 operands, fp32 sums of up to 2048 products; ids: near ties only
        return {"rel": 1.2e-6, "max": 1e-5, "differ": 0.03}
    if k == "greedy":   # fp32 activations, sums and cache throughout
        return {"rel": 1e-5, "max": 1e-4, "differ": 0.0}
    if k == "score":    # means of seq - 1 log-probabilities near log V: their errors average out
        n = math.sqrt(case["seq"] - 1)
        return {"rel": 5e-4 / n, "max": 1e-3 / n}
    return {"rel": 5e-3, "max": 2e-2}   # fp16 GEMM operands and cache: up to 1.2e-3 and 5e-3 seen


# ---- the same in 64 bits ---------------------------------------------------------------

def _forward64(c, w, at, toks):
    """Final-norm rows [n, T, D] of the causal forward of toks [n, T], float64 on the device."""
    D, F, L, H, G = c["dim"], c["hidden"], c["layers"], c["heads"], c["kv_heads"]
    hd = D // H
    nkv = G * hd
    n, T = toks.shape

    def ten(t, l, shape):
        size = math.prod(shape)
        return w[at[t] + l * size:at[t] + (l + 1) * size].double().view(shape)

    # the rotation table is defined in fp32 (frequencies and angles)
    freq = torch.tensor([1.0 / np.power(np.float32(10000.0), np.float32(2 * i) / np.float32(hd))
                         for i in range(hd // 2)], dtype=torch.float32, device="cuda")
    ang = (torch.arange(T, dtype=torch.float32, device="cuda")[:, None] * freq).double()
    cos, sin = ang.cos()[None, :, None], ang.sin()[None, :, None]

    def norm(x, gain):
        return x / (x.square().mean(-1, keepdim=True) + 1e-5).sqrt() * gain

    def rope(x):   # [n, T, heads, hd], pairs (2i, 2i + 1)
        a, b = x[..., 0::2], x[..., 1::2]
        return torch.stack((a * cos - b * sin, a * sin + b * cos), -1).flatten(-2)

    x = w[at[0]:at[1]].view(-1, D)[torch.from_numpy(toks).long().cuda()].double()
    mask = torch.ones(T, T, dtype=torch.bool, device="cuda").triu(1)
    for l in range(L):
        h = norm(x, ten(1, l, (D,)))
        q = rope((h @ ten(2, l, (D, D)).t()).view(n, T, H, hd))
        k = rope((h @ ten(3, l, (nkv, D)).t()).view(n, T, G, hd)).repeat_interleave(H // G, 2)
        v = (h @ ten(4, l, (nkv, D)).t()).view(n, T, G, hd).repeat_interleave(H // G, 2)
        kt, v = k.permute(0, 2, 3, 1).contiguous(), v.permute(0, 2, 1, 3).contiguous()
        s = torch.matmul(q.permute(0, 2, 1, 3).contiguous(), kt) / math.sqrt(hd)
        o = torch.matmul(s.masked_fill_(mask, float("-inf")).softmax(-1), v)
        del s, kt
        x = x + o.permute(0, 2, 1, 3).reshape(n, T, D) @ ten(5, l, (D, D)).t()
        h = norm(x, ten(6, l, (D,)))
        g = h @ ten(7, l, (F, D)).t()
        x = x + (g * torch.sigmoid(g) * (h @ ten(9, l, (F, D)).t())) @ ten(8, l, (D, F)).t()
    return norm(x, w[at[10]:at[11]].double())


def exact(case, seed):
    c = case
    if c["kind"] == "head":
        st = prepare(c, seed)
        out = st["a"].double() @ st["w"].double().t()
        return out, out.argmax(1).to(torch.int32)
    w, at = _weights(c, seed)
    cls = w[at[11]:at[12]].double().view(-1, c["dim"])
    if c["kind"] == "step":
        toks = _tokens(c, seed, c["batch"], c["ctx"] + 1)
        pos = _positions(c)
        part = max(1, int(2e9 / (8.0 * c["heads"] * (c["ctx"] + 1) ** 2)))
        rows = [_forward64(c, w, at, toks[i:i + part])[torch.arange(len(pos[i:i + part])),
                                                       torch.from_numpy(pos[i:i + part]).long()]
                for i in range(0, c["batch"], part)]
        out = torch.cat(rows) @ cls.t()
        return (out[0] if c["batch"] == 1 else out).cpu().numpy()
    if c["kind"] == "greedy":
        toks = _tokens(c, seed, 1, c["ctx"] + 1)
        ids = []
        for _ in range(c["steps"]):
            row = _forward64(c, w, at, toks)[:, -1] @ cls.t()
            ids.append(int(row.argmax()))
            toks = np.concatenate([toks, np.array([[ids[-1]]], np.int32)], 1)
        return np.array(ids, np.int32)[:, None], row.cpu().numpy()
    toks = _tokens(c, seed, c["nseq"], c["seq"])
    outs = []
    for i in range(c["nseq"]):
        h = _forward64(c, w, at, toks[i:i + 1])[0]
        if c["kind"] == "last":
            outs.append(h[-1:] @ cls.t())
        elif c["kind"] == "logits":
            outs.append(h @ cls.t())
        else:
            lp = (h[:-1] @ cls.t()).log_softmax(-1)
            nxt = torch.from_numpy(toks[i, 1:]).long().cuda()
            outs.append(-lp.gather(1, nxt[:, None]).mean()[None])
    return torch.cat(outs).cpu().numpy()
