"""Timed workloads of the attention path: what a program that uses this library has it do.

Each case is one pass through the public entry points (``bnhip``, the binding of the C ABI) at the
shapes of TinyLLaMA-1.1B (32 query heads, 4 KV heads of 64, hidden 2048, SwiGLU 5632, vocabulary
32000, 22 layers), the model that the repository's configurations, tests and benchmark use, and at
its neighbours (other group sizes, odd lengths, other batches).  A case names its path:

``decode``      one new token per sequence against KV caches (bf16 serving caches, head-major or
                token-major; fp32 ones): ``gqa_decode`` or ``gqa_decode_planned``
``prefill``     causal GQA attention of a prompt, or of a chunk of new rows behind cached ones
``train``       the attention of a training step: forward with log-sum-exp, then backward
``project``     the front of a decoder layer: residual add + RMSNorm, then the Q/K/V projection
                with RoPE in its epilogue
``fused_head``  the one-softmax-for-all-heads attention that the reference's own layers compute
``generate``    greedy steps of the whole model in native code (``bn_llama_decode``)

``exact`` is the same mathematics in plain torch float64.
"""
import ctypes as C
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "baranet-bdml_amd"))
import bnhip  # noqa: E402

D = 64          # head_dim, fixed by the kernels
THETA = 10000.0
EPS = 1e-5


def _decode(batch, max_len, shortest, longest, heads=32, kv_heads=4, dtype="bf16", head_major=True,
            planned=False):
    return dict(path="decode", dtype=dtype, batch=batch, heads=heads, kv_heads=kv_heads,
                max_len=max_len, shortest=shortest, longest=longest, head_major=head_major,
                planned=planned)


def _prefill(batch, seq_q, seq_kv, heads=32, kv_heads=4, dtype="bf16", causal=True):
    return dict(path="prefill", dtype=dtype, batch=batch, seq_q=seq_q, seq_kv=seq_kv, heads=heads,
                kv_heads=kv_heads, causal=causal)


def _train(batch, seq, heads=32, kv_heads=4):
    return dict(path="train", dtype="bf16", batch=batch, seq=seq, heads=heads, kv_heads=kv_heads)


def _project(rows, hidden=2048, heads=32, kv_heads=4, position=0, dtype="bf16"):
    return dict(path="project", dtype=dtype, rows=rows, hidden=hidden, heads=heads,
                kv_heads=kv_heads, position=position)


def _fused_head(rows, past=0):
    return dict(path="fused_head", dtype="fp32", rows=rows, past=past, heads=32, kv_heads=4)


def _generate(layers, position, tokens):
    return dict(path="generate", dtype="fp32", layers=layers, position=position, tokens=tokens)


def listed():
    return [
        # one user's chat: a single sequence, the smallest call of the path; launches count
        dict(name="decode_one", **_decode(1, 2048, 1543, 1543)),
        # a small server: some sequences of different lengths, token-major caches that its
        # appends write one row at a time
        dict(name="decode_some", **_decode(12, 4096, 200, 4000, head_major=False)),
        # a full batch, ragged U[512, 4096] on 64 caches: the serving configuration
        dict(name="decode_batch", **_decode(64, 4096, 512, 4096)),
        # two ordinary prompts of an odd length
        dict(name="prefill_prompt", **_prefill(2, 777, 777)),
        # a batch of prompts: the headline configuration
        dict(name="prefill_batch", **_prefill(4, 2048, 2048)),
        # chunked prefill: 256 new rows behind 4096 cached ones
        dict(name="prefill_chunk", **_prefill(1, 256, 4352)),
        # one long document
        dict(name="prefill_long", **_prefill(1, 16384, 16384)),
        # the fp32 model's 512-token prompt, one layer
        dict(name="prefill_fp32", **_prefill(1, 512, 512, dtype="fp32")),
        # the attention of a training step on the headline batch
        dict(name="train_batch", **_train(4, 2048)),
        # a layer's norm and Q/K/V projection over a batch of prompts
        dict(name="project_prompt", **_project(2048)),
        # the reference layers' own attention over a 512-token prompt
        dict(name="fused_head_prompt", **_fused_head(512)),
        # four greedy steps of the whole fp32 model behind a 512-token prompt
        dict(name="generate_model", **_generate(22, 512, 4)),
    ]


def _log(rng, lo, hi):
    """An integer in [lo, hi], spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    heads, kv_heads = rng.choice([(32, 4), (32, 4), (32, 4), (32, 8), (16, 4), (8, 8)])
    path = rng.choice(["decode"] * 3 + ["prefill"] * 4 + ["train", "train", "project", "project",
                                                          "fused_head", "generate"])
    if path == "decode":
        fp32 = rng.random() < 0.25
        max_len = _log(rng, 128, 8192)
        batch = min(_log(rng, 1, 96), (1 << 19) // max_len)
        longest = max(1, int(max_len * rng.uniform(0.5, 1.0)))
        shortest = max(1, int(longest * rng.choice([1.0, rng.uniform(0.05, 1.0)])))
        return _decode(batch, max_len, shortest, longest, heads, kv_heads, "fp32" if fp32 else "bf16",
                       rng.random() < 0.5, not fp32 and rng.random() < 0.3)
    if path == "prefill":
        fp32 = rng.random() < 0.25
        most = (1 << 28) // 8 if fp32 else 1 << 28       # score pairs over batch and heads / 16
        while True:
            batch, seq_q = _log(rng, 1, 8), _log(rng, 16, 8192)
            past = rng.choice([0, 0, _log(rng, 16, 16384)])
            if batch * seq_q * (seq_q // 2 + past) * heads // 16 <= most:
                break
        causal = rng.random() < 0.9
        return _prefill(batch, seq_q, seq_q + past, heads, kv_heads, "fp32" if fp32 else "bf16", causal)
    if path == "train":
        while True:
            batch, seq = _log(rng, 1, 8), _log(rng, 64, 4096)
            if batch * seq * seq <= 4 * 2048 * 2048:
                return _train(batch, seq, heads, kv_heads)
    if path == "project":
        fp32 = rng.random() < 0.25
        rows = _log(rng, 16, 1024 if fp32 else 8192)
        return _project(rows, rng.choice([1024, 2048, 2048, 4096]), heads, kv_heads,
                        rng.randrange(0, 4096), "fp32" if fp32 else "bf16")
    if path == "fused_head":
        return _fused_head(_log(rng, 16, 2048), rng.choice([0, 0, _log(rng, 16, 1024)]))
    return _generate(_log(rng, 2, 22), _log(rng, 16, 1000), rng.randrange(1, 5))


# ------------------------------------------------------------------- inputs
_DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}


def _inputs(case, seed):
    """The call's tensors, from the seed alone (rotated queries and keys, values and activations of
    unit scale, weights of the model's initial scale)."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    dt = _DTYPES[case["dtype"]]

    def normal(*shape, std=1.0, dtype=dt):
        return (torch.randn(shape, generator=g, device="cuda") * std).to(dtype)

    path = case["path"]
    if path == "decode":
        B, H, Hkv, L = case["batch"], case["heads"], case["kv_heads"], case["max_len"]
        lens = np.random.default_rng(seed).integers(case["shortest"], case["longest"] + 1, B)
        q = normal(B, H, D)
        if case["head_major"]:
            k, v = (normal(B, Hkv, L, D).transpose(1, 2) for _ in range(2))
        else:
            k, v = (normal(B, L, Hkv, D) for _ in range(2))
        return dict(q=q, k=k, v=v, lens=[int(n) for n in lens])
    if path in ("prefill", "train"):
        B, H, Hkv = case["batch"], case["heads"], case["kv_heads"]
        sq = case["seq_q"] if path == "prefill" else case["seq"]
        skv = case["seq_kv"] if path == "prefill" else case["seq"]
        t = dict(q=normal(B, sq, H, D), k=normal(B, skv, Hkv, D), v=normal(B, skv, Hkv, D))
        if path == "train":
            t["dout"] = normal(B, sq, H, D)
        return t
    if path == "project":
        m, k = case["rows"], case["hidden"]
        n = (case["heads"] + 2 * case["kv_heads"]) * D
        return dict(x=normal(m, k), delta=normal(m, k, std=0.3), norm=1 + normal(1, k, std=0.1),
                    w=normal(k, n, std=0.02))
    if path == "fused_head":
        m, n = case["rows"], case["rows"] + case["past"]
        return dict(q=normal(m, case["heads"] * D, std=0.3), k=normal(n, case["kv_heads"] * D, std=0.3),
                    v=normal(n, case["kv_heads"] * D))
    # generate: projection weights output-major ([out, in]), as the model driver stores them
    hid, inter, vocab, kv, n = 2048, 5632, 32000, 4 * D, case["layers"]
    max_len = case["position"] + case["tokens"]
    t = dict(embed=normal(vocab, hid, std=0.02), ln_f=1 + normal(hid, std=0.1),
             lm_head=normal(vocab, hid, std=0.02), k=normal(n, max_len, 4, D), v=normal(n, max_len, 4, D))
    for name, shape in (("wqkv", (hid + 2 * kv, hid)), ("wo", (hid, hid)), ("wgu", (2 * inter, hid)),
                        ("wd", (hid, inter))):
        t[name] = [normal(*shape, std=0.02) for _ in range(n)]
    for name in ("ln1", "ln2"):
        t[name] = [1 + normal(hid, std=0.1) for _ in range(n)]
    t["first"] = seed % vocab
    return t


def _bytes(n):
    return torch.empty(max(int(n), 16), dtype=torch.uint8, device="cuda")


def prepare(case, seed):
    t = _inputs(case, seed)
    path, L = case["path"], bnhip.lib()
    if path == "decode":
        t["seq_lens"] = torch.tensor(t["lens"], dtype=torch.int32, device="cuda")
        size = (L.bn_gqa_decode_planned_workspace_size(case["batch"], case["max_len"], case["heads"],
                                                       case["kv_heads"], D) if case["planned"] else
                L.bn_gqa_decode_workspace_size(case["batch"], case["max_len"], case["heads"], D))
        t["workspace"] = _bytes(size)
    elif path == "train":
        t["workspace"] = _bytes(L.bn_gqa_prefill_backward_workspace_size(
            case["batch"], case["seq"], case["seq"], case["heads"], case["kv_heads"], D, 1))
    elif path == "project":
        t["workspace"] = _bytes(L.bn_linear_rope_workspace_size(
            bnhip.BN_BF16 if case["dtype"] == "bf16" else bnhip.BN_F32, case["rows"],
            t["w"].shape[1], case["hidden"]))
    elif path == "generate":
        c = bnhip.BnLlamaConfig(case["layers"], 2048, 32, 4, 5632, 32000,
                                case["position"] + case["tokens"], EPS, THETA, 1)
        t["config"] = c
        t["layers"] = (bnhip.BnLlamaLayer * case["layers"])(*[
            bnhip.BnLlamaLayer(*[t[w][i].data_ptr() for w in ("ln1", "wqkv", "wo", "ln2", "wgu", "wd",
                                                              "k", "v")])
            for i in range(case["layers"])])
        t["tokens"] = torch.zeros(case["tokens"], dtype=torch.int32, device="cuda")
        t["workspace"] = _bytes(L.bn_llama_decode_workspace_size(C.byref(c)))
    t["case"] = case
    return t


# ------------------------------------------------------------------- a pass
def run(state):
    t, case = state, state["case"]
    path = case["path"]
    if path == "decode":
        if case["planned"]:
            return bnhip.gqa_decode_planned(t["q"], t["k"], t["v"], t["seq_lens"], t["lens"],
                                            workspace=t["workspace"])
        return bnhip.gqa_decode(t["q"], t["k"], t["v"], t["seq_lens"], workspace=t["workspace"])
    if path == "prefill":
        offset = case["seq_kv"] - case["seq_q"]
        return bnhip.gqa_prefill(t["q"], t["k"], t["v"], causal=case["causal"], seq_offset=offset)
    if path == "train":
        o, lse = bnhip.gqa_prefill_lse(t["q"], t["k"], t["v"])
        dq, dk, dv = bnhip.gqa_prefill_backward(t["q"], t["k"], t["v"], o, t["dout"], lse,
                                                workspace=t["workspace"])
        return dict(o=o, lse=lse, dq=dq, dk=dk, dv=dv)
    if path == "project":
        h, y = bnhip.add_rmsnorm(t["x"], t["delta"], t["norm"], EPS)
        qkv = bnhip.linear_rope(y, t["w"], rope_cols=(case["heads"] + case["kv_heads"]) * D,
                                position_offset=case["position"], head_dim=D, theta=THETA,
                                workspace=t["workspace"])
        return dict(h=h, y=y, qkv=qkv)
    if path == "fused_head":
        return bnhip.fused_head_attention(t["q"], t["k"], t["v"], case["heads"], case["kv_heads"], D,
                                          seq_offset=case["past"])
    bnhip.call("bn_llama_decode", C.byref(t["config"]), t["embed"].data_ptr(), t["ln_f"].data_ptr(),
               t["lm_head"].data_ptr(), t["layers"], t["first"], case["position"], case["tokens"],
               t["tokens"].data_ptr(), t["workspace"].data_ptr(), t["workspace"].numel(),
               bnhip.stream_of())
    # the caches whole, and the rows that these steps appended
    new = slice(case["position"], case["position"] + case["tokens"])
    return dict(tokens=t["tokens"], k=t["k"], v=t["v"], k_new=t["k"][:, new], v_new=t["v"][:, new])


# ------------------------------------------------------------------- its cost
def _pairs(case):
    """Visible (query, key) pairs of one head of one sequence."""
    sq = case["seq_q"] if case["path"] == "prefill" else case["seq"]
    skv = case["seq_kv"] if case["path"] == "prefill" else case["seq"]
    if not case.get("causal", True):
        return sq * skv
    return sq * (skv - sq) + sq * (sq + 1) // 2


def work(case):
    path, e = case["path"], 2 if case["dtype"] == "bf16" else 4
    H, Hkv = case.get("heads", 32), case.get("kv_heads", 4)
    if path == "decode":
        keys = case["batch"] * (case["shortest"] + case["longest"]) / 2
        return {"bytes": keys * 2 * Hkv * D * e + 2 * case["batch"] * H * D * e,
                "flops": 4 * keys * H * D}
    if path == "prefill":
        b = case["batch"]
        return {"bytes": e * D * b * (2 * case["seq_q"] * H + 2 * case["seq_kv"] * Hkv),
                "flops": 4 * b * H * D * _pairs(case)}
    if path == "train":  # two products forward, five backward; q k v dout in, o lse dq dk dv out
        b, s = case["batch"], case["seq"]
        return {"bytes": b * s * (e * D * (4 * H + 4 * Hkv) + 4 * H),
                "flops": 14 * b * H * D * _pairs(case)}
    if path == "project":
        m, k, n = case["rows"], case["hidden"], (H + 2 * Hkv) * D
        return {"bytes": e * (4 * m * k + k + k * n + m * n), "flops": 2 * m * n * k}
    if path == "fused_head":  # group sums of q against the KV heads' width, once for all heads
        m, n = case["rows"], case["rows"] + case["past"]
        pairs = m * case["past"] + m * (m + 1) // 2
        return {"bytes": e * D * (2 * m * H + 2 * n * Hkv), "flops": 4 * Hkv * D * pairs}
    weights = case["layers"] * (2048 * 2560 + 2048 * 2048 + 3 * 2048 * 5632) + 2048 * 32000
    keys = case["layers"] * (case["position"] + case["tokens"] / 2) * 2 * 4 * D
    return {"bytes": case["tokens"] * e * (weights + keys), "flops": case["tokens"] * 2 * weights}


def tolerance(case):
    # about four times what the outputs differ by from the same mathematics in 64 bits
    path = case["path"]
    if path == "generate":
        return {"rel": 4e-5, "max": 2e-3}
    if case["dtype"] == "fp32":
        return {"rel": 2e-6, "max": 1e-4}
    return {"rel": 1e-2, "max": 0.1}


# ------------------------------------------------------------------- the same in 64 bits
def _rope64(x, position):
    """op_rope: adjacent pairs of each head rotated by position * theta^(-2p/D)."""
    rows = x.shape[0]
    freq = THETA ** (-torch.arange(0, D, 2, dtype=torch.float64, device=x.device) / D)
    a = (position + torch.arange(rows, dtype=torch.float64, device=x.device))[:, None] * freq
    cos, sin = a.cos()[:, None], a.sin()[:, None]
    h = x.reshape(rows, -1, D // 2, 2)
    return torch.stack([h[..., 0] * cos - h[..., 1] * sin, h[..., 0] * sin + h[..., 1] * cos],
                       dim=-1).reshape(rows, -1)


def _norm64(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w


def _head64(q, k, v, hidden):
    """One head: q [S, D], k/v [T, D] float64, hidden [S, T] or None -> o, probabilities, lse."""
    s = q @ k.T / math.sqrt(D)
    if hidden is not None:
        s.masked_fill_(hidden, -math.inf)
    lse = torch.logsumexp(s, dim=1, keepdim=True)
    p = s.sub_(lse).exp_()
    return p @ v, p, lse[:, 0]


def _hidden(sq, skv, causal):
    if not causal:
        return None
    return torch.ones(sq, skv, dtype=torch.bool, device="cuda").triu(skv - sq + 1)


def exact(case, seed):
    t = _inputs(case, seed)
    path = case["path"]
    H, Hkv = case.get("heads", 32), case.get("kv_heads", 4)
    G = H // Hkv
    if path == "decode":
        out = torch.empty(case["batch"], H, D, dtype=torch.float64, device="cuda")
        for b, n in enumerate(t["lens"]):
            for g in range(Hkv):
                rows = slice(g * G, (g + 1) * G)
                out[b, rows] = _head64(t["q"][b, rows].double(), t["k"][b, :n, g].double(),
                                       t["v"][b, :n, g].double(), None)[0]
        return out
    if path in ("prefill", "train"):
        B, sq, skv = t["q"].shape[0], t["q"].shape[1], t["k"].shape[1]
        hidden = _hidden(sq, skv, case.get("causal", True))
        o = torch.empty(t["q"].shape, dtype=torch.float64, device="cuda")
        if path == "train":
            lse = torch.empty(B, H, sq, dtype=torch.float64, device="cuda")
            dq = torch.empty_like(o)
            dk, dv = (torch.zeros(t["k"].shape, dtype=torch.float64, device="cuda") for _ in range(2))
        for b in range(B):
            for h in range(H):
                g = h // G
                q, k, v = t["q"][b, :, h].double(), t["k"][b, :, g].double(), t["v"][b, :, g].double()
                oh, p, row = _head64(q, k, v, hidden)
                o[b, :, h] = oh
                if path == "train":
                    do = t["dout"][b, :, h].double()
                    ds = p * (do @ v.T - (do * oh).sum(1, keepdim=True)) / math.sqrt(D)
                    lse[b, h] = row
                    dq[b, :, h] = ds @ k
                    dk[b, :, g] += ds.T @ q
                    dv[b, :, g] += p.T @ do
        return dict(o=o, lse=lse, dq=dq, dk=dk, dv=dv) if path == "train" else o
    if path == "project":
        h = t["x"].double() + t["delta"].double()
        y = _norm64(h, t["norm"].double())
        qkv = y @ t["w"].double()
        n = (H + Hkv) * D
        return dict(h=h, y=y, qkv=torch.cat([_rope64(qkv[:, :n].contiguous(), case["position"]),
                                             qkv[:, n:]], dim=1))
    if path == "fused_head":
        m, n = case["rows"], case["rows"] + case["past"]
        q, k, v = (t[w].double() for w in ("q", "k", "v"))
        s = q.reshape(m, Hkv, G, D).sum(2).reshape(m, Hkv * D) @ k.T / math.sqrt(D)
        s.masked_fill_(_hidden(m, n, True), -math.inf)
        o = (torch.softmax(s, dim=1) @ v).reshape(m, Hkv, 1, D)
        return o.expand(m, Hkv, G, D).reshape(m, H * D)
    # generate
    hid, inter = 2048, 5632
    k_cache, v_cache = t["k"].double(), t["v"].double()
    token, lm_head = t["first"], t["lm_head"].double()
    for step in range(case["tokens"]):
        pos = case["position"] + step
        x = t["embed"][token:token + 1].double()
        for i in range(case["layers"]):
            qkv = _norm64(x, t["ln1"][i].double()) @ t["wqkv"][i].double().T
            qk = _rope64(qkv[:, :hid + 4 * D].contiguous(), pos)
            k_cache[i, pos] = qk[0, hid:].reshape(4, D)
            v_cache[i, pos] = qkv[0, hid + 4 * D:].reshape(4, D)
            q = qk[0, :hid].reshape(4, 8, D)
            o = torch.cat([_head64(q[g], k_cache[i, :pos + 1, g], v_cache[i, :pos + 1, g], None)[0]
                           for g in range(4)])
            x = x + o.reshape(1, hid) @ t["wo"][i].double().T
            gu = _norm64(x, t["ln2"][i].double()) @ t["wgu"][i].double().T
            x = x + (torch.nn.functional.silu(gu[:, :inter]) * gu[:, inter:]) @ t["wd"][i].double().T
        token = int(torch.argmax(_norm64(x, t["ln_f"].double()) @ lm_head.T))
    new = slice(case["position"], case["position"] + case["tokens"])
    return dict(tokens=None, k=k_cache, v=v_cache, k_new=k_cache[:, new], v_new=v_cache[:, new])
