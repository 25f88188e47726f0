"""Workloads of mtlattn on one MI355X, through its public entry points.

Each case is a dict of plain values; the functions below build its inputs,
run one pass of it, count its unavoidable work and give its result in 64 bits.
The listed cases cover what a program does with the library: training steps
(forward and backward), prompt prefill, chunked prefill against a KV cache,
decode over contiguous and paged caches, and dense models through the SDPA
adapter, from a few hundred tokens to the library's largest configurations.
`draw` spreads sizes, head counts, head dims, types and options over the
ranges that the listed cases stand for.
"""

import math
import random

import torch
import torch.nn.functional as F

import mtlattn

_DTYPES = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}

# kind: "train" (forward, then gradients), "fwd" (forward only), "paged"
# (paged_decode), "sdpa" (dense adapter).
# api: "varlen" (separate q/k/v), "qkvpacked" or "kvpacked".
# Sequence lengths are drawn from lens_seed: kv lengths spread over
# [kv_lo, kv_hi], query lengths over [q_lo, q_hi], or equal to the kv lengths
# (self-attention) when q_hi is 0.
_BASE = {"kind": "fwd", "api": "varlen", "n": 1, "q_lo": 0, "q_hi": 0, "kv_lo": 1, "kv_hi": 1, "lens_seed": 0,
         "hq": 8, "hkv": 8, "d": 128, "dtype": "bf16", "causal": True, "window": 0, "bias": "none",
         "page": 0, "mask": "none"}


def _case(**kw):
    c = dict(_BASE)
    c.update(kw)
    return c


def listed():
    return [
        # the fp32 plumbing configuration: a few hundred tokens, where the
        # launches and the host path count
        _case(name="train_fp32_small", kind="train", n=4, kv_lo=17, kv_hi=250, hq=4, hkv=4, d=64, dtype="fp32",
              causal=False),
        # sparse-transformer / 3D encoder batch, ragged, non-causal, packed qkv
        _case(name="train_ragged_qkvpacked", kind="train", api="qkvpacked", n=32, kv_lo=256, kv_hi=4096, hq=16,
              hkv=16, d=64, causal=False),
        # causal GQA training step at full size
        _case(name="train_causal_gqa", kind="train", n=8, kv_lo=4096, kv_hi=4096, hq=32, hkv=8, d=128),
        # sliding window with an additive (ALiBi-like) fp32 bias, long sequences
        _case(name="train_window_bias", kind="train", n=2, kv_lo=16384, kv_hi=16384, hq=32, hkv=8, d=128,
              window=4096, bias="alibi"),
        # fine-tuning on a small ragged batch of a GQA model
        _case(name="train_small_batch", kind="train", api="kvpacked", n=4, kv_lo=200, kv_hi=2048, lens_seed=3,
              hq=16, hkv=4, d=128, dtype="fp16"),
        # prefill of a few short prompts: the smallest forward of a server
        _case(name="prefill_prompts", n=3, kv_lo=33, kv_hi=500, lens_seed=5, hq=32, hkv=8, d=128),
        # one chunk of a long prompt per sequence, against the cache so far
        _case(name="prefill_chunk", api="kvpacked", n=2, q_lo=512, q_hi=512, kv_lo=8192, kv_hi=32768, lens_seed=2,
              hq=32, hkv=8, d=128),
        # decode over long contexts: the largest KV stream
        _case(name="decode_long", n=64, q_lo=1, q_hi=1, kv_lo=8192, kv_hi=65536, hq=64, hkv=8, d=128),
        # decode of a chat batch: contexts of a few hundred to two thousand tokens
        _case(name="decode_chat", n=16, q_lo=1, q_hi=1, kv_lo=128, kv_hi=2048, lens_seed=1, hq=32, hkv=8, d=128),
        # decode over a paged cache with speculative tokens
        _case(name="paged_speculative", kind="paged", n=24, q_lo=1, q_hi=4, kv_lo=1024, kv_hi=8192, lens_seed=4,
              hq=32, hkv=8, d=128, dtype="fp16", page=16),
        # encoder batch with a key-padding mask under replace_sdpa()
        _case(name="sdpa_padding", kind="sdpa", n=8, kv_lo=1536, kv_hi=1536, lens_seed=6, hq=16, hkv=16, d=64,
              causal=False, mask="padding"),
        # dense causal prefill through the adapter
        _case(name="sdpa_causal", kind="sdpa", n=2, kv_lo=2048, kv_hi=2048, hq=32, hkv=8, d=128),
    ]


def _loguniform(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.5)))))))


def _heads(rng, d):
    """Head counts in use at this head dim (MHA and GQA of 2 to 8)."""
    return rng.choice([(16, 16), (12, 12), (16, 4), (32, 8), (32, 4)] if d >= 128 else
                      [(16, 16), (12, 12), (32, 32), (16, 4), (32, 8)])


def draw(rng):
    kind = rng.choice(["train_fp32", "train_ragged", "train_gqa", "train_window", "train_small", "prefill", "chunk",
                       "decode_long", "decode_chat", "paged", "sdpa_padding", "sdpa_dense"])
    seed = rng.randrange(1 << 20)
    t16 = rng.choice(["bf16", "bf16", "fp16"])
    if kind == "train_fp32":
        lo = _loguniform(rng, 8, 256)
        return _case(kind="train", n=rng.randint(1, 8), kv_lo=lo, kv_hi=_loguniform(rng, lo, 1024), lens_seed=seed,
                     hq=8, hkv=rng.choice([8, 8, 4, 2]), d=rng.choice([64, 64, 96, 128]), dtype="fp32",
                     causal=rng.random() < 0.5)
    if kind == "train_ragged":
        lo = _loguniform(rng, 32, 512)
        d = rng.choice([64, 64, 80, 128])
        return _case(kind="train", api="qkvpacked", n=rng.randint(4, 24), kv_lo=lo, kv_hi=_loguniform(rng, lo, 4096),
                     lens_seed=seed, hq=16, hkv=16, d=d, dtype=t16, causal=rng.random() < 0.3)
    if kind == "train_gqa":
        d = rng.choice([64, 96, 128, 128, 128, 256])
        hq, hkv = _heads(rng, d)
        lo = _loguniform(rng, 512, 4096)
        return _case(kind="train", n=rng.randint(1, 6 if d < 256 else 3), kv_lo=lo, kv_hi=lo, lens_seed=seed, hq=hq,
                     hkv=hkv, d=d, dtype=t16)
    if kind == "train_window":
        L = _loguniform(rng, 1024, 12288)
        return _case(kind="train", n=rng.randint(1, 2), kv_lo=L, kv_hi=L, lens_seed=seed, hq=32, hkv=8, d=128,
                     dtype=t16, window=_loguniform(rng, 128, 4096), bias=rng.choice(["none", "alibi"]))
    if kind == "train_small":
        d = rng.choice([64, 80, 128, 128, 128])
        hq, hkv = _heads(rng, d)
        lo = _loguniform(rng, 16, 512)
        return _case(kind="train", api="kvpacked", n=rng.randint(1, 6), kv_lo=lo, kv_hi=_loguniform(rng, lo, 2048),
                     lens_seed=seed, hq=hq, hkv=hkv, d=d, dtype=t16)
    if kind == "prefill":
        d = rng.choice([64, 96, 128, 128, 128, 256])
        hq, hkv = _heads(rng, d)
        lo = _loguniform(rng, 16, 1024)
        return _case(n=rng.randint(1, 8), kv_lo=lo, kv_hi=_loguniform(rng, lo, 4096), lens_seed=seed, hq=hq, hkv=hkv,
                     d=d, dtype=t16)
    if kind == "chunk":
        d = rng.choice([64, 128, 128, 128])
        hq, hkv = _heads(rng, d)
        c = _loguniform(rng, 32, 1024)
        lo = _loguniform(rng, 1024, 16384)
        return _case(api="kvpacked", n=rng.randint(1, 4), q_lo=max(1, c // 2) if rng.random() < 0.5 else c, q_hi=c,
                     kv_lo=lo, kv_hi=_loguniform(rng, lo, 32768), lens_seed=seed, hq=hq, hkv=hkv, d=d, dtype=t16,
                     window=rng.choice([0, 0, 0, 4096]))
    if kind == "decode_long":
        d = rng.choice([64, 128, 128, 128])
        hq, hkv = _heads(rng, d)
        lo = _loguniform(rng, 4096, 32768)
        return _case(n=_loguniform(rng, 1, 32), q_lo=1, q_hi=1, kv_lo=lo, kv_hi=_loguniform(rng, lo, 65536),
                     lens_seed=seed, hq=hq, hkv=hkv, d=d, dtype=t16)
    if kind == "decode_chat":
        d = rng.choice([64, 128, 128, 128])
        hq, hkv = _heads(rng, d)
        lo = _loguniform(rng, 32, 1024)
        return _case(n=_loguniform(rng, 1, 64), q_lo=1, q_hi=1, kv_lo=lo, kv_hi=_loguniform(rng, lo, 4096),
                     lens_seed=seed, hq=hq, hkv=hkv, d=d, dtype=t16)
    if kind == "paged":
        d = rng.choice([64, 128, 128, 128])
        hq, hkv = _heads(rng, d)
        lo = _loguniform(rng, 64, 4096)
        return _case(kind="paged", n=_loguniform(rng, 1, 64), q_lo=1, q_hi=rng.choice([1, 1, 2, 4, 8]), kv_lo=lo,
                     kv_hi=_loguniform(rng, lo, 16384), lens_seed=seed, hq=hq, hkv=hkv, d=d, dtype=t16,
                     page=rng.choice([16, 64, 256]), window=rng.choice([0, 0, 0, 2048]))
    if kind == "sdpa_padding":
        L = _loguniform(rng, 1024, 4096)
        return _case(kind="sdpa", n=rng.randint(1, 8), kv_lo=L, kv_hi=L, lens_seed=seed, hq=16, hkv=16,
                     d=rng.choice([64, 64, 80, 128]), dtype=t16, causal=False, mask="padding")
    d = rng.choice([64, 128, 128])
    hq, hkv = _heads(rng, d)
    L = _loguniform(rng, 128, 4096)
    mask = rng.choice(["none", "none", "bool", "float"])
    return _case(kind="sdpa", n=rng.randint(1, 4), kv_lo=L, kv_hi=L, lens_seed=seed, hq=hq, hkv=hkv, d=d, dtype=t16,
                 causal=mask == "none" and rng.random() < 0.6, mask=mask)


def _lens(case):
    """(query lengths, kv lengths); every query has at least one key."""
    rng = random.Random(case["lens_seed"])
    kv = [rng.randint(case["kv_lo"], case["kv_hi"]) for _ in range(case["n"])]
    if case["q_hi"] == 0:
        return list(kv), kv
    return [min(x, rng.randint(case["q_lo"], case["q_hi"])) for x in kv], kv


def _pad_lens(case):
    """Kept tokens per batch row of a padded batch (the longest row is full)."""
    rng = random.Random(case["lens_seed"])
    N = case["kv_lo"]
    out = [rng.randint(max(1, N // 4), N) for _ in range(case["n"])]
    out[0] = N
    return out


def _cu(lens, device):
    c = [0]
    for x in lens:
        c.append(c[-1] + x)
    return torch.tensor(c, dtype=torch.int32, device=device)


def _inputs(case, seed):
    """Every tensor of the case from the seed, as a program holds it on the GPU."""
    dev = "cuda"
    g = torch.Generator(device=dev).manual_seed(seed)
    dt = _DTYPES[case["dtype"]]

    def rand(*shape):
        return torch.randn(shape, generator=g, device=dev, dtype=torch.float32).to(dt)

    hq, hkv, d, n = case["hq"], case["hkv"], case["d"], case["n"]
    s = {"case": case}
    if case["kind"] == "sdpa":
        N = case["kv_lo"]
        s["q"], s["k"], s["v"] = rand(n, hq, N, d), rand(n, hkv, N, d), rand(n, hkv, N, d)
        s["mask"] = None
        if case["mask"] == "padding":
            lens = torch.tensor(_pad_lens(case), device=dev)
            s["mask"] = (torch.arange(N, device=dev)[None, :] < lens[:, None])[:, None, None, :]
        elif case["mask"] == "bool":        # a random block-sparse pattern, the diagonal kept
            keep = torch.rand((n, 1, N, N), generator=g, device=dev) < 0.7
            s["mask"] = keep | torch.eye(N, dtype=torch.bool, device=dev)
        elif case["mask"] == "float":       # a relative-position bias shared by the batch
            r = torch.arange(N, device=dev)
            s["mask"] = (-(r[:, None] - r[None, :]).abs().float() / 64.0)[None, None]
        return s
    ql, kl = _lens(case)
    mq, mk = sum(ql), sum(kl)
    s["max_q"], s["max_kv"] = max(ql), max(kl)
    s["cu_q"], s["cu_kv"] = _cu(ql, dev), _cu(kl, dev)
    if case["api"] == "qkvpacked":
        s["qkv"] = rand(mk, 3, hq, d)
    elif case["api"] == "kvpacked":
        s["q"], s["kv"] = rand(mq, hq, d), rand(mk, 2, hkv, d)
    elif case["kind"] == "paged":
        # a cache with a fifth of its pages free, the sequences' pages scattered in it
        page = case["page"]
        pages = [-(-x // page) for x in kl]
        total = sum(pages) + sum(pages) // 4 + 1
        s["q"] = rand(mq, hq, d)
        s["k_cache"], s["v_cache"] = rand(total, page, hkv, d), rand(total, page, hkv, d)
        perm = torch.randperm(total, generator=g, device=dev).to(torch.int32)
        table = torch.zeros((n, max(pages)), dtype=torch.int32, device=dev)
        used = 0
        for i, p in enumerate(pages):
            table[i, :p] = perm[used:used + p]
            used += p
        s["table"] = table
    else:
        s["q"], s["k"], s["v"] = rand(mq, hq, d), rand(mk, hkv, d), rand(mk, hkv, d)
    if case["kind"] == "train":
        s["do"] = rand(mq, hq, d)
    s["bias"] = None
    if case["bias"] == "alibi":             # -(i - j) / 16 on sequence-local positions, 0 past the diagonal
        bias = torch.zeros((mq, 1, max(kl)), dtype=torch.float32, device=dev)
        off = 0
        for a, b in zip(ql, kl):
            i = torch.arange(a, device=dev, dtype=torch.float32)[:, None] + (b - a)
            j = torch.arange(b, device=dev, dtype=torch.float32)[None, :]
            bias[off:off + a, 0, :b] = (j - i).clamp_(max=0) / 16.0
            off += a
        s["bias"] = bias
    return s


def prepare(case, seed):
    s = _inputs(case, seed)
    if case["kind"] == "train":
        s["leaves"] = [s[x].requires_grad_() for x in ("qkv", "q", "k", "v", "kv") if x in s]
    if case["mask"] == "padding":
        mtlattn.replace_sdpa()
    return s


def _attend(s):
    c = s["case"]
    if c["api"] == "qkvpacked":
        return mtlattn.flash_attn_varlen_qkvpacked_func(s["qkv"], s["cu_kv"], s["max_kv"], causal=c["causal"],
                                                        window=c["window"])
    if c["api"] == "kvpacked":
        return mtlattn.flash_attn_varlen_kvpacked_func(s["q"], s["kv"], s["cu_q"], s["cu_kv"], s["max_q"],
                                                       s["max_kv"], causal=c["causal"], window=c["window"])
    return mtlattn.varlen_attention(s["q"], s["k"], s["v"], s["cu_q"], s["cu_kv"], s["max_q"], causal=c["causal"],
                                    window=c["window"], attn_bias=s["bias"])


def run(state):
    c = state["case"]
    if c["kind"] == "train":
        out = _attend(state)
        grads = torch.autograd.grad(out, state["leaves"], state["do"])
        return (out.detach(), *grads)
    if c["kind"] == "paged":
        return mtlattn.paged_decode(state["q"], state["k_cache"], state["v_cache"], state["cu_q"], state["cu_kv"],
                                    state["table"], state["max_q"], state["max_kv"], causal=c["causal"],
                                    window=c["window"])
    if c["kind"] == "sdpa":
        if c["mask"] == "padding":
            return F.scaled_dot_product_attention(state["q"], state["k"], state["v"], attn_mask=state["mask"])
        return mtlattn.sdpa(state["q"], state["k"], state["v"], attn_mask=state["mask"], is_causal=c["causal"])
    return _attend(state)


def _pairs(ql, kl, causal, window):
    """Attended (query, key) pairs of one head: per sequence, query i sees
    keys (i + off - window, i + off] of [0, kv), off = kv - q."""
    total = 0
    for a, b in zip(ql, kl):
        off = b - a
        i = torch.arange(a, dtype=torch.int64)
        hi = torch.clamp(i + off + 1, max=b) if causal else torch.full_like(i, b)
        lo = torch.clamp(i + off - window + 1, min=0) if window > 0 else torch.zeros_like(i)
        total += int((hi - lo).clamp(min=0).sum())
    return total


def work(case):
    hq, hkv, d = case["hq"], case["hkv"], case["d"]
    es = 4 if case["dtype"] == "fp32" else 2
    if case["kind"] == "sdpa":
        N, n = case["kv_lo"], case["n"]
        lens = _pad_lens(case) if case["mask"] == "padding" else [N] * n
        pairs = _pairs(lens, lens, case["causal"], 0)
        # valid rows of q, k and v in, the whole dense output out
        nbytes = sum(lens) * (hq + 2 * hkv) * d * es + n * N * hq * d * es
        nbytes += {"none": 0, "padding": n * N, "bool": n * N * N, "float": 4 * N * N}[case["mask"]]
        return {"bytes": nbytes, "flops": 4 * d * hq * pairs}
    ql, kl = _lens(case)
    pairs = _pairs(ql, kl, case["causal"], case["window"])
    if case["window"] > 0:                  # keys that some query sees
        kv = sum(min(b, case["window"] + a - 1) for a, b in zip(ql, kl))
    else:
        kv = sum(kl)
    q_bytes, kv_bytes = sum(ql) * hq * d * es, kv * hkv * d * es
    bias = 4 * pairs if case["bias"] != "none" else 0
    if case["kind"] == "train":             # q, k, v, do in; out, dq, dk, dv out
        return {"bytes": 4 * q_bytes + 2 * kv_bytes + 2 * sum(kl) * hkv * d * es + bias, "flops": 14 * d * hq * pairs}
    return {"bytes": 2 * q_bytes + 2 * kv_bytes + bias, "flops": 4 * d * hq * pairs}


def tolerance(case):
    # 16-bit: P, dS and the outputs are rounded to the input type; measured
    # against 64 bits at most 3.0e-3 (bf16) and 3.4e-4 (fp16). fp32: 3.6e-7
    # on a few hundred keys, more terms at the top of the range.
    return {"rel": {"bf16": 1e-2, "fp16": 1.5e-3, "fp32": 4e-6}[case["dtype"]]}


def _exact_attention(q, k, v, do, ql, kl, causal, window, bias):
    """Attention in float64, per sequence and block of queries, all heads at
    once; with `do` also the gradients. bias(s, i0, i1, j0, j1) gives the
    additive mask of sequence s for those rows and keys."""
    hq, d, hkv = q.shape[1], q.shape[2], k.shape[1]
    g, scale = hq // hkv, 1.0 / math.sqrt(d)
    f64 = dict(dtype=torch.float64, device=q.device)
    out = torch.zeros(q.shape, **f64)
    grads = [torch.zeros(t.shape, **f64) for t in (q, k, v)] if do is not None else None
    q0 = k0 = 0
    for s, (a, b) in enumerate(zip(ql, kl)):
        K = k[k0:k0 + b].double().transpose(0, 1).contiguous()      # [hkv, b, d]
        V = v[k0:k0 + b].double().transpose(0, 1).contiguous()
        off = b - a
        rows = max(1, min(a, (1 << 26) // (hq * b)))
        for i0 in range(0, a, rows):
            i1 = min(a, i0 + rows)
            j0 = max(0, i0 + off - window + 1) if window > 0 else 0
            j1 = min(b, i1 + off) if causal else b
            Kb, Vb = K[:, j0:j1].contiguous(), V[:, j0:j1].contiguous()
            Kt, Vt = Kb.transpose(1, 2).contiguous(), Vb.transpose(1, 2).contiguous()

            def fold(t):                                            # [rows, hq, d] -> [hkv, g * rows, d]
                return t[q0 + i0:q0 + i1].double().transpose(0, 1).reshape(hkv, g * (i1 - i0), d)

            def unfold(t):
                return t.reshape(hq, i1 - i0, d).transpose(0, 1)

            Q = fold(q)
            S = (torch.matmul(Q, Kt) * scale).view(hkv, g, i1 - i0, j1 - j0)
            if bias is not None:
                S += bias(s, i0, i1, j0, j1)
            i = torch.arange(i0, i1, device=q.device)[:, None] + off
            j = torch.arange(j0, j1, device=q.device)[None, :]
            if causal:
                S.masked_fill_(j > i, float("-inf"))
            if window > 0:
                S.masked_fill_(j <= i - window, float("-inf"))
            P = torch.softmax(S, -1).view(hkv, g * (i1 - i0), j1 - j0)
            O = torch.matmul(P, Vb)
            out[q0 + i0:q0 + i1] = unfold(O)
            if do is None:
                continue
            dO = fold(do)
            dS = torch.matmul(dO, Vt)
            dS -= (dO * O).sum(-1, keepdim=True)
            dS *= P
            grads[0][q0 + i0:q0 + i1] = unfold(torch.matmul(dS, Kb) * scale)
            grads[1][k0 + j0:k0 + j1] += torch.matmul(dS.transpose(1, 2).contiguous(), Q).transpose(0, 1) * scale
            grads[2][k0 + j0:k0 + j1] += torch.matmul(P.transpose(1, 2).contiguous(), dO).transpose(0, 1)
        q0, k0 = q0 + a, k0 + b
    return out, grads


def exact(case, seed):
    s = _inputs(case, seed)
    if case["kind"] == "sdpa":
        n, hq, N, d = s["q"].shape
        lens = _pad_lens(case) if case["mask"] == "padding" else [N] * n
        out = torch.zeros((n, hq, N, d), dtype=torch.float64, device=s["q"].device)
        m = s["mask"]
        for b in range(n):                  # padded query rows are defined as 0
            L = lens[b]
            q, k, v = (s[x][b, :, :L].transpose(0, 1) for x in ("q", "k", "v"))
            bias = None
            if case["mask"] in ("bool", "float"):
                mb = m[min(b, m.shape[0] - 1), 0].double()
                if case["mask"] == "bool":
                    mb = torch.where(mb > 0, 0.0, float("-inf")).double()

                def bias(_, i0, i1, j0, j1, mb=mb):
                    return mb[i0:i1, j0:j1]
            o, _ = _exact_attention(q, k, v, None, [L], [L], case["causal"], 0, bias)
            out[b, :, :L] = o.transpose(0, 1)
        return out
    ql, kl = _lens(case)
    if case["api"] == "qkvpacked":
        q, k, v = s["qkv"].unbind(1)
    elif case["api"] == "kvpacked":
        q, (k, v) = s["q"], s["kv"].unbind(1)
    elif case["kind"] == "paged":
        page = case["page"]
        rows = []
        for i, L in enumerate(kl):
            j = torch.arange(L, device=s["q"].device)
            rows.append(s["table"][i, j // page].long() * page + j % page)
        rows = torch.cat(rows)
        q = s["q"]
        k, v = (s[x].flatten(0, 1)[rows] for x in ("k_cache", "v_cache"))
    else:
        q, k, v = s["q"], s["k"], s["v"]
    bias = None
    if s["bias"] is not None:
        starts = [sum(ql[:i]) for i in range(len(ql))]

        def bias(i, i0, i1, j0, j1):
            return s["bias"][starts[i] + i0:starts[i] + i1, 0, j0:j1].double()
    out, grads = _exact_attention(q, k, v, s.get("do"), ql, kl, case["causal"], case["window"], bias)
    if case["kind"] != "train":
        return out
    if case["api"] == "qkvpacked":
        return out, torch.stack(grads, 1)
    if case["api"] == "kvpacked":
        return out, grads[0], torch.stack(grads[1:], 1)
    return (out, *grads)
