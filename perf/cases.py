"""Workloads the attention operators are timed on, each through a public entry point.

Decode (contiguous, paged bf16 and fp8 KV caches), prefill (grouped-query,
head dim 64, sliding window, sparse index) and training steps (forward and
backward of the grouped-query, sliding-window and MLA attention).  `listed()`
names twelve of them; `draw()` gives others from the ranges they stand for.
"""
import math
import random

import torch

import cuda_llm_ops_amd as fg

DEV = "cuda:0"

# The ranges that the listed cases stand for (`draw` takes sizes from them).
# (query heads, KV heads) of a layer or of one tensor-parallel shard of it.
DECODE_HEADS = ((16, 2), (32, 8), (64, 8), (128, 8), (16, 1), (8, 8), (28, 4))
PREFILL_HEADS = ((16, 1), (32, 8), (16, 2), (8, 8), (28, 4), (16, 16))
MAX_KV_BYTES = 1 << 30            # of a drawn uniform or ragged decode
MAX_FLOPS = 2e12                  # of a drawn prefill or training step


# ------------------------------------------------------------------ cases
def listed():
    return [
        # Two short conversations on one shard of a model: latency only.
        dict(name="decode_tiny", kind="decode", B=2, S=512, Hq=16, Hkv=2, lens_seed=-1),
        # A full batch of equal lengths, the reference's decode benchmark: HBM-bound.
        dict(name="decode_uniform", kind="decode", B=60, S=4096, Hq=128, Hkv=8, lens_seed=-1),
        # One user with a long context.
        dict(name="decode_long", kind="decode", B=1, S=32768, Hq=64, Hkv=8, lens_seed=-1),
        # A lightly loaded server: a few sequences of different lengths in 16-token pages.
        dict(name="decode_paged_light", kind="paged", B=8, S=6000, Hq=32, Hkv=8, page=16, fp8=False, lens_seed=5),
        # A fully loaded server with an fp8 cache, ragged up to 32K tokens.
        dict(name="decode_paged_fp8", kind="paged", B=64, S=32768, Hq=64, Hkv=8, page=16, fp8=True, lens_seed=3),
        # Prompts of chat length, odd size.
        dict(name="prefill_chat", kind="prefill", B=2, S=777, Hq=32, Hkv=8, D=128, layout="bshd", causal=True),
        # Long prompts: the largest case.
        dict(name="prefill_long", kind="prefill", B=4, S=16384, Hq=32, Hkv=8, D=128, layout="bshd", causal=True),
        # A small model's head dim.
        dict(name="prefill_d64", kind="prefill", B=2, S=2048, Hq=32, Hkv=8, D=64, layout="bhsd", causal=True),
        # Sparse-index attention over a long prompt: a key list per row.
        dict(name="prefill_sparse", kind="sparse", B=1, S=16384, Hq=16, Hkv=1, n=512),
        # A training step's attention, forward and backward: the reference's
        # prefill, sliding-window and MLA benchmark shapes.
        dict(name="train_gqa", kind="train", B=1, S=4096, Hq=16, Hkv=1, D=128, Dv=128, window=0),
        dict(name="train_swa", kind="train", B=1, S=4096, Hq=16, Hkv=1, D=128, Dv=128, window=512),
        dict(name="train_mla", kind="train", B=1, S=4096, Hq=16, Hkv=16, D=192, Dv=128, window=0),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    family = rng.choice(("decode", "ragged", "paged", "paged", "prefill", "prefill", "small_head", "sparse",
                         "train", "train_swa", "train_mla"))
    if family in ("decode", "ragged", "paged"):
        hq, hkv = rng.choice(DECODE_HEADS)
        s = _log_int(rng, 128, 32768)
        b = _log_int(rng, 1, 64)
        b = max(1, min(b, MAX_KV_BYTES // (s * hkv * 512)))
        case = dict(kind="paged" if family == "paged" else "decode", B=b, S=s, Hq=hq, Hkv=hkv,
                    lens_seed=-1 if family == "decode" else rng.randrange(1 << 20))
        if family == "paged":
            case.update(page=rng.choice((16, 16, 32, 64, 128)), fp8=rng.random() < 0.5)
        return case
    if family == "sparse":
        s = _log_int(rng, 512, 24576)
        return dict(kind="sparse", B=1, S=s, Hq=16, Hkv=1, n=min(s, rng.choice((64, 128, 256, 384, 512, 1024))))
    if family in ("prefill", "small_head"):
        hq, hkv = rng.choice(PREFILL_HEADS)
        d = 128 if family == "prefill" else rng.choice((64, 64, 96, 80))
        s, b = _log_int(rng, 64, 8192), _log_int(rng, 1, 4)
        case = dict(kind="prefill", B=b, S=s, Hq=hq, Hkv=hkv, D=d, layout=rng.choice(("bshd", "bhsd")),
                    causal=rng.random() < 0.85)
    else:
        hq, hkv = rng.choice(PREFILL_HEADS) if family != "train_mla" else rng.choice(((16, 16), (8, 8)))
        s, b = _log_int(rng, 256, 4096), _log_int(rng, 1, 2)
        window = _log_int(rng, 64, 2048) if family == "train_swa" else 0
        case = dict(kind="train", B=b, S=s, Hq=hq, Hkv=hkv, D=192 if family == "train_mla" else 128, Dv=128,
                    window=window)
    while case["B"] > 1 and work(case)["flops"] > MAX_FLOPS:
        case["B"] -= 1
    return case


# ------------------------------------------------------------------ sizes
def _lens(case):
    """The sequences' lengths: the cache's when uniform, else 1 .. S from the case's own seed."""
    if case["lens_seed"] < 0:
        return [case["S"]] * case["B"]
    r = random.Random(case["lens_seed"])
    return [r.randint(1, case["S"]) for _ in range(case["B"])]


def _pairs(s, window, causal=True):
    """Query-key pairs of one head: the causal triangle (or band), or all."""
    if not causal:
        return s * s
    if window <= 0 or window >= s:
        return s * (s + 1) // 2
    return window * (window + 1) // 2 + (s - window) * window


def work(case):
    B, S, Hq, Hkv = case["B"], case["S"], case["Hq"], case["Hkv"]
    kind = case["kind"]
    if kind in ("decode", "paged"):
        tokens = sum(_lens(case))
        elem = 1 if case.get("fp8") else 2
        q_o = 2 * B * Hq * 128 * 2
        return dict(bytes=tokens * Hkv * 2 * 128 * elem + q_o, flops=4 * 128 * Hq * tokens)
    if kind == "sparse":
        n = case["n"]
        entries = B * sum(min(n, i + 1) for i in range(S))
        return dict(bytes=2 * B * S * 128 * (2 * Hq + 2 * Hkv) + B * Hkv * S * n * 4 + B * Hq * S * 4,
                    flops=4 * 128 * Hq * entries)
    D = case["D"]
    Dv = case.get("Dv", D)
    pairs = B * Hq * _pairs(S, case.get("window", 0), case.get("causal", True))
    fwd = 2 * pairs * (D + Dv)
    q, o, k, v = B * S * Hq * D * 2, B * S * Hq * Dv * 2, B * S * Hkv * D * 2, B * S * Hkv * Dv * 2
    if kind == "prefill":
        return dict(bytes=q + k + v + o + B * Hq * S * 4, flops=fwd)
    # forward, then S, dP, dV, dQ and dK of the backward; each input (q, k, v,
    # dO) read and each output (o, lse, dq, dk, dv) written once
    bwd = 2 * pairs * (3 * D + 2 * Dv)
    return dict(bytes=2 * q + 2 * k + 2 * v + 2 * o + B * Hq * S * 4, flops=fwd + bwd)


# ------------------------------------------------------------------ inputs
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _normal(g, *shape):
    return torch.randn(shape, generator=g, device=DEV, dtype=torch.bfloat16)


def _key_lists(g, B, Hkv, S, n, recent=16):
    """int32 [B, Hkv, S, n]: row i lists its latest keys, then keys drawn from
    the rest of its causal prefix; -1 where the prefix is shorter than the list."""
    pos = torch.arange(S, device=DEV)[:, None]
    slot = torch.arange(n, device=DEV)[None, :]
    n_valid = (pos + 1).clamp(max=n)
    near = torch.minimum(n_valid, torch.full_like(n_valid, min(recent, n)))
    start = pos + 1 - near
    rnd = (torch.rand((B, Hkv, S, n), generator=g, device=DEV) * start.clamp(min=1)).to(torch.int32)
    idx = torch.where(slot < near, (start + slot).to(torch.int32), rnd)
    return torch.where(slot < n_valid, idx, torch.full_like(idx, -1)).contiguous()


def prepare(case, seed):
    g = _gen(seed)
    B, S, Hq, Hkv = case["B"], case["S"], case["Hq"], case["Hkv"]
    kind = case["kind"]
    st = dict(case=case)
    if kind in ("decode", "paged"):
        st["q"] = _normal(g, B, Hq, 128)
        lens = _lens(case)
        if case["lens_seed"] >= 0:
            st["lens"] = torch.tensor(lens, device=DEV, dtype=torch.int32)
    if kind == "decode":
        st["k"] = _normal(g, B, S, Hkv, 128)
        st["v"] = _normal(g, B, S, Hkv, 128)
        return st
    if kind == "paged":
        page = case["page"]
        per_seq = [-(-n // page) for n in lens]
        pages = sum(per_seq) + 8
        perm = torch.randperm(pages, generator=g, device=DEV).to(torch.int32)
        table = torch.zeros((B, -(-S // page)), device=DEV, dtype=torch.int32)
        at = 0
        for b, n in enumerate(per_seq):
            table[b, :n] = perm[at:at + n]
            at += n
        st["table"] = table
        for name in ("k", "v"):
            if case["fp8"]:
                # the cache holds K / scale and V / scale
                cache = torch.empty((pages, page, Hkv, 128), device=DEV, dtype=torch.float8_e4m3fn)
                step = max(1, (1 << 28) // (page * Hkv * 128))
                for p0 in range(0, pages, step):
                    part = _normal(g, min(step, pages - p0), page, Hkv, 128)
                    cache[p0:p0 + step] = (part * 16.0).to(torch.float8_e4m3fn)
                st[name] = cache
            else:
                st[name] = _normal(g, pages, page, Hkv, 128)
        st["kv_scale"] = 1.0 / 16.0 if case["fp8"] else 1.0
        return st
    if kind == "sparse":
        st["q"], st["k"], st["v"] = (_normal(g, B, S, h, 128) for h in (Hq, Hkv, Hkv))
        st["idx"] = _key_lists(g, B, Hkv, S, case["n"])
        return st
    D = case["D"]
    Dv = case.get("Dv", D)
    if case.get("layout") == "bshd":
        st["q"], st["k"], st["v"] = _normal(g, B, S, Hq, D), _normal(g, B, S, Hkv, D), _normal(g, B, S, Hkv, Dv)
        return st
    st["q"], st["k"], st["v"] = _normal(g, B, Hq, S, D), _normal(g, B, Hkv, S, D), _normal(g, B, Hkv, S, Dv)
    if kind == "train":
        st["do"] = _normal(g, B, Hq, S, Dv)
        if case["window"] > 0:
            st["sink"] = torch.rand((Hq,), generator=g, device=DEV, dtype=torch.float32) + 0.5
    return st


# ------------------------------------------------------------------ one pass
def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "decode":
        return fg.decode_flash_gqa_bshd(st["q"], st["k"], st["v"], seqlens=st.get("lens"))
    if kind == "paged":
        return fg.decode_flash_gqa_paged(st["q"], st["k"], st["v"], st["table"], st["lens"], k_scale=st["kv_scale"],
                                         v_scale=st["kv_scale"], max_seqlen=case["S"])
    if kind == "sparse":
        return fg.flash_sgqa_forward_bshd(st["q"], st["k"], st["v"], st["idx"])
    if kind == "prefill":
        f = fg.flash_gqa_forward_bshd if case["layout"] == "bshd" else fg.launch_flash_gqa_forward_bf16_kernel
        return f(st["q"], st["k"], st["v"], causal=case["causal"])
    q, k, v, do = st["q"], st["k"], st["v"], st["do"]
    if case["window"] > 0:
        o, lse = fg.launch_flash_swa_forward_bf16_kernel(q, k, v, window_size=case["window"], sink_value=st["sink"])
        dq, dk, dv = fg.launch_flash_swa_backward_bf16_kernel(q, k, v, o, lse, do, window_size=case["window"])
    elif case["D"] != case["Dv"]:
        o, lse = fg.launch_flash_mla_forward_bf16_kernel(q, k, v)
        dq, dk, dv = fg.launch_flash_mla_backward_bf16_kernel(q, k, v, o, lse, do)
    else:
        o, lse = fg.launch_flash_gqa_forward_bf16_kernel(q, k, v)
        dq, dk, dv = fg.launch_flash_gqa_backward_bf16_kernel(q, k, v, o, lse, do)
    return o, lse, dq, dk, dv


# ------------------------------------------------------------------ tolerance
def tolerance(case):
    # bf16 results of fp32 sums, with P (and dS) rounded to bf16.  About four
    # times the largest error against 64 bits over the listed cases and
    # fourteen drawn ones: rel 2.3e-3 (gradients 2.5e-3); max 1.4e-2 (decode),
    # 6.7e-2 (prefill) and 1.7e-1 (dq of the first rows, whose few keys leave
    # single roundings of P and dS visible).
    if case["kind"] in ("decode", "paged"):
        return {"rel": 9e-3, "max": 6e-2}
    if case["kind"] == "train":
        return {"rel": 1e-2, "max": 7e-1}
    return {"rel": 9e-3, "max": 2.7e-1}


# ------------------------------------------------------------------ 64 bits
_ROWS = 1024   # query rows of a head at a time


def _attend(q, k, v, scale, causal, window=0, sink=None, do=None):
    """One head in float64: q [S, D], k [S, D], v [S, Dv] -> out, lse and, with
    do, dq and this head's dk and dv."""
    S = q.shape[0]
    out = torch.empty((S, v.shape[1]), device=DEV, dtype=torch.float64)
    lse = torch.empty((S,), device=DEV, dtype=torch.float64)
    if do is not None:
        dq, dk, dv = torch.empty_like(q), torch.zeros_like(k), torch.zeros_like(v)
    for r0 in range(0, S, _ROWS):
        r1 = min(S, r0 + _ROWS)
        c0 = max(0, r0 - window + 1) if window > 0 else 0
        c1 = r1 if causal else S
        s = (q[r0:r1] @ k[c0:c1].t().contiguous()) * scale
        if causal:
            i = torch.arange(r0, r1, device=DEV)[:, None]
            j = torch.arange(c0, c1, device=DEV)[None, :]
            hidden = j > i
            if window > 0:
                hidden = hidden | (j <= i - window)
            s.masked_fill_(hidden, -math.inf)
        m = s.max(dim=1).values
        p = torch.exp(s - m[:, None])
        total = p.sum(dim=1)
        if sink is not None:
            total = total + sink * torch.exp(-m)
        p /= total[:, None]
        lse[r0:r1] = m + torch.log(total)
        out[r0:r1] = p @ v[c0:c1]
        if do is not None:
            g = do[r0:r1]
            dv[c0:c1] += p.t().contiguous() @ g
            delta = (out[r0:r1] * g).sum(dim=1, keepdim=True)
            ds = p * (g @ v[c0:c1].t().contiguous() - delta) * scale
            dq[r0:r1] = ds @ k[c0:c1]
            dk[c0:c1] += ds.t().contiguous() @ q[r0:r1]
    return (out, lse) if do is None else (out, lse, dq, dk, dv)


def exact(case, seed):
    st = prepare(case, seed)
    B, S, Hq, Hkv = case["B"], case["S"], case["Hq"], case["Hkv"]
    G = Hq // Hkv
    kind = case["kind"]
    if kind in ("decode", "paged"):
        out = torch.empty((B, Hq, 128), device=DEV, dtype=torch.float64)
        for b, n in enumerate(_lens(case)):
            if kind == "paged":
                pages = st["table"][b, :-(-n // case["page"])].long()
                k, v = (st[x][pages].reshape(-1, Hkv, 128)[:n] for x in ("k", "v"))
            else:
                k, v = st["k"][b, :n], st["v"][b, :n]
            for h in range(Hkv):
                kh, vh = k[:, h].double() * st.get("kv_scale", 1.0), v[:, h].double() * st.get("kv_scale", 1.0)
                s = st["q"][b, h * G:(h + 1) * G].double() @ kh.t().contiguous() / math.sqrt(128)
                out[b, h * G:(h + 1) * G] = torch.softmax(s, dim=1) @ vh
        return out
    if kind == "sparse":
        out = torch.zeros((B, S, Hq, 128), device=DEV, dtype=torch.float64)
        lse = torch.empty((B, Hq, S), device=DEV, dtype=torch.float64)
        for b in range(B):
            for h in range(Hkv):
                k, v = st["k"][b, :, h].double(), st["v"][b, :, h].double()
                for r0 in range(0, S, 256):
                    r1 = min(S, r0 + 256)
                    idx = st["idx"][b, h, r0:r1].long()
                    used = (idx >= 0) & (idx < S) & (idx <= torch.arange(r0, r1, device=DEV)[:, None])
                    rows = idx.clamp(0, S - 1)
                    q = st["q"][b, r0:r1, h * G:(h + 1) * G].double()
                    s = torch.matmul(q, k[rows].transpose(1, 2).contiguous()) / math.sqrt(128)
                    s.masked_fill_(~used[:, None, :], -math.inf)
                    lse[b, h * G:(h + 1) * G, r0:r1] = torch.logsumexp(s, dim=2).t()
                    out[b, r0:r1, h * G:(h + 1) * G] = torch.matmul(torch.softmax(s, dim=2), v[rows])
        return out, lse
    bshd = case.get("layout") == "bshd"
    q, k, v = ((st[x].transpose(1, 2) if bshd else st[x]) for x in ("q", "k", "v"))   # [B, H, S, D]
    D, Dv = q.shape[3], v.shape[3]
    train = kind == "train"
    out = torch.empty((B, Hq, S, Dv), device=DEV, dtype=torch.float64)
    lse = torch.empty((B, Hq, S), device=DEV, dtype=torch.float64)
    if train:
        dq = torch.empty((B, Hq, S, D), device=DEV, dtype=torch.float64)
        dk = torch.zeros((B, Hkv, S, D), device=DEV, dtype=torch.float64)
        dv = torch.zeros((B, Hkv, S, Dv), device=DEV, dtype=torch.float64)
    for b in range(B):
        for h in range(Hq):
            kd, vd = k[b, h // G].double().contiguous(), v[b, h // G].double().contiguous()
            r = _attend(q[b, h].double().contiguous(), kd, vd, 1.0 / math.sqrt(D), case.get("causal", True),
                        case.get("window", 0), st["sink"][h].double() if "sink" in st else None,
                        st["do"][b, h].double() if train else None)
            out[b, h], lse[b, h] = r[0], r[1]
            if train:
                dq[b, h] = r[2]
                dk[b, h // G] += r[3]
                dv[b, h // G] += r[4]
    if bshd:
        out = out.transpose(1, 2).contiguous()
    return (out, lse, dq, dk, dv) if train else (out, lse)
