"""The calls whose speed this repository watches, through its public Python entry points.

The framework is one attention backend, so a user's program makes five kinds of call: the
cache-latent forward of a prompt (prefill), the paged decode of a batch, a training step of the
cache-latent mode (forward and backward), and the forward and the training step of the on-the-fly
mode.  `listed()` names a dozen of them from one short prompt to the benchmark's largest shapes;
`draw()` gives others from the same ranges.  Shapes, scales and distributions are the benchmark's
(N(0, 1) * 0.5 latents, N(0, 1) elsewhere, Xavier-uniform weights).
"""
import math
import os
import random
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "ds-flashdmla-moe_amd"))

from python import ops  # noqa: E402

D_QK, D_V, PAGE = 576, 512, 64     # latent row, its value part, tokens per cache page
D_IN, D_LAT = 128, 64              # on-the-fly mode: raw and latent dims per head
MLA_SCALE = 1.0 / math.sqrt(192.0)


def listed():
    return [
        # -- prefill: the forward of a prompt, with the row statistics a later merge needs --------
        # A batch of full prompts on a 16-head share of the model: the benchmark's prefill.
        dict(name="prefill_b4_s2048", op="prefill", B=4, H=16, Sq=2048, Sk=2048, causal=True),
        # One short user prompt of no particular length: few row tiles, latency counts.
        dict(name="prefill_b1_s333", op="prefill", B=1, H=16, Sq=333, Sk=333, causal=True),
        # Chunked prefill: the next 512 tokens of one long prompt against its cached 8192.
        dict(name="prefill_b1_chunk512_of_8192", op="prefill", B=1, H=16, Sq=512, Sk=8192, causal=True),
        # -- decode: one new token per sequence over the paged cache ------------------------------
        # A serving batch with all 128 heads, contexts 1024..8192: the benchmark's decode.
        dict(name="decode_b64_h128", op="decode", B=64, H=128, lo=1024, hi=8192, planned=False, append=False),
        # A single user's token at a context of 5000: launches and latency.
        dict(name="decode_b1_h128", op="decode", B=1, H=128, lo=5000, hi=5000, planned=False, append=False),
        # A decode step on a 16-head tensor-parallel share: the token's row is appended, then read.
        dict(name="decode_b16_h16_append", op="decode", B=16, H=16, lo=1024, hi=8192, planned=False, append=True),
        # -- training steps of the cache-latent mode: forward, then the gradients ----------------
        dict(name="train_b4_s2048", op="train", B=4, H=16, Sq=2048, Sk=2048, causal=True),
        dict(name="train_b2_s391", op="train", B=2, H=16, Sq=391, Sk=391, causal=True),
        # -- on-the-fly mode: forward (evaluation) and training step ------------------------------
        dict(name="otf_b2_s4096", op="otf", B=2, H=32, Sq=4096, Sk=4096, causal=True),
        dict(name="otf_b1_s500", op="otf", B=1, H=32, Sq=500, Sk=500, causal=True),
        dict(name="otf_train_b2_s4096", op="otf_train", B=2, H=32, Sq=4096, Sk=4096, causal=True),
        dict(name="otf_train_b1_s777", op="otf_train", B=1, H=32, Sq=777, Sk=777, causal=True),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
    """A case of the same five kinds: lengths from a few tokens to 8192, odd ones among them."""
    limit = work(listed()[6])["flops"]   # the largest listed case's
    while True:
        op = rng.choice(("prefill", "decode", "train", "otf", "otf_train"))
        if op == "decode":
            case = dict(op=op, B=_log_int(rng, 1, 128), H=rng.choice((8, 16, 32, 64, 128)), lo=_log_int(rng, 16, 2048),
                        planned=rng.random() < 0.5, append=rng.random() < 0.5)
            case["hi"] = _log_int(rng, case["lo"], 8192)
        else:
            heads = (8, 16, 32) if op.startswith("otf") else (4, 8, 16, 32, 64, 128)
            case = dict(op=op, B=_log_int(rng, 1, 16), H=rng.choice(heads), Sq=_log_int(rng, 16, 8192))
            case["Sk"] = case["Sq"]
            if op in ("prefill", "otf") and rng.random() < 0.35:   # a chunk of a longer prompt
                case["Sk"] = _log_int(rng, case["Sq"], 8192)
            case["causal"] = rng.random() < 0.85
        if work(case)["flops"] <= limit and work(case)["bytes"] <= 4e9:
            return case


# ---- sizes --------------------------------------------------------------------------------------
def _lens(case):
    """The batch's context lengths: uniform in [lo, hi], a property of the case (not of the seed)."""
    r = random.Random(case["B"] * 1000003 + case["lo"] * 8209 + case["hi"])
    return [r.randint(case["lo"], case["hi"]) for _ in range(case["B"])]


def _pairs(case):
    """Unmasked (row, key) pairs per (batch, head)."""
    sq, sk = case["Sq"], case["Sk"]
    if not case["causal"]:
        return sq * sk
    return sum(min(sk, i + 1 + sk - sq) for i in range(sq))


def work(case):
    op = case["op"]
    if op == "decode":
        b, h, ctx = case["B"], case["H"], sum(_lens(case))
        n = ctx * D_QK * 2 + b * h * (D_QK + D_V) * 2 + b * h * 4
        if case["append"]:
            n += 2 * b * D_QK * 2
        return {"bytes": n, "flops": 2 * ctx * h * (D_QK + D_V)}
    b, h, sq, sk = case["B"], case["H"], case["Sq"], case["Sk"]
    pairs = b * h * _pairs(case)
    if op in ("prefill", "train"):
        q, k, o = b * h * sq * D_QK * 2, b * sk * D_QK * 2, b * h * sq * D_V * 2
        if op == "prefill":
            return {"bytes": q + k + o + 2 * b * h * sq * 4, "flops": 2 * pairs * (D_QK + D_V)}
        return {"bytes": 2 * q + 2 * k + 2 * o, "flops": 2 * pairs * (4 * D_QK + 3 * D_V)}
    q, kv, w = b * h * sq * D_LAT * 2, b * sk * h * D_IN * 2, h * D_IN * D_LAT * 2
    proj = 2 * 2 * b * sk * h * D_IN * D_LAT
    if op == "otf":
        return {"bytes": 2 * q + 2 * kv + 2 * w, "flops": 4 * pairs * D_LAT + proj}
    return {"bytes": 4 * q + 4 * kv + 4 * w, "flops": 14 * pairs * D_LAT + 3 * proj}


def tolerance(case):
    """bf16 results of fp32 sums.  Largest seen against `exact`: 2.6e-3 (a bf16 rounding and a bf16
    P); with the sums in another order outputs differ by as much."""
    return {"rel": 1e-2}


# ---- inputs -------------------------------------------------------------------------------------
def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)

    def randn(*shape, std=1.0):
        return (torch.randn(*shape, generator=gen, device="cuda") * std).to(torch.bfloat16)

    s = dict(case)
    b, h = case["B"], case["H"]
    if case["op"] == "decode":
        lens = torch.tensor(_lens(case), dtype=torch.int32)
        pages = (lens + PAGE - 1) // PAGE
        total, width = int(pages.sum()), int(pages.max())
        perm = torch.randperm(total, generator=gen, device="cuda").to(torch.int32).cpu()
        table = torch.zeros(b, width, dtype=torch.int32)
        at = 0
        for i in range(b):
            n = int(pages[i])
            table[i, :n] = perm[at:at + n]
            at += n
        s.update(q=randn(b, h, D_QK, std=0.5), pool=randn(total, PAGE, D_QK, std=0.5), table=table.cuda(),
                 lens=lens.cuda(), plan=None)
        if case["append"]:
            s.update(cached=(lens - 1).cuda(), new_kv=randn(b, 1, D_QK, std=0.5))
        if case["planned"]:   # one plan serves every layer of a decode step
            s["plan"] = ops.flash_dmla_decode_plan(s["lens"], h, width)
        return s
    sq, sk = case["Sq"], case["Sk"]
    if case["op"] in ("prefill", "train"):
        s.update(q=randn(b, h, sq, D_QK, std=0.5), k_lat=randn(b, sk, D_QK, std=0.5))
        if case["op"] == "train":
            s["do"] = randn(b, h, sq, D_V)
            s["q"].requires_grad_(True)
            s["k_lat"].requires_grad_(True)
        return s
    bound = math.sqrt(6.0 / (D_IN + D_LAT))

    def xavier():
        u = torch.rand(h, D_IN, D_LAT, generator=gen, device="cuda")
        return ((2.0 * u - 1.0) * bound).to(torch.bfloat16)

    s.update(q=randn(b, h, sq, D_LAT), k=randn(b, sk, h, D_IN), v=randn(b, sk, h, D_IN), wk=xavier(), wv=xavier())
    if case["op"] == "otf_train":
        s["do"] = randn(b, h, sq, D_LAT)
        for name in ("q", "k", "v", "wk", "wv"):
            s[name].requires_grad_(True)
    return s


# ---- one pass -----------------------------------------------------------------------------------
def run(s):
    op = s["op"]
    if op == "prefill":
        return ops.flash_dmla_fwd(s["q"], s["k_lat"], D_V, MLA_SCALE, s["causal"])
    if op == "decode":
        if s["append"]:
            ops.flash_dmla_kv_append(s["pool"], s["table"], s["cached"], s["new_kv"])
        o, lse = ops.flash_dmla_decode_paged(s["q"], s["pool"], s["table"], s["lens"], D_V, MLA_SCALE,
                                             return_lse=True, plan=s["plan"])
        return (o, lse, s["pool"]) if s["append"] else (o, lse)
    if op == "train":
        o = ops.flash_dmla(s["q"], s["k_lat"], D_V, MLA_SCALE, s["causal"])
        return (o.detach(),) + torch.autograd.grad(o, (s["q"], s["k_lat"]), s["do"])
    if op == "otf":
        return ops.flash_dmla_fwd_onthefly(s["q"], s["k"], s["v"], s["wk"], s["wv"], None, s["causal"])
    leaves = tuple(s[n] for n in ("q", "k", "v", "wk", "wv"))
    o = ops.flash_dmla_onthefly(*leaves, None, s["causal"])
    return (o.detach(),) + torch.autograd.grad(o, leaves, s["do"])


# ---- the same in 64 bits ------------------------------------------------------------------------
def _attention64(q, k, v, scale, causal, do=None):
    """One head (or heads over one latent): q [H, Sq, d], k [Sk, d], v [Sk, e] in float64.
    Returns o, m, l and, with do, dq, dk, dv (dk, dv summed over the heads)."""
    sq, sk = q.shape[1], k.shape[0]
    o = q.new_empty(q.shape[0], sq, v.shape[1])
    m, l = q.new_empty(q.shape[0], sq), q.new_empty(q.shape[0], sq)
    grads = (torch.empty_like(q), torch.zeros_like(k), torch.zeros_like(v)) if do is not None else None
    keys = torch.arange(sk, device=q.device)
    limit = torch.arange(sq, device=q.device) + (sk - sq)
    for h in range(q.shape[0]):
        x = q[h] @ k.T * scale
        if causal:
            x.masked_fill_(keys[None, :] > limit[:, None], float("-inf"))
        m[h] = x.max(dim=1).values
        p = torch.exp(x - m[h][:, None])
        l[h] = p.sum(dim=1)
        p /= l[h][:, None]
        o[h] = p @ v
        if do is not None:
            ds = p * (do[h] @ v.T - (do[h] * o[h]).sum(dim=1, keepdim=True)) * scale
            grads[0][h] = ds @ k
            grads[1].add_(ds.T @ q[h])
            grads[2].add_(p.T @ do[h])
    return (o, m, l) if do is None else (o, m, l) + grads


@torch.no_grad()
def exact(case, seed):
    s = prepare(case, seed)
    op, b, h = case["op"], case["B"], case["H"]
    q = s["q"].double()
    if op == "decode":
        o = q.new_empty(b, h, D_V)
        lse = q.new_empty(b, h)
        pool = s["pool"].double()
        table, lens = s["table"].long(), _lens(case)
        for i, n in enumerate(lens):
            if case["append"]:
                pool[table[i, (n - 1) // PAGE], (n - 1) % PAGE] = s["new_kv"][i, 0].double()
            rows = pool[table[i, :(n + PAGE - 1) // PAGE]].reshape(-1, D_QK)[:n]
            x = q[i] @ rows.T * MLA_SCALE
            lse[i] = torch.logsumexp(x, dim=1)
            o[i] = torch.exp(x - lse[i][:, None]) @ rows[:, :D_V]
        return (o, lse, pool) if case["append"] else (o, lse)
    if op in ("prefill", "train"):
        k = s["k_lat"].double()
        do = s["do"].double() if op == "train" else None
        parts = [_attention64(q[i], k[i], k[i][:, :D_V], MLA_SCALE, case["causal"], None if do is None else do[i])
                 for i in range(b)]
        outs = [torch.stack(x) for x in zip(*parts)]
        if op == "prefill":
            return tuple(outs)
        dk = outs[4]
        dk[..., :D_V] += outs[5]
        return outs[0], outs[3], dk
    wk, wv = s["wk"].double(), s["wv"].double()
    do = s["do"].double() if op == "otf_train" else None
    o = torch.empty_like(q)
    if do is not None:
        dq = torch.empty_like(q)
        dk = q.new_empty(s["k"].shape)
        dv = torch.empty_like(dk)
        dwk, dwv = torch.zeros_like(wk), torch.zeros_like(wv)
    for i in range(b):
        for j in range(h):
            kr, vr = s["k"][i, :, j].double(), s["v"][i, :, j].double()
            r = _attention64(q[i, j][None], kr @ wk[j], vr @ wv[j], 1.0 / math.sqrt(D_LAT), case["causal"],
                             None if do is None else do[i, j][None])
            o[i, j] = r[0][0]
            if do is not None:
                dq[i, j] = r[3][0]
                dk[i, :, j] = r[4] @ wk[j].T
                dv[i, :, j] = r[5] @ wv[j].T
                dwk[j] += kr.T @ r[4]
                dwv[j] += vr.T @ r[5]
    return o if do is None else (o, dq, dk, dv, dwk, dwv)
