"""Parity of the on-the-fly backward (dmla_bwd_onthefly) with fp32 references.

Each case runs this library's on-the-fly forward, then its backward from the saved (o, m, l)
twice: once with every gradient in fp32 (dq_dtype, dkv_dtype, dw_dtype float32) and once with
the default dtypes (dq, dk, dv bf16; dwk, dwv fp32).  The default outputs must be exactly the
fp32 ones rounded to bf16 (the kernels compute the same fp32 values and round them last), so
the tolerance checks run on the fp32 outputs, which carry no output rounding:
  * against the closed-form oracle backward fed with the same o, m, l -- isolates the
    backward kernels -- at the north-star tolerance: 2e-2 max-abs and 1e-2 mean-rel, flat;
  * against fp32 torch.autograd through the exact on-the-fly forward -- the end-to-end gradient
    of the op.  No kernel can meet the flat bar there: D = rowsum(dO * O) takes the forward's
    bf16 O, and that rounding alone moves dwk by up to ~3e-2 at these sizes (the exact math fed
    with the bf16-rounded O, in fp64, against the exact gradient).  So against autograd each
    gradient may differ by that same-O error of the oracle plus 2e-2 max-abs, and by 1e-2
    mean-rel.
The few-keys cases (a handful of keys seen by hundreds or thousands of rows) are where the
gradients grow largest (|dwv| 100-300): they are held to the same flat bar.  Inputs follow
benchmark config 4: q, k, v ~ N(0, 1), Xavier-uniform weights, scale 1/8, dO ~ N(0, 1).
"""
import math

import pytest
import torch

from conftest import OUT_MAX_ABS, OUT_MEAN_REL, assert_out_close, seeded
from oracle import dmla_ref as R
from python import ops

NAMES = ("dq", "dk", "dv", "dwk", "dwv")
FP32 = dict(dq_dtype=torch.float32, dkv_dtype=torch.float32, dw_dtype=torch.float32)


def _inputs(B, H, Sq, Sk, seed):
    q = seeded((B, H, Sq, 64), seed, 1.0, torch.bfloat16)
    k = seeded((B, Sk, H, 128), seed + 1, 1.0, torch.bfloat16)
    v = seeded((B, Sk, H, 128), seed + 2, 1.0, torch.bfloat16)
    bound = math.sqrt(6.0 / (128 + 64))
    g = torch.Generator().manual_seed(seed + 3)
    wk = ((torch.rand(H, 128, 64, generator=g) * 2 - 1) * bound).to(torch.bfloat16)
    wv = ((torch.rand(H, 128, 64, generator=g) * 2 - 1) * bound).to(torch.bfloat16)
    do = seeded((B, H, Sq, 64), seed + 4, 1.0, torch.bfloat16)
    return q, k, v, wk, wv, do


def _run(gpu, xs, causal, scale=0.125, **kw):
    q, k, v, wk, wv, do = (t.to(gpu) for t in xs)
    o, m, l = ops.flash_dmla_fwd_onthefly(q, k, v, wk, wv, scale, causal, return_stats=True)
    grads = ops.flash_dmla_bwd_onthefly(q, k, v, wk, wv, o, do, m, l, scale, causal, **kw)
    torch.cuda.synchronize()
    return o, m, l, grads


def _check(gpu, B, H, Sq, Sk, causal, seed, ref_device="cpu", autograd=True, scale=0.125):
    xs = _inputs(B, H, Sq, Sk, seed)
    o, m, l, grads = _run(gpu, xs, causal, scale, **FP32)
    assert all(g.dtype == torch.float32 for g in grads)
    # The default dtypes: the same values, dq / dk / dv rounded to bf16 last.
    q, k, v, wk, wv, do = (t.to(gpu) for t in xs)
    dflt = ops.flash_dmla_bwd_onthefly(q, k, v, wk, wv, o, do, m, l, scale, causal)
    assert [g.dtype for g in dflt] == [torch.bfloat16] * 3 + [torch.float32] * 2
    for name, a, b in zip(NAMES, grads, dflt):
        assert torch.equal(a.to(b.dtype), b), f"{name}: default-dtype output is not the rounded fp32 one"
    dev = gpu if ref_device == "gpu" else torch.device("cpu")
    q, k, v, wk, wv, do = (t.to(dev).float() for t in xs)
    ref = R.dmla_bwd_onthefly(q, k, v, wk, wv, o.to(dev).float(), do, m.to(dev), l.to(dev), scale, causal)
    # One key: softmax is 1 wherever the key is seen and the exact dS = dP - D is 0, so the exact
    # dq, dK_lat and with it dk and dwk are 0.  What remains is rounding (D from the saved bf16 O,
    # dP from V_lat itself), in the oracle as in the kernel, so these are held to the absolute bar
    # only: mean-rel against a reference that is itself rounding noise means nothing.  dv and dwv
    # carry the gradient and keep the full bar.
    zero = ("dq", "dk", "dwk") if Sk == 1 else ()
    for name, g, r in zip(NAMES, grads, ref):
        assert tuple(g.shape) == tuple(r.shape), name
        if name in zero:
            err = (g - r.to(g.device)).abs().max().item()
            assert err <= OUT_MAX_ABS, f"{name} of a single key vs oracle backward: max-abs {err:.3e}"
            continue
        assert_out_close(g, r, f"{name} vs oracle backward")
    if autograd:
        ag = R.dmla_grads_onthefly_autograd(q, k, v, wk, wv, do, scale, causal, torch.float32)
        for name, g, r, a in zip(NAMES, grads, ref, ag):
            a = a.to(g.device)
            same_o = (r.to(g.device) - a).abs().max().item()   # the bf16 O's share, no kernel involved
            diff = (g - a).abs()
            assert diff.max().item() <= same_o + OUT_MAX_ABS, \
                f"{name} vs fp32 autograd: max-abs {diff.max().item():.3e} > {same_o:.3e} + {OUT_MAX_ABS}"
            if name in zero:
                continue
            mean_rel = (diff.mean() / a.abs().mean().clamp_min(1e-30)).item()
            assert mean_rel <= OUT_MEAN_REL, f"{name} vs fp32 autograd: mean-rel {mean_rel:.3e}"
    return grads


@pytest.mark.gpu
@pytest.mark.parametrize(
    "B,H,Sq,Sk,causal",
    [
        (1, 2, 64, 64, True),       # one key block, one row block
        (2, 3, 200, 200, True),     # ragged rows and keys, padded blocks
        (1, 2, 77, 130, True),      # Sq < Sk: bottom-right aligned causal
        (1, 2, 150, 70, True),      # Sq > Sk: the first rows see no key and get no gradient
        (2, 2, 96, 96, False),      # non-causal
        (1, 2, 100, 1100, False),   # nine 128-key weight-gradient chunks
        (1, 1, 1030, 1030, True),   # causal, the last chunk with six keys
        (1, 3, 5, 5, True),         # a handful of tokens
    ],
)
def test_otf_bwd_small_shapes(gpu, B, H, Sq, Sk, causal):
    grads = _check(gpu, B, H, Sq, Sk, causal, seed=B * 100 + H * 10 + Sq)
    if causal and Sq > Sk:
        assert torch.equal(grads[0][:, :, :Sq - Sk].cpu(), torch.zeros(B, H, Sq - Sk, 64))


@pytest.mark.gpu
@pytest.mark.parametrize(
    "B,H,Sq,Sk,seed",
    [
        (1, 2, 233, 2, 353),      # |dk| ~12, |dv| ~25, |dwk| ~50, |dwv| ~120
        (1, 2, 233, 2, 5009),
        (1, 2, 266, 2, 1),
        (1, 2, 600, 2, 7),        # |dwk| ~90, |dwv| ~130
        (1, 2, 1000, 3, 8),       # |dwv| ~180
        (1, 2, 2000, 4, 10),      # |dwk| ~130, |dwv| ~170
        (1, 4, 512, 8, 11),
    ],
)
def test_otf_bwd_large_gradients(gpu, B, H, Sq, Sk, seed):
    """A few keys seen by hundreds or thousands of rows (non-causal): the gradients of the keys
    and weights sum one term per row without averaging out.  With dwk[i, j] = sum over keys of
    k[key, i] dK_lat[key, j], whose terms often cancel, an operand rounded once to 16 bits
    (2^-11) carries an error proportional to the terms, not to their sum: in an fp64 emulation
    of fp16 operands these cases reach 0.03-0.07, over the bar; with the bf16 hi + lo operands
    of the dK/dV side the emulation stays below 1e-3.  Held to the flat bar."""
    _check(gpu, B, H, Sq, Sk, False, seed=seed)


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,Sq,causal", [(1, 2, 49, False), (1, 2, 42, False), (2, 2, 60, True), (1, 1, 173, True),
                                           (1, 2, 2000, False)])
def test_otf_bwd_single_key_many_rows(gpu, B, H, Sq, causal):
    """One key seen by many rows (causal: bottom-right aligned, so only the last row sees it).
    The exact dq, dk and dwk are 0 and what the kernel and the oracle compute for them is the
    rounding of dS = dP - D (D from the saved bf16 O): held to the absolute bar against the
    oracle, without mean-rel.  dv and dwv sum every row's dO over the single key (|dwv| ~300 at
    2000 rows) and are held to the flat bar."""
    _check(gpu, B, H, Sq, 1, causal, seed=B * 100 + H * 10 + Sq)


@pytest.mark.gpu
def test_otf_bwd_small_gradients_scale_exactly(gpu):
    """Gradients as small as training produces.  dQ's fp16 operands would turn dO ~ 1e-7 into
    subnormals; the dQ kernel scales dO, D and dS by a power of two chosen on the device from
    max |dO| and dQ back, and the dK/dV side keeps bf16's range, so dO 2^-24 yields exactly 2^-24
    times every gradient of dO, bit for bit."""
    xs = _inputs(1, 4, 256, 256, seed=43)
    small = (xs[5].float() * 2.0 ** -24).to(torch.bfloat16)   # exact: a power of two
    _, _, _, grads = _run(gpu, xs, True, **FP32)
    _, _, _, grads_s = _run(gpu, xs[:5] + (small,), True, **FP32)
    for name, a, b in zip(NAMES, grads, grads_s):
        assert a.abs().max().item() > 0.01, name
        assert torch.equal(b * 2.0 ** 24, a), f"{name} of a scaled dO"


@pytest.mark.gpu
def test_otf_bwd_zero_output_gradient_gives_zero(gpu):
    """dO = 0: every gradient of the on-the-fly backward is exactly 0."""
    xs = _inputs(1, 2, 130, 130, seed=47)
    _, _, _, grads = _run(gpu, xs[:5] + (torch.zeros_like(xs[5]),), True, **FP32)
    for name, t in zip(NAMES, grads):
        assert int(torch.count_nonzero(t)) == 0, name


@pytest.mark.gpu
def test_otf_bwd_single_token(gpu):
    """One key: softmax is constant, so the exact dq, dk and dwk are 0 and dS = dP - D is pure
    rounding (the recomputed V_lat against the bf16 O); they must stay small, while dv = dO and
    dwv = v^T dO are checked at the bar."""
    xs = _inputs(1, 2, 1, 1, 5)
    _, _, _, grads = _run(gpu, xs, True, **FP32)
    q, k, v, wk, wv, do = (t.float() for t in xs)
    ag = R.dmla_grads_onthefly_autograd(q, k, v, wk, wv, do, 0.125, True, torch.float32)
    for name, g, a in zip(NAMES, grads, ag):
        if name in ("dq", "dk", "dwk"):
            assert a.abs().max().item() == 0.0
            assert g.abs().max().item() <= OUT_MAX_ABS, name
        else:
            assert_out_close(g, a, name)


@pytest.mark.gpu
def test_otf_bwd_config4_shape(gpu):
    """benchmark config 4 at full size (B=2, H=32, S=4096), oracle on the GPU in fp32."""
    _check(gpu, 2, 32, 4096, 4096, True, seed=4, ref_device="gpu", autograd=False)


@pytest.mark.gpu
def test_otf_bwd_config4_autograd_heads(gpu):
    """Full sequence length on 4 heads against fp32 autograd on the GPU."""
    _check(gpu, 2, 4, 4096, 4096, True, seed=44, ref_device="gpu")


@pytest.mark.gpu
def test_otf_bwd_deterministic_and_bf16_weights(gpu):
    xs = _inputs(1, 4, 300, 300, 7)
    _, _, _, g1 = _run(gpu, xs, True)
    _, _, _, g2 = _run(gpu, xs, True)
    for name, a, b in zip(NAMES, g1, g2):
        assert torch.equal(a, b), f"{name} differs between identical calls"
    _, _, _, g3 = _run(gpu, xs, True, dw_dtype=torch.bfloat16)
    for name, a, b in zip(NAMES, g1, g3):
        assert b.dtype == torch.bfloat16
        assert torch.equal(a.to(torch.bfloat16), b), f"{name}: bf16 output is not the rounded fp32 one"


@pytest.mark.gpu
def test_otf_autograd_function(gpu):
    xs = _inputs(1, 2, 140, 140, 11)
    leaves = [t.to(gpu).requires_grad_(True) for t in xs[:5]]
    o = ops.flash_dmla_onthefly(*leaves, 0.125, True)
    o.backward(xs[5].to(gpu))
    _, _, _, grads = _run(gpu, xs, True)
    for name, leaf, g in zip(NAMES, leaves, grads):
        assert leaf.grad is not None and leaf.grad.dtype == torch.bfloat16, name
        assert torch.equal(leaf.grad, g.to(torch.bfloat16)), f"{name}: autograd differs from the direct call"


@pytest.mark.gpu
def test_otf_bwd_strided_inputs(gpu):
    """Non-contiguous views: k, v inside a wider [B, Sk, H, 2*128] buffer, q/o/do head-major views."""
    B, H, Sq, Sk = 1, 2, 96, 96
    q, k, v, wk, wv, do = _inputs(B, H, Sq, Sk, 13)
    kv = torch.cat([k, v], dim=-1).to(gpu)
    kg, vg = kv[..., :128], kv[..., 128:]
    qg = q.transpose(1, 2).contiguous().to(gpu).transpose(1, 2)      # [B, H, Sq, 64] with seq-major storage
    dog = do.transpose(1, 2).contiguous().to(gpu).transpose(1, 2)
    o, m, l = ops.flash_dmla_fwd_onthefly(qg, kg, vg, wk.to(gpu), wv.to(gpu), 0.125, True, return_stats=True)
    grads = ops.flash_dmla_bwd_onthefly(qg, kg, vg, wk.to(gpu), wv.to(gpu), o, dog, m, l, 0.125, True)
    _, _, _, ref = _run(gpu, (q, k, v, wk, wv, do), True)
    for name, a, b in zip(NAMES, grads, ref):
        assert torch.equal(a, b), f"{name}: strided inputs change the result"


def _wgrad_chunk(gpu, B, H, Sk):
    """Keys per weight-gradient workgroup: 1024, halved down to 128 while that leaves less than two per CU."""
    cus = torch.cuda.get_device_properties(gpu).multi_processor_count
    chunk = 1024
    while chunk > 128 and 2 * B * H * -(-Sk // chunk) < 2 * cus:
        chunk //= 2
    return chunk


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,Sq,Sk", [(1, 2, 200, 700), (2, 1, 70, 1500)])
def test_otf_bwd_smaller_workspace(gpu, B, H, Sq, Sk):
    """The query's workspace holds a partial per chunk of the length that fills the device; one that holds
    only the partials of 1024-key chunks (its size on any device) runs with those, a byte less is
    refused.  dq, dk and dv do not depend on the chunks; the weight gradients are the same fp32 sums in
    another order, Sk terms of at most ~1e2 that add to values of that size: 1e-3 absolute is > 100 ulps."""
    from python import _lib
    q, k, v, wk, wv, do = (t.to(gpu) for t in _inputs(B, H, Sq, Sk, seed=Sk))
    o, m, l = ops.flash_dmla_fwd_onthefly(q, k, v, wk, wv, 0.125, True, return_stats=True)
    ref = ops.flash_dmla_bwd_onthefly(q, k, v, wk, wv, o, do, m, l, 0.125, True)
    chunks = -(-Sk // _wgrad_chunk(gpu, B, H, Sk))
    need = _lib.lib().dmla_bwd_onthefly_workspace_bytes(B, H, Sq, Sk, 128, 64)
    least = need - 65536 * B * H * (chunks - -(-Sk // 1024))
    assert least < need

    def call(ws_bytes):
        out = [torch.full_like(t, float("nan")) for t in ref]
        ws = torch.empty((ws_bytes,), dtype=torch.uint8, device=gpu)
        P, st = ops._ptr, lambda t: tuple(t.stride())
        rc = _lib.lib().dmla_bwd_onthefly(
            *map(P, (q, k, v, wk, wv, o, do, m, l)), *map(P, out), B, H, Sq, Sk, 128, 64, *st(q)[:3], *st(k)[:3],
            *st(v)[:3], *st(wk)[:2], *st(o)[:3], *st(do)[:3], *st(out[0])[:3], *st(out[1])[:3], *st(out[3])[:2],
            0, 0, 1, 0.125, 1, P(ws), ws_bytes, ops._stream(q))
        return rc, out

    assert call(least - 1)[0] == _lib.DMLA_ERR_WORKSPACE
    for ws_bytes in (least, need - 1):
        rc, out = call(ws_bytes)
        assert rc == _lib.DMLA_OK
        for name, a, b in zip(NAMES[:3], out, ref):
            assert torch.equal(a, b), name
        for name, a, b in zip(NAMES[3:], out[3:], ref[3:]):
            assert (a - b).abs().max().item() <= 1e-3, name


@pytest.mark.gpu
@pytest.mark.parametrize(
    "B,H,Sq,Sk,causal,chunk",
    [
        (8, 32, 5, 1100, False, 1024),    # two chunks, the last one a whole 64-key block and 12 keys
        (8, 32, 3, 1024, True, 1024),     # one whole chunk
        (2, 32, 5, 1700, False, 512),     # four chunks, the last one ragged
        (2, 32, 9, 1100, True, 256),      # five chunks, the last one ragged
        (1, 32, 40, 777, True, 128),      # seven chunks, the last one with nine keys
    ],
)
def test_otf_bwd_weight_gradient_chunks(gpu, B, H, Sq, Sk, causal, chunk):
    """Every chunk length of the weight-gradient kernel, its serial loop over 64-key blocks up to a
    ragged end, in fp32 and with the 16-byte bf16 dK / dV stores (the default dtypes, compared bit
    for bit with the rounded fp32 ones)."""
    assert _wgrad_chunk(gpu, B, H, Sk) == chunk
    _check(gpu, B, H, Sq, Sk, causal, seed=Sk + chunk, ref_device="gpu", autograd=False)
