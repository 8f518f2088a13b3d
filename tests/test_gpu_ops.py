"""GPU parity tests of every C-ABI operator against the CPU oracle on identical seeded
inputs (ctypes through include/edgefm_hip.h). Shapes are the BASELINE head / layer
shapes: Qwen2.5-0.5B (14/2, hd 64), 1.5B (12/2, hd 128), 3B (16/2), 7B (28/4).
Mirrors tests/operators/test_attention_decode.py, test_norm_sampler.py,
test_decode_linear.py and test_fused_gate_up_activation.py of the reference."""
import math

import numpy as np
import pytest
import torch

import efm_capi as C
from oracle import efm_oracle as O
from _util import assert_close_bf16, ptr, stream

pytestmark = pytest.mark.gpu

HEAD_CASES = [
    pytest.param(14, 2, 64, id="0p5b"),
    pytest.param(12, 2, 128, id="1p5b"),
    pytest.param(16, 2, 128, id="3b"),
    pytest.param(28, 4, 128, id="7b"),
]


def _decode(ctx, q, k, v, kv_len, d_kv_len=None, max_kv_len=0):
    ws_bytes = C.load().efm_attention_decode_workspace_bytes(ctx, max_kv_len if d_kv_len is not None else kv_len)
    ws = torch.zeros(max(ws_bytes, 256), dtype=torch.uint8, device=q.device)
    o = torch.empty_like(q)
    C.call("efm_attention_decode", ctx, ptr(q), ptr(k), ptr(v), ptr(o), kv_len, ptr(d_kv_len), max_kv_len,
           ptr(ws), ws.numel(), stream())
    torch.cuda.synchronize()
    return o, ws


@pytest.mark.parametrize("hq,hkv,hd", HEAD_CASES)
@pytest.mark.parametrize("kv_len", [1, 7, 33, 512, 1024, 2048])
def test_attention_decode_matches_oracle(gpu, hq, hkv, hd, kv_len):
    torch.manual_seed(0)
    q = torch.randn(1, hq, hd, dtype=torch.bfloat16)
    k = torch.randn(kv_len, hkv, hd, dtype=torch.bfloat16)
    v = torch.randn(kv_len, hkv, hd, dtype=torch.bfloat16)
    ref = O.attention_decode(q, k, v, kv_len, O.AttnCtx(hq, hkv, hd))
    ctx = C.make_attention_ctx(hq, hkv, hd)
    out, _ = _decode(ctx, q.to(gpu), k.to(gpu), v.to(gpu), kv_len)
    assert_close_bf16(out, ref, what=f"decode hq={hq} hkv={hkv} hd={hd} kv={kv_len}")


@pytest.mark.parametrize("hq,hkv,hd", [pytest.param(28, 4, 128, id="7b")])
def test_attention_decode_long_context(gpu, hq, hkv, hd):
    torch.manual_seed(1)
    kv_len = 16385
    q = torch.randn(1, hq, hd, dtype=torch.bfloat16)
    k = torch.randn(kv_len, hkv, hd, dtype=torch.bfloat16)
    v = torch.randn(kv_len, hkv, hd, dtype=torch.bfloat16)
    ref = O.attention_decode(q, k, v, kv_len, O.AttnCtx(hq, hkv, hd))
    out, _ = _decode(C.make_attention_ctx(hq, hkv, hd), q.to(gpu), k.to(gpu), v.to(gpu), kv_len)
    assert_close_bf16(out, ref, what="decode 16k")


@pytest.mark.parametrize("hq,hkv,hd", HEAD_CASES)
@pytest.mark.parametrize("kv_len", [512, 1024, 2048])
def test_attention_decode_graph_like_path_matches_plain(gpu, hq, hkv, hd, kv_len):
    """d_kv_len + max_kv_len over a larger cache == plain call on the first kv_len rows
    (tests/operators/test_attention_decode.py:155-179). Called twice to check that the
    in-workspace merge counters reset themselves."""
    torch.manual_seed(0)
    max_kv = 2048
    q = torch.randn(1, hq, hd, dtype=torch.bfloat16, device=gpu)
    k = torch.randn(max_kv, hkv, hd, dtype=torch.bfloat16, device=gpu)
    v = torch.randn(max_kv, hkv, hd, dtype=torch.bfloat16, device=gpu)
    ctx = C.make_attention_ctx(hq, hkv, hd)
    d_len = torch.tensor([kv_len], dtype=torch.int32, device=gpu)
    ws_bytes = C.load().efm_attention_decode_workspace_bytes(ctx, max_kv)
    ws = torch.zeros(ws_bytes, dtype=torch.uint8, device=gpu)
    outs = []
    for _ in range(2):
        o = torch.empty_like(q)
        C.call("efm_attention_decode", ctx, ptr(q), ptr(k), ptr(v), ptr(o), 0, ptr(d_len), max_kv, ptr(ws),
               ws.numel(), stream())
        torch.cuda.synchronize()
        outs.append(o)
    plain, _ = _decode(ctx, q, k[:kv_len].contiguous(), v[:kv_len].contiguous(), kv_len)
    assert_close_bf16(outs[0], plain)
    assert torch.equal(outs[0], outs[1])


def test_attention_decode_no_rope_and_prerotated(gpu):
    """pos_encoding NONE equals plain softmax attention; k_already_prerotated with
    pre-rotated K equals RoPE-on-read (tests/operators/test_attention_prefill.py:118-164)."""
    torch.manual_seed(3)
    hq, hkv, hd, L = 12, 2, 128, 300
    q = torch.randn(1, hq, hd, dtype=torch.bfloat16)
    k = torch.randn(L, hkv, hd, dtype=torch.bfloat16)
    v = torch.randn(L, hkv, hd, dtype=torch.bfloat16)
    ref = O.attention_decode(q, k, v, L, O.AttnCtx(hq, hkv, hd, rope=False))
    out, _ = _decode(C.make_attention_ctx(hq, hkv, hd, rope=False), q.to(gpu), k.to(gpu), v.to(gpu), L)
    assert_close_bf16(out, ref, what="no-rope")
    k_rot = O.rope_llama(k, torch.arange(L), 1.0e6).to(torch.bfloat16)
    rot_ref = O.attention_decode(q, k, v, L, O.AttnCtx(hq, hkv, hd))
    out2, _ = _decode(C.make_attention_ctx(hq, hkv, hd, k_already_prerotated=True), q.to(gpu), k_rot.to(gpu),
                      v.to(gpu), L)
    assert_close_bf16(out2, rot_ref, what="prerotated")


@pytest.mark.parametrize("hq,hkv,hd", HEAD_CASES)
@pytest.mark.parametrize("kv_len", [1, 129, 767, 1025, 4099])
@pytest.mark.parametrize("merge", [True, False])
def test_attention_decode_prerotated_except_newest(gpu, hq, hkv, hd, kv_len, merge):
    """EFM_K_PREROTATED_EXCEPT_NEWEST: rows [0, L-1) hold rotated keys, row L-1 the
    un-rotated key of this step. The output equals RoPE-on-read over the un-rotated cache
    (and the oracle), row L-1 is stored back rotated (within one bf16 rounding of the
    oracle's rotation) and no other row changes. Rows >= L of the max_kv_len allocation
    hold NaN: the split loads issued before the length is read must not leak them."""
    torch.manual_seed(kv_len)
    max_kv = kv_len + 77
    q = torch.randn(1, hq, hd, dtype=torch.bfloat16)
    k = torch.randn(kv_len, hkv, hd, dtype=torch.bfloat16)
    v = torch.randn(kv_len, hkv, hd, dtype=torch.bfloat16)
    ref = O.attention_decode(q, k, v, kv_len, O.AttnCtx(hq, hkv, hd))
    k_rot = O.rope_llama(k, torch.arange(kv_len), 1.0e6).to(torch.bfloat16)
    kc = torch.full((max_kv, hkv, hd), float("nan"), dtype=torch.bfloat16)
    vc = torch.full((max_kv, hkv, hd), float("nan"), dtype=torch.bfloat16)
    kc[: kv_len - 1] = k_rot[: kv_len - 1]
    kc[kv_len - 1] = k[kv_len - 1]
    vc[:kv_len] = v
    kc, vc, qg = kc.to(gpu), vc.to(gpu), q.to(gpu)
    ctx = C.make_attention_ctx(hq, hkv, hd)
    ctx.k_already_prerotated = C.EFM_K_PREROTATED_EXCEPT_NEWEST
    d_len = torch.tensor([kv_len], dtype=torch.int32, device=gpu)
    ws = torch.zeros(C.load().efm_attention_decode_workspace_bytes(ctx, max_kv), dtype=torch.uint8, device=gpu)
    if merge:
        o = torch.empty_like(qg)
        C.call("efm_attention_decode", ctx, ptr(qg), ptr(kc), ptr(vc), ptr(o), 0, ptr(d_len), max_kv, ptr(ws),
               ws.numel(), stream())
        torch.cuda.synchronize()
        assert_close_bf16(o, ref, what=f"prerotated-except-newest L={kv_len}")
        plain, _ = _decode(C.make_attention_ctx(hq, hkv, hd), qg, k.to(gpu), v.to(gpu), kv_len)
        assert_close_bf16(o, plain, what="vs rope-on-read")
    else:
        C.call("efm_decode_attention_partials", ctx, ptr(qg), ptr(kc), ptr(vc), ptr(d_len), max_kv, ptr(ws),
               ws.numel(), stream())
        torch.cuda.synchronize()
    got = kc.cpu()
    assert torch.equal(got[: kv_len - 1], k_rot[: kv_len - 1]), "rows before the newest must not change"
    assert torch.isnan(got[kv_len:].float()).all(), "rows past L must not be written"
    assert_close_bf16(got[kv_len - 1], k_rot[kv_len - 1], rtol=1e-2, atol=1e-2, what="newest row stored rotated")


@pytest.mark.parametrize("hq,hkv,hd", HEAD_CASES)
@pytest.mark.parametrize("kv_len,max_kv", [(1, 64), (31, 31), (33, 700), (640, 768), (1025, 1100), (3000, 3000),
                                           (5000, 5000)])
@pytest.mark.parametrize("layout", ["rope_on_read", "rotated_except_newest", "no_rope"])
def test_attention_decode_one_wave_splits(gpu, knob, hq, hkv, hd, kv_len, max_kv, layout):
    """The one-wave split kernel of short and mid contexts (32- and 64-key splits, a
    partial last tile, a single split that writes the output itself) against the oracle
    and against the kernels those lengths ran before it (EFM_KNOB_DECODE_TILE), over the
    three cache layouts: un-rotated keys rotated on read (the reference's), rotated keys
    with this step's row still un-rotated (the engine's), and no RoPE (M-RoPE models).
    Rows >= L hold NaN."""
    torch.manual_seed(kv_len * 7 + hd)
    q = torch.randn(1, hq, hd, dtype=torch.bfloat16)
    k = torch.randn(kv_len, hkv, hd, dtype=torch.bfloat16)
    v = torch.randn(kv_len, hkv, hd, dtype=torch.bfloat16)
    rope = layout != "no_rope"
    ref = O.attention_decode(q, k, v, kv_len, O.AttnCtx(hq, hkv, hd, rope=rope))
    kstore = k
    if layout == "rotated_except_newest":
        kstore = O.rope_llama(k, torch.arange(kv_len), 1.0e6).to(torch.bfloat16)
        kstore[kv_len - 1] = k[kv_len - 1]
    ctx = C.make_attention_ctx(hq, hkv, hd, rope=rope)
    if layout == "rotated_except_newest":
        ctx.k_already_prerotated = C.EFM_K_PREROTATED_EXCEPT_NEWEST
    d_len = torch.tensor([kv_len], dtype=torch.int32, device=gpu)
    ws = torch.zeros(C.load().efm_attention_decode_workspace_bytes(ctx, max_kv), dtype=torch.uint8, device=gpu)
    qg = q.to(gpu)
    outs, caches = [], []
    for tile_off in (0, 1):
        knob(C.EFM_KNOB_DECODE_TILE, tile_off)
        kc = torch.full((max_kv, hkv, hd), float("nan"), dtype=torch.bfloat16)
        vc = torch.full((max_kv, hkv, hd), float("nan"), dtype=torch.bfloat16)
        kc[:kv_len] = kstore
        vc[:kv_len] = v
        kc, vc = kc.to(gpu), vc.to(gpu)
        o = torch.empty_like(qg)
        C.call("efm_attention_decode", ctx, ptr(qg), ptr(kc), ptr(vc), ptr(o), 0, ptr(d_len), max_kv, ptr(ws),
               ws.numel(), stream())
        torch.cuda.synchronize()
        outs.append(o)
        caches.append(kc.cpu())
    what = f"{layout} hq={hq} hkv={hkv} hd={hd} L={kv_len}"
    assert torch.isfinite(outs[0].float()).all(), what
    assert_close_bf16(outs[0], ref, what="one-wave splits vs oracle, " + what)
    assert_close_bf16(outs[0], outs[1], what="one-wave splits vs previous kernels, " + what)
    if layout == "rotated_except_newest":
        # the newest row is stored back rotated the same way by both paths; no other row moves
        assert torch.equal(caches[0][: kv_len - 1], kstore[: kv_len - 1])
        assert torch.isnan(caches[0][kv_len:].float()).all()
        assert torch.equal(caches[0][kv_len - 1], caches[1][kv_len - 1])
    else:
        assert torch.equal(caches[0][:kv_len], kstore), "the call must not write the cache"


def test_attention_decode_partials_ignore_stale_rows(gpu):
    """Rows >= L of the cache hold NaN / Inf; the partials + merge path must give the
    same result as a cache that ends at L."""
    torch.manual_seed(9)
    hq, hkv, hd, L, max_kv = 12, 2, 128, 300, 1024
    q = torch.randn(1, hq, hd, dtype=torch.bfloat16, device=gpu)
    k = torch.randn(max_kv, hkv, hd, dtype=torch.bfloat16, device=gpu)
    v = torch.randn(max_kv, hkv, hd, dtype=torch.bfloat16, device=gpu)
    k[L:] = float("inf")
    v[L:] = float("nan")
    ctx = C.make_attention_ctx(hq, hkv, hd)
    d_len = torch.tensor([L], dtype=torch.int32, device=gpu)
    ws = torch.zeros(C.load().efm_attention_decode_workspace_bytes(ctx, max_kv), dtype=torch.uint8, device=gpu)
    o = torch.empty_like(q)
    C.call("efm_attention_decode", ctx, ptr(q), ptr(k), ptr(v), ptr(o), 0, ptr(d_len), max_kv, ptr(ws), ws.numel(),
           stream())
    torch.cuda.synchronize()
    ref = O.attention_decode(q.cpu(), k[:L].cpu(), v[:L].cpu(), L, O.AttnCtx(hq, hkv, hd))
    assert torch.isfinite(o.float()).all()
    assert_close_bf16(o, ref)


@pytest.mark.parametrize("S,base,hq,hkv,hd", [(37, 0, 12, 2, 128), (5, 1000, 14, 2, 64), (300, 16000, 28, 4, 128)])
def test_rope_llama_inplace_matches_oracle(gpu, S, base, hq, hkv, hd):
    """Q in a fused QKV buffer (token stride) and K rows rotated in place at positions
    base + t; one bf16 rounding of the oracle's fp32 rotation."""
    torch.manual_seed(S)
    tot = (hq + 2 * hkv) * hd
    qkv = torch.randn(S, tot, dtype=torch.bfloat16)
    kc = torch.randn(S, hkv, hd, dtype=torch.bfloat16)
    pos = base + torch.arange(S)
    want_q = O.rope_llama(qkv[:, : hq * hd].reshape(S, hq, hd), pos, 1.0e6).to(torch.bfloat16)
    want_k = O.rope_llama(kc, pos, 1.0e6).to(torch.bfloat16)
    qkv_g, kc_g = qkv.to(gpu), kc.to(gpu)
    C.call("efm_rope_llama_inplace", ptr(qkv_g), ptr(kc_g), S, hq, hkv, hd, tot, hkv * hd, base, 1.0e6, 1.0,
           stream())
    torch.cuda.synchronize()
    got = qkv_g.cpu()
    assert_close_bf16(got[:, : hq * hd].reshape(S, hq, hd), want_q, rtol=1e-2, atol=1e-2, what="q")
    assert torch.equal(got[:, hq * hd:], qkv[:, hq * hd:]), "K/V columns of the QKV buffer untouched"
    assert_close_bf16(kc_g, want_k, rtol=1e-2, atol=1e-2, what="k")


@pytest.mark.parametrize("mode,S,base,hq,hkv,hd", [
    ("text", 77, 0, 12, 2, 128), ("text", 300, 513, 28, 4, 128), ("text", 33, 5, 14, 2, 64),
    ("mrope", 70, 0, 16, 2, 128),
])
def test_prefill_rope_write_kv_matches_two_step_and_oracle(gpu, mode, S, base, hq, hkv, hd):
    """One-pass q rotation + rotated K / raw V into the cache rows equals the two-step
    path (K / V copies, then efm_rope_llama_inplace or efm_mrope over the cache rows) bit
    for bit, and the oracle's rotation within one bf16 rounding; cache rows outside
    [base, base + S) and the QKV buffer's K / V columns stay untouched."""
    torch.manual_seed(S + hd)
    kvd, qd = hkv * hd, hq * hd
    tot = qd + 2 * kvd
    rows = base + S + 9
    qkv = torch.randn(S, tot, dtype=torch.bfloat16)
    kc0 = torch.randn(rows, kvd, dtype=torch.bfloat16)
    vc0 = torch.randn(rows, kvd, dtype=torch.bfloat16)
    if mode == "mrope":
        sections = (16, 24, 24)
        pos = (torch.stack([torch.zeros(S, dtype=torch.int32), torch.arange(S, dtype=torch.int32) // 7,
                            torch.arange(S, dtype=torch.int32) % 7]) + 3).contiguous()
        pos_g = pos.to(gpu)
    else:
        sections, pos_g = (hd // 2, 0, 0), None
    # one pass
    q1, k1, v1 = qkv.to(gpu), kc0.to(gpu), vc0.to(gpu)
    C.call("efm_prefill_rope_write_kv", ptr(q1), tot, ptr(k1[base:]), ptr(v1[base:]), kvd, S, hq, hkv, hd,
           ptr(pos_g), S, base if mode == "text" else 0, *sections, 1.0e6, 1.0, stream())
    # two steps
    q2, k2, v2 = qkv.to(gpu), kc0.to(gpu), vc0.to(gpu)
    k2[base:base + S] = q2[:, qd:qd + kvd]
    v2[base:base + S] = q2[:, qd + kvd:]
    if mode == "mrope":
        C.call("efm_mrope", ptr(q2), ptr(k2[base:]), ptr(pos_g), S, S, hq, hkv, hd, tot, kvd, *sections, 1.0e6,
               1.0, stream())
    else:
        C.call("efm_rope_llama_inplace", ptr(q2), ptr(k2[base:]), S, hq, hkv, hd, tot, kvd, base, 1.0e6, 1.0,
               stream())
    torch.cuda.synchronize()
    assert torch.equal(q1, q2) and torch.equal(k1, k2) and torch.equal(v1, v2), "differs from the two-step path"
    assert torch.equal(k1[:base].cpu(), kc0[:base]) and torch.equal(k1[base + S:].cpu(), kc0[base + S:])
    assert torch.equal(q1[:, qd:].cpu(), qkv[:, qd:]), "K / V columns of the QKV buffer untouched"
    if mode == "mrope":
        want_q = O.mrope(qkv[:, :qd].reshape(S, hq, hd), pos, sections, 1.0e6)
        want_k = O.mrope(qkv[:, qd:qd + kvd].reshape(S, hkv, hd), pos, sections, 1.0e6)
    else:
        p = base + torch.arange(S)
        want_q = O.rope_llama(qkv[:, :qd].reshape(S, hq, hd), p, 1.0e6).to(torch.bfloat16)
        want_k = O.rope_llama(qkv[:, qd:qd + kvd].reshape(S, hkv, hd), p, 1.0e6).to(torch.bfloat16)
    assert_close_bf16(q1[:, :qd].reshape(S, hq, hd), want_q, rtol=1e-2, atol=1e-2, what="q")
    assert_close_bf16(k1[base:base + S].reshape(S, hkv, hd), want_k, rtol=1e-2, atol=1e-2, what="k")
    assert torch.equal(v1[base:base + S].cpu(), qkv[:, qd + kvd:]), "V rows copied"


def test_attention_decode_strided_views(gpu):
    """q read from a fused QKV row and K/V from strided views equals contiguous inputs
    (tests/operators/test_attention_prefill.py:167-300)."""
    torch.manual_seed(4)
    hq, hkv, hd, L = 12, 2, 128, 257
    qkv = torch.randn(1, (hq + 2 * hkv) * hd, dtype=torch.bfloat16, device=gpu)
    kv = torch.randn(L, 2, hkv, hd, dtype=torch.bfloat16, device=gpu)  # interleaved K/V rows
    q = qkv[:, : hq * hd].reshape(1, hq, hd)
    k = kv[:, 0]
    v = kv[:, 1]
    ctx = C.make_attention_ctx(hq, hkv, hd, q_stride_n=(hq + 2 * hkv) * hd, q_stride_h=hd,
                               k_stride_n=2 * hkv * hd, k_stride_h=hd, kv_stride_n=2 * hkv * hd, kv_stride_h=hd)
    ws = torch.zeros(C.load().efm_attention_decode_workspace_bytes(ctx, L), dtype=torch.uint8, device=gpu)
    o = torch.empty(1, hq, hd, dtype=torch.bfloat16, device=gpu)
    C.call("efm_attention_decode", ctx, qkv.data_ptr(), kv.data_ptr(), kv[:, 1].data_ptr(), ptr(o), L, None, 0,
           ptr(ws), ws.numel(), stream())
    torch.cuda.synchronize()
    ref, _ = _decode(C.make_attention_ctx(hq, hkv, hd), q.contiguous(), k.contiguous(), v.contiguous(), L)
    assert_close_bf16(o, ref)


def test_attention_decode_rejects_unsupported(gpu):
    ctx = C.make_attention_ctx(10, 2, 128)  # group size 5
    with pytest.raises(C.EfmError) as e:
        C.call("efm_attention_decode", ctx, 1, 1, 1, 1, 1, None, 0, 1, 1 << 20, stream())
    assert e.value.code == C.EFM_ERR_UNSUPPORTED


@pytest.mark.parametrize("batch,hidden", [(1, 896), (1, 1536), (4, 2048), (7, 3584), (512, 1536)])
def test_rms_norm_and_fused_add(gpu, batch, hidden):
    torch.manual_seed(0)
    x = torch.randn(batch, hidden, dtype=torch.bfloat16)
    r = torch.randn(batch, hidden, dtype=torch.bfloat16)
    w = (1 + 0.1 * torch.randn(hidden)).to(torch.bfloat16)
    eps = 1e-6
    xg, rg, wg = x.to(gpu), r.to(gpu), w.to(gpu)
    out = torch.empty_like(xg)
    C.call("efm_rms_norm", batch, hidden, eps, ptr(xg), ptr(wg), ptr(out), stream())
    torch.cuda.synchronize()
    assert_close_bf16(out, O.rms_norm(x, w, eps), what="rms_norm")
    C.call("efm_fused_add_rms_norm", batch, hidden, eps, ptr(xg), ptr(rg), ptr(wg), stream())
    torch.cuda.synchronize()
    ref_out, ref_res = O.fused_add_rms_norm(x, r, w, eps)
    assert torch.equal(rg.cpu(), ref_res), "residual must be bf16(x + r) exactly"
    assert_close_bf16(xg, ref_out, what="fused_add_rms_norm")


@pytest.mark.parametrize("layout", [C.EFM_LAYOUT_UP_GATE, C.EFM_LAYOUT_GATE_UP])
@pytest.mark.parametrize("batch,inter", [(1, 4864), (1, 8960), (5, 11008)])
def test_act_and_mul(gpu, layout, batch, inter):
    torch.manual_seed(0)
    x = torch.randn(batch, 2 * inter, dtype=torch.bfloat16) * 3
    out = torch.empty(batch, inter, dtype=torch.bfloat16, device=gpu)
    xg = x.to(gpu)
    C.call("efm_act_and_mul", batch, inter, layout, ptr(xg), ptr(out), stream())
    torch.cuda.synchronize()
    ref = O.act_and_mul(x, up_first=(layout == C.EFM_LAYOUT_UP_GATE))
    # the north star's per-operator bound (2e-2 / 2e-2; the reference's own test allows
    # atol 6.25e-2, tests/operators/test_fused_gate_up_activation.py:75-79)
    assert_close_bf16(out, ref, rtol=2e-2, atol=2e-2)


@pytest.mark.parametrize("up", [1.0, 0.7421875, -1.3984375, 3.0])
def test_act_and_mul_every_bf16_gate(gpu, up):
    """Every bf16 gate value (signed zeros, infinities and NaNs included) through the
    kernels' silu, against the oracle's g / (1 + exp(-g)): bf16(silu(g) * up) is the same
    bf16 value except for a handful of 1-ulp roundings and, for g in (-88.7, -87.3), results
    under 1e-35 that come out as zeros of the same sign."""
    g = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)
    n = g.numel()
    x = torch.cat([torch.full((n,), up, dtype=torch.bfloat16), g]).reshape(1, 2 * n)
    xg = x.to(gpu)
    out = torch.empty(1, n, dtype=torch.bfloat16, device=gpu)
    C.call("efm_act_and_mul", 1, n, C.EFM_LAYOUT_UP_GATE, ptr(xg), ptr(out), stream())
    torch.cuda.synchronize()
    o, ref = out.cpu().flatten(), O.act_and_mul(x, up_first=True).flatten()
    of, rf = o.float(), ref.float()
    same = (o.view(torch.int16) == ref.view(torch.int16)) | (torch.isnan(of) & torch.isnan(rf))
    bad = (~same).nonzero().flatten()
    tiny = (rf[bad].abs() < 1e-35) & (of[bad] == 0) & (torch.signbit(of[bad]) == torch.signbit(rf[bad]))
    assert tiny.sum() <= 3 and bool(((g[bad].float() > -88.75) & (g[bad].float() < -87.25))[tiny].all())
    near = bad[~tiny]
    assert near.numel() <= 4, [(float(g[i]), float(o[i]), float(ref[i])) for i in near[:8]]
    assert bool(((o.view(torch.int16)[near].int() - ref.view(torch.int16)[near].int()).abs() == 1).all())
    assert torch.signbit(of[g.float() == 0]).tolist() == torch.signbit(rf[g.float() == 0]).tolist()


LINEAR_CASES = [
    pytest.param(1536, 2048, True, id="1p5b_qkv"),
    pytest.param(1536, 1536, False, id="1p5b_o"),
    pytest.param(8960, 1536, False, id="1p5b_down"),
    pytest.param(896, 1152, True, id="0p5b_qkv"),
    pytest.param(4864, 896, False, id="0p5b_down"),
    pytest.param(18944, 3584, False, id="7b_down"),
    pytest.param(3584, 4608, True, id="7b_qkv"),
]


@pytest.mark.parametrize("k,n,bias", LINEAR_CASES)
@pytest.mark.parametrize("m", [1, 3, 64, 512])
def test_linear(gpu, k, n, bias, m):
    torch.manual_seed(0)
    x = torch.randn(m, k, dtype=torch.bfloat16)
    w = (torch.randn(n, k) * 0.02).to(torch.bfloat16)
    b = (torch.randn(n) * 0.02).to(torch.bfloat16) if bias else None
    y = torch.empty(m, n, dtype=torch.bfloat16, device=gpu)
    xg, wg, bg = x.to(gpu), w.to(gpu), (b.to(gpu) if bias else None)
    C.call("efm_linear", m, k, n, ptr(xg), ptr(wg), ptr(bg), ptr(y), C.EFM_DTYPE_BF16, stream())
    torch.cuda.synchronize()
    assert_close_bf16(y, O.linear(x, w, b), what=f"linear m={m}")


@pytest.mark.parametrize("m", [1, 17])
def test_linear_fp32_logits(gpu, m):
    torch.manual_seed(0)
    k, n = 1536, 151936
    x = torch.randn(m, k, dtype=torch.bfloat16)
    w = (torch.randn(n, k) * 0.02).to(torch.bfloat16)
    y = torch.empty(m, n, dtype=torch.float32, device=gpu)
    xg, wg = x.to(gpu), w.to(gpu)
    C.call("efm_linear", m, k, n, ptr(xg), ptr(wg), None, ptr(y), C.EFM_DTYPE_F32, stream())
    torch.cuda.synchronize()
    torch.testing.assert_close(y.cpu(), O.linear(x, w, out_f32=True), rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("m,k,n,bias,kind", [
    pytest.param(4100, 1024, 12345, True, "bf16", id="ragged_bias"),
    pytest.param(6144, 1536, 8192, False, "bf16", id="1p5b_like"),
    pytest.param(4096, 2048, 11008, False, "swiglu", id="vl3b_gate_up"),
    pytest.param(300, 1536, 151936, False, "f32", id="logits_f32"),
])
def test_gemm_large_shapes_row_sample_vs_oracle(gpu, m, k, n, bias, kind):
    """Large and ragged prefill shapes (partial edge tiles in M and N) against the oracle
    on a row sample."""
    torch.manual_seed(m + n)
    x = torch.randn(m, k, dtype=torch.bfloat16, device=gpu)
    nw = 2 * n if kind == "swiglu" else n
    w = (torch.randn(nw, k, device=gpu) * 0.05).to(torch.bfloat16)
    b = (torch.randn(n, device=gpu) * 0.05).to(torch.bfloat16) if bias else None
    if kind == "swiglu":
        y = torch.empty(m, n, dtype=torch.bfloat16, device=gpu)
        C.call("efm_fused_gate_up_swiglu", m, k, n, ptr(x), ptr(w), ptr(y), stream())
    else:
        dt = torch.float32 if kind == "f32" else torch.bfloat16
        y = torch.empty(m, n, dtype=dt, device=gpu)
        C.call("efm_linear", m, k, n, ptr(x), ptr(w), ptr(b), ptr(y),
               C.EFM_DTYPE_F32 if kind == "f32" else C.EFM_DTYPE_BF16, stream())
    torch.cuda.synchronize()
    rows = torch.tensor([0, m // 2, m - 1])
    xs = x[rows].cpu()
    if kind == "swiglu":
        assert_close_bf16(y[rows], O.gate_up_swiglu(xs, w.cpu()), rtol=2e-2, atol=2e-2)
    elif kind == "f32":
        torch.testing.assert_close(y[rows].cpu(), O.linear(xs, w.cpu(), out_f32=True), rtol=1e-4, atol=1e-4)
    else:
        assert_close_bf16(y[rows], O.linear(xs, w.cpu(), None if b is None else b.cpu()))


@pytest.mark.parametrize("hidden,inter", [(896, 4864), (1536, 8960), (3584, 18944)])
@pytest.mark.parametrize("m", [1, 5, 300])
def test_fused_gate_up_swiglu(gpu, hidden, inter, m):
    torch.manual_seed(0)
    x = torch.randn(m, hidden, dtype=torch.bfloat16)
    w = (torch.randn(2 * inter, hidden) * 0.05).to(torch.bfloat16)
    out = torch.empty(m, inter, dtype=torch.bfloat16, device=gpu)
    xg, wg = x.to(gpu), w.to(gpu)
    C.call("efm_fused_gate_up_swiglu", m, hidden, inter, ptr(xg), ptr(wg), ptr(out), stream())
    torch.cuda.synchronize()
    assert_close_bf16(out, O.gate_up_swiglu(x, w), rtol=2e-2, atol=2e-2)


def _top1_ref_ok(logits: torch.Tensor, tok: int) -> bool:
    """GPU top-1 equals the oracle argmax, or the two differ by less than the fp32
    accumulation-order noise (near tie)."""
    ref = int(O.argmax_lowest(logits.unsqueeze(0))[0])
    if tok == ref:
        return True
    return abs(float(logits[tok]) - float(logits[ref])) < 1e-4 * max(1.0, abs(float(logits[ref])))


@pytest.mark.parametrize("hidden,vocab", [(896, 151936), (1536, 151936), (3584, 152064)])
def test_lm_head_top1(gpu, hidden, vocab):
    torch.manual_seed(0)
    x = torch.randn(1, hidden, dtype=torch.bfloat16)
    w = (torch.randn(vocab, hidden) * 0.02).to(torch.bfloat16)
    ws = torch.zeros(C.load().efm_lm_head_top1_workspace_bytes(vocab), dtype=torch.uint8, device=gpu)
    tok = torch.full((1,), -1, dtype=torch.int32, device=gpu)
    xg, wg = x.to(gpu), w.to(gpu)
    for _ in range(3):  # counter must reset itself between calls
        C.call("efm_lm_head_top1", hidden, vocab, ptr(xg), ptr(wg), ptr(tok), ptr(ws), ws.numel(), stream())
        torch.cuda.synchronize()
        assert _top1_ref_ok(O.linear(x, w, out_f32=True)[0], int(tok.item()))


def test_lm_head_top1_ties_pick_lowest_index(gpu):
    """Duplicate the winning row at a higher and a lower index: the lowest wins
    (src/layers/linear.cu:155-160)."""
    torch.manual_seed(5)
    hidden, vocab = 1536, 151936
    x = torch.randn(1, hidden, dtype=torch.bfloat16)
    w = (torch.randn(vocab, hidden) * 0.02).to(torch.bfloat16)
    w[99_000] = x[0] * 0.1
    w[150_000] = w[99_000]
    w[1234] = w[99_000]
    ws = torch.zeros(C.load().efm_lm_head_top1_workspace_bytes(vocab), dtype=torch.uint8, device=gpu)
    tok = torch.full((1,), -1, dtype=torch.int32, device=gpu)
    xg, wg = x.to(gpu), w.to(gpu)
    C.call("efm_lm_head_top1", hidden, vocab, ptr(xg), ptr(wg), ptr(tok), ptr(ws), ws.numel(), stream())
    torch.cuda.synchronize()
    assert int(tok.item()) == 1234


def test_lm_head_top1_negative_scores_edges_and_clean_workspace(gpu):
    """All scores negative (the order-preserving key must rank negative values by
    magnitude), winner in the last row, then tied with row 0 (row 0 wins); every launch
    leaves the workspace zeroed for the next."""
    torch.manual_seed(6)
    hidden, vocab = 1536, 151936
    x = torch.rand(1, hidden).add(0.5).to(torch.bfloat16)
    w = -(torch.rand(vocab, hidden) * 0.02 + 0.01)
    w[vocab - 1] *= 0.25
    w = w.to(torch.bfloat16)
    ws = torch.zeros(C.load().efm_lm_head_top1_workspace_bytes(vocab), dtype=torch.uint8, device=gpu)
    tok = torch.full((1,), -1, dtype=torch.int32, device=gpu)
    xg, wg = x.to(gpu), w.to(gpu)
    ref = O.linear(x, w, out_f32=True)[0]
    assert float(ref.max()) < 0
    for expect in (vocab - 1, 0):
        if expect == 0:
            wg[0] = wg[vocab - 1]
        C.call("efm_lm_head_top1", hidden, vocab, ptr(xg), ptr(wg), ptr(tok), ptr(ws), ws.numel(), stream())
        torch.cuda.synchronize()
        assert int(tok.item()) == expect
        assert int(ws.count_nonzero()) == 0


@pytest.mark.parametrize("kind", ["bf16", "swiglu"])
def test_gemm_tile_shapes_agree_bit_exact(gpu, kind):
    """The slab kernel's tile follows M (bf16: 64 x 64 at 100 rows, 128 x 128 at 300, 192 x 256
    at 1344, 256 x 256 at 6144, with many tiles per XCD in the grouped order). Every tile sums
    each output over K in the same order, so the first 100 rows must agree bit for bit across
    all launches (and with the oracle on a sample)."""
    torch.manual_seed(17)
    k, n = 1024, 8192
    x = torch.randn(6144, k, dtype=torch.bfloat16, device=gpu)
    nw = 2 * n if kind == "swiglu" else n
    w = (torch.randn(nw, k, device=gpu) * 0.05).to(torch.bfloat16)
    b = (torch.randn(n, device=gpu) * 0.05).to(torch.bfloat16) if kind == "bf16" else None
    heads = []
    for m in (100, 300, 1344, 6144):
        y = torch.empty(m, n, dtype=torch.bfloat16, device=gpu)
        if kind == "swiglu":
            C.call("efm_fused_gate_up_swiglu", m, k, n, ptr(x), ptr(w), ptr(y), stream())
        else:
            C.call("efm_linear", m, k, n, ptr(x), ptr(w), ptr(b), ptr(y), C.EFM_DTYPE_BF16, stream())
        torch.cuda.synchronize()
        heads.append(y[:100].clone())
    for m, h in zip((300, 1344, 6144), heads[1:]):
        assert torch.equal(h, heads[0]), f"{kind}: rows of the M={m} launch differ from the M=100 launch"
    rows = torch.tensor([0, 57, 99])
    xs = x[rows].cpu()
    if kind == "swiglu":
        assert_close_bf16(heads[0][rows], O.gate_up_swiglu(xs, w.cpu()), rtol=2e-2, atol=2e-2)
    else:
        assert_close_bf16(heads[0][rows], O.linear(xs, w.cpu(), b.cpu()))


@pytest.mark.parametrize("m,k,n,kind", [
    pytest.param(4096, 1024, 3072, "bf16", id="aligned"),
    pytest.param(1000, 2048, 1000, "bias", id="ragged_m_n"),
    pytest.param(777, 1536, 2400, "swiglu", id="ragged_swiglu"),
    pytest.param(513, 3584, 4608, "f32", id="f32_bias"),
    pytest.param(512, 1536, 8960, "swiglu", id="c2_gate_up"),
])
def test_gemm_wide_kernel_matches_narrow_bit_exact(gpu, knob, m, k, n, kind):
    """The slab kernel's 256 x 256 (EFM_KNOB_GEMM_TILE 2) and 192 x 256 tiles (knob 3) against
    its tiles up to 128 x 128 (knob 1) on aligned and ragged shapes and every epilogue:
    bit-identical outputs, and a row sample against the oracle."""
    torch.manual_seed(m + n)
    x = torch.randn(m, k, dtype=torch.bfloat16, device=gpu)
    nw = 2 * n if kind == "swiglu" else n
    w = (torch.randn(nw, k, device=gpu) * 0.05).to(torch.bfloat16)
    b = (torch.randn(n, device=gpu) * 0.05).to(torch.bfloat16) if kind in ("bias", "f32") else None
    odt = torch.float32 if kind == "f32" else torch.bfloat16
    outs = []
    for path in (1, 2, 3):
        knob(C.EFM_KNOB_GEMM_TILE, path)
        y = torch.full((m, n), float("nan"), dtype=odt, device=gpu)
        if kind == "swiglu":
            C.call("efm_fused_gate_up_swiglu", m, k, n, ptr(x), ptr(w), ptr(y), stream())
        else:
            cd = C.EFM_DTYPE_F32 if kind == "f32" else C.EFM_DTYPE_BF16
            C.call("efm_linear", m, k, n, ptr(x), ptr(w), ptr(b), ptr(y), cd, stream())
        torch.cuda.synchronize()
        outs.append(y)
    for path, y in zip((2, 3), outs[1:]):
        assert not torch.isnan(y).any(), f"tile of knob {path} left outputs unwritten"
        assert torch.equal(outs[0], y), f"{kind}: tiles of knobs {path} and 1 differ"
    rows = torch.tensor([0, m // 2, m - 1])
    xs = x[rows].cpu()
    if kind == "swiglu":
        assert_close_bf16(outs[1][rows], O.gate_up_swiglu(xs, w.cpu()), rtol=2e-2, atol=2e-2)
    elif kind == "f32":
        ref = O.linear(xs, w.cpu(), b.cpu(), out_f32=True)
        torch.testing.assert_close(outs[1][rows].cpu(), ref, rtol=1e-3, atol=1e-3)
    else:
        assert_close_bf16(outs[1][rows], O.linear(xs, w.cpu(), b.cpu() if b is not None else None))


def _gemm_call(kind, m, k, n, x, w, b, y, ws=None):
    cd = C.EFM_DTYPE_F32 if kind == "f32" else C.EFM_DTYPE_BF16
    if kind == "swiglu":
        C.call("efm_fused_gate_up_swiglu", m, k, n, ptr(x), ptr(w), ptr(y), stream())
    elif ws is not None:
        C.call("efm_linear_ws", m, k, n, ptr(x), ptr(w), ptr(b), ptr(y), cd, ptr(ws), ws.numel(), stream())
    else:
        C.call("efm_linear", m, k, n, ptr(x), ptr(w), ptr(b), ptr(y), cd, stream())
    torch.cuda.synchronize()


def _gemm_reference(kind, x, w, b, n):
    """Float64 products of the same bf16 operands, and what a result may be off: an fp32 sum of
    k products in any order is within k 2^-24 of sum |x w|; a bf16 output adds half an ulp (2^-8
    of its value), SwiGLU's two rounded factors and its silu (slope at most 1.1) three more."""
    h = x.double() @ w.double().T
    mag = x.double().abs() @ w.double().abs().T * (x.shape[1] * 2.0 ** -24)
    if kind == "swiglu":
        u, g = h[:, :n], h[:, n:]
        ref = torch.nn.functional.silu(g) * u
        return ref, (2.0 ** -8 * (2 * ref.abs() + 1.1 * (g * u).abs()) + 1.1 * (mag[:, n:] * u.abs() + mag[:, :n] * g.abs())
                     + 1e-6)
    ref = h if b is None else h + b.double()
    return ref, mag + (0 if kind == "f32" else 2.0 ** -8 * ref.abs()) + 1e-6


@pytest.mark.parametrize("m,k,n,kind", [
    pytest.param(2, 64, 8, "bf16", id="one_slab_two_rows"),
    pytest.param(130, 64, 1001, "f32", id="one_slab_odd_columns"),
    pytest.param(65, 128, 65, "swiglu", id="swiglu_two_slabs"),
    pytest.param(193, 128, 257, "f32", id="two_slabs_odd_columns"),
    pytest.param(192, 192, 264, "bias", id="three_slabs"),
    pytest.param(300, 256, 268, "f32", id="four_columns"),
    pytest.param(257, 320, 132, "swiglu", id="swiglu_second_tile"),
    pytest.param(255, 384, 1003, "bias", id="odd_columns_bias"),
    pytest.param(385, 448, 129, "swiglu", id="swiglu_odd_columns"),
    pytest.param(129, 640, 516, "bias", id="four_columns_bias"),
])
def test_gemm_tall_kernel_edges(gpu, knob, m, k, n, kind):
    """Every tile and ring of the slab kernel (knobs 10 to 18) at its tile edges, with fewer
    slabs than its ring and more, whole and partial column stores: within the bound of float64
    products, bit for bit the same for all tiles (knob 1: the cheapest one), every output written
    and nothing past the last."""
    torch.manual_seed(m + n)
    x = torch.randn(m, k, dtype=torch.bfloat16, device=gpu)
    w = (torch.randn((2 if kind == "swiglu" else 1) * n, k, device=gpu) * 0.05).to(torch.bfloat16)
    b = (torch.randn(n, device=gpu) * 0.05).to(torch.bfloat16) if kind in ("bias", "f32") else None
    ref, err = _gemm_reference(kind, x, w, b, n)
    first = None
    for path in (1, *range(10, 19)):
        knob(C.EFM_KNOB_GEMM_TILE, path)
        y = torch.full((m * n + 8,), -7.0, dtype=torch.float32 if kind == "f32" else torch.bfloat16, device=gpu)
        _gemm_call(kind, m, k, n, x, w, b, y)
        assert (y[-8:] == -7.0).all(), path
        assert ((y[:-8].reshape(m, n).double() - ref).abs() <= err).all(), path
        first = y if first is None else first
        assert torch.equal(first, y), path


@pytest.mark.parametrize("m,k,n,kind", [
    pytest.param(70, 32, 200, "f32", id="one_step"),
    pytest.param(300, 608, 1000, "f32", id="f32"),
    pytest.param(130, 1504, 520, "swiglu", id="swiglu"),
    pytest.param(2100, 352, 2100, "bias", id="128_x_128"),
])
def test_gemm_slab_kernel_matches_register_staged_bit_exact(gpu, knob, m, k, n, kind):
    """K % 64 == 32 runs the register-staged kernel (32 x 32 x 16 MFMAs); the same operands
    with 32 zero keys behind run the slab kernel (16 x 16 x 32 MFMAs), and the added products
    are zeros: the same bits, so both sum keys in the same order."""
    torch.manual_seed(m + k)
    nw = (2 if kind == "swiglu" else 1) * n
    x = torch.randn(m, k, dtype=torch.bfloat16, device=gpu)
    w = (torch.randn(nw, k, device=gpu) * 0.05).to(torch.bfloat16)
    b = (torch.randn(n, device=gpu) * 0.05).to(torch.bfloat16) if kind == "bias" else None
    xp, wp = (torch.nn.functional.pad(t, (0, 32)).contiguous() for t in (x, w))
    y = [torch.empty(m, n, dtype=torch.float32 if kind == "f32" else torch.bfloat16, device=gpu) for _ in range(3)]
    _gemm_call(kind, m, k, n, x, w, b, y[0])
    for out, path in ((y[1], 10), (y[2], 18)):
        knob(C.EFM_KNOB_GEMM_TILE, path)
        _gemm_call(kind, m, k + 32, n, xp, wp, b, out)
    assert torch.equal(y[0], y[1]) and torch.equal(y[0], y[2])


@pytest.mark.parametrize("m,k,n,kind", [
    pytest.param(20, 16384, 81921, "bf16", id="k_split"),
    pytest.param(40, 16384, 81921, "bf16", id="slab"),
    pytest.param(40, 98304, 16384, "bf16", id="split_k"),
    pytest.param(20, 3584, 160000, "swiglu", id="k_split_swiglu"),
    pytest.param(70, 3584, 160000, "swiglu", id="slab_swiglu"),
])
def test_gemm_operands_past_2gb(gpu, m, k, n, kind):
    """Weights of more than 2^31 bytes: the first and last output columns of the tiled kernels
    against fp32 products (both round an fp32 sum to bf16; the sums differ by a few ulps of
    fp32 times sqrt(k), far below bf16's 2^-8)."""
    nw = 2 * n if kind == "swiglu" else n
    assert nw * k * 2 > 1 << 31
    g = torch.Generator(device=gpu).manual_seed(m)
    x = torch.empty(m, k, dtype=torch.bfloat16, device=gpu).normal_(generator=g)
    w = torch.empty(nw, k, dtype=torch.bfloat16, device=gpu).normal_(std=k ** -0.5, generator=g)
    y = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=gpu)
    if kind == "swiglu":
        C.call("efm_fused_gate_up_swiglu", m, k, n, ptr(x), ptr(w), ptr(y), stream())
    else:
        ws = torch.empty(max(C.load().efm_linear_workspace_bytes(m, k, n), 256), dtype=torch.uint8, device=gpu)
        C.call("efm_linear_ws", m, k, n, ptr(x), ptr(w), None, ptr(y), C.EFM_DTYPE_BF16, ptr(ws), ws.numel(), stream())
    torch.cuda.synchronize()
    for c in (slice(0, 256), slice(n // 2, n // 2 + 256), slice(n - 256, n)):
        ref = x.float() @ w[:n][c].float().T
        if kind == "swiglu":
            up, gate = ref.bfloat16().float(), (x.float() @ w[n:][c].float().T).bfloat16().float()
            ref = torch.nn.functional.silu(gate) * up
        torch.testing.assert_close(y[:, c].float(), ref, rtol=2 ** -6, atol=2 ** -6)
    assert not y.isnan().any()


@pytest.mark.parametrize("m,k,n,kind", [
    pytest.param(512, 8960, 1536, "bf16", id="c2_down"),
    pytest.param(300, 18944, 3584, "bf16", id="7b_down"),
    pytest.param(300, 4096, 1000, "bias", id="ragged_bias"),
    pytest.param(200, 8192, 2048, "f32", id="f32"),
    pytest.param(1024, 8960, 1536, "bf16", id="shallow_split"),
])
def test_linear_split_k_matches_unsplit_and_oracle(gpu, m, k, n, kind):
    """efm_linear_ws splits K for these under-filled, long-K shapes: its result equals
    efm_linear to fp32 rounding, is deterministic, matches the oracle on a row sample, and
    with too small a workspace the call is exactly efm_linear."""
    torch.manual_seed(m + k)
    need = C.load().efm_linear_workspace_bytes(m, k, n)
    assert need > 0
    x = torch.randn(m, k, dtype=torch.bfloat16, device=gpu)
    w = (torch.randn(n, k, device=gpu) * 0.02).to(torch.bfloat16)
    b = (torch.randn(n, device=gpu) * 0.05).to(torch.bfloat16) if kind == "bias" else None
    f32 = kind == "f32"
    dt, cd = (torch.float32, C.EFM_DTYPE_F32) if f32 else (torch.bfloat16, C.EFM_DTYPE_BF16)
    ws = torch.full((need,), 0x7f, dtype=torch.uint8, device=gpu)
    outs = []
    for wsz in (need, need, 64):
        y = torch.empty(m, n, dtype=dt, device=gpu)
        C.call("efm_linear_ws", m, k, n, ptr(x), ptr(w), ptr(b), ptr(y), cd, ptr(ws), wsz, stream())
        torch.cuda.synchronize()
        outs.append(y)
    ref = torch.empty(m, n, dtype=dt, device=gpu)
    C.call("efm_linear", m, k, n, ptr(x), ptr(w), ptr(b), ptr(ref), cd, stream())
    torch.cuda.synchronize()
    assert torch.equal(outs[0], outs[1]), "split-K is not deterministic"
    assert torch.equal(outs[2], ref), "too small a workspace must run the unsplit GEMM"
    if f32:
        torch.testing.assert_close(outs[0], ref, rtol=1e-5, atol=1e-4)
    else:
        diff = (outs[0].float() - ref.float()).abs()
        assert float(diff.max()) <= float(ref.float().abs().max()) * 2 ** -7, "split-K differs beyond one bf16 ulp"
    rows = torch.tensor([0, m // 2, m - 1])
    exp = O.linear(x[rows].cpu(), w.cpu(), None if b is None else b.cpu(), out_f32=f32)
    if f32:
        torch.testing.assert_close(outs[0][rows].cpu(), exp, rtol=1e-4, atol=1e-4)
    else:
        assert_close_bf16(outs[0][rows], exp)


@pytest.mark.parametrize("m,k,n,kind,split", [
    # tile edges in rows and columns, waves with unequal slabs (K 832), ragged columns that
    # take scalar stores, every epilogue, and the sliced forms of the three tiles
    pytest.param(2, 768, 32, "bf16", False, id="one_tile"),
    pytest.param(31, 832, 100, "bias", False, id="unequal_slabs"),
    pytest.param(32, 1536, 1001, "f32", False, id="ragged_f32"),
    pytest.param(33, 1536, 2048, "bias", False, id="second_row_block"),
    pytest.param(64, 896, 1154, "f32", False, id="f32_64_rows"),
    pytest.param(200, 2048, 2048, "bias", False, id="64x32_tiles"),
    pytest.param(257, 2048, 1090, "f32", False, id="64x32_ragged"),
    pytest.param(700, 4864, 896, "bf16", False, id="64x64_long_k"),
    pytest.param(700, 4864, 898, "bias", False, id="64x64_ragged"),
    pytest.param(700, 3072, 1001, "f32", False, id="64x64_odd_f32"),
    pytest.param(2, 896, 8, "swiglu", False, id="swiglu_one_tile"),
    pytest.param(32, 1536, 8950, "swiglu", False, id="swiglu_ragged"),
    pytest.param(24, 8960, 1536, "bias", True, id="sliced_32x32"),
    pytest.param(61, 11008, 2044, "f32", True, id="sliced_64x32"),
    pytest.param(130, 8960, 1000, "bias", True, id="sliced_64x64"),
])
def test_gemm_k_split_over_waves(gpu, knob, m, k, n, kind, split):
    """Launches that split K over the waves of a workgroup (and, with a workspace, over
    workgroups): within the bound of float64 products, every output written and nothing past the
    last one, deterministic, and not the slab kernel's bits (knob 1, held to the same bound)."""
    torch.manual_seed(m + n)
    x = torch.randn(m, k, dtype=torch.bfloat16, device=gpu)
    w = (torch.randn((2 if kind == "swiglu" else 1) * n, k, device=gpu) * 0.02).to(torch.bfloat16)
    b = (torch.randn(n, device=gpu) * 0.05).to(torch.bfloat16) if kind in ("bias", "f32") else None
    need = C.load().efm_linear_workspace_bytes(m, k, n)
    assert (need > 0) == split
    ws = torch.full((need,), 0x7f, dtype=torch.uint8, device=gpu) if split else None
    ref, err = _gemm_reference(kind, x, w, b, n)
    outs = []
    for path in (0, 0, 1):
        knob(C.EFM_KNOB_GEMM_TILE, path)
        y = torch.full((m * n + 8,), -7.0, dtype=torch.float32 if kind == "f32" else torch.bfloat16, device=gpu)
        _gemm_call(kind, m, k, n, x, w, b, y, ws if path == 0 else None)
        assert (y[m * n:] == -7.0).all()
        outs.append(y[:m * n].reshape(m, n))
        assert ((outs[-1].double() - ref).abs() <= err).all()
    assert torch.equal(outs[0], outs[1])
    # another order of the sums: fp32 results differ somewhere, bf16 ones of many elements too
    if kind == "f32" or m * n > 20000:
        assert not torch.equal(outs[0], outs[2])


def test_gemm_long_k_tiles_agree_bit_exact(gpu):
    """K = 11008 (the VL-3B down projection) at three M: 64 x 64 tiles at 100 rows, 128 x 128
    ones over rings of four slabs at 1344 (at most one per CU), 192 x 128 ones at 2300. All sum
    each output over K in the same order: the first 100 rows agree bit for bit, and a row
    sample of each launch matches the oracle."""
    torch.manual_seed(29)
    k, n = 11008, 2048
    x = torch.randn(2300, k, dtype=torch.bfloat16, device=gpu)
    w = (torch.randn(n, k, device=gpu) * 0.02).to(torch.bfloat16)
    b = (torch.randn(n, device=gpu) * 0.05).to(torch.bfloat16)
    outs = {}
    for m in (100, 1344, 2300):
        y = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=gpu)
        C.call("efm_linear", m, k, n, ptr(x), ptr(w), ptr(b), ptr(y), C.EFM_DTYPE_BF16, stream())
        torch.cuda.synchronize()
        assert not torch.isnan(y).any(), f"M={m}: outputs left unwritten"
        outs[m] = y
    for m in (1344, 2300):
        assert torch.equal(outs[m][:100], outs[100]), f"rows of the M={m} launch differ from the M=100 launch"
        rows = torch.tensor([0, m // 2, m - 1])
        assert_close_bf16(outs[m][rows], O.linear(x[rows].cpu(), w.cpu(), b.cpu()))


def test_linear_workspace_bytes_zero_without_split(gpu):
    lib = C.load()
    assert lib.efm_linear_workspace_bytes(1, 8960, 1536) == 0          # GEMV
    assert lib.efm_linear_workspace_bytes(16384, 18944, 3584) == 0     # enough tiles
    assert lib.efm_linear_workspace_bytes(512, 1536, 1536) == 0        # short K
    assert lib.efm_linear_workspace_bytes(1344, 11008, 2048) == 0      # 176 tiles: no gain
    assert lib.efm_linear_workspace_bytes(512, 8960, 1536) > 0


@pytest.mark.parametrize("m,k,n,bias", [
    pytest.param(1344, 2048, 2560, True, id="c3_qkv"),
    pytest.param(1344, 11008, 2048, False, id="c3_down"),
    pytest.param(512, 8960, 1536, False, id="c2_down"),
    pytest.param(77, 1536, 2048, True, id="ragged_m"),
    pytest.param(2, 896, 1000, False, id="m2"),
])
def test_linear_workspace_path_matches_oracle_and_repeats(gpu, m, k, n, bias):
    """The prefill GEMM with its workspace (split-K where the plan asks for it) and without
    one: both match the oracle on a row sample, each repeats bit for bit, and the two agree
    to bf16 rounding (the split sums K in another order)."""
    torch.manual_seed(m + n)
    x = torch.randn(m, k, dtype=torch.bfloat16, device=gpu)
    w = (torch.randn(n, k, device=gpu) * 0.02).to(torch.bfloat16)
    b = (torch.randn(n, device=gpu) * 0.05).to(torch.bfloat16) if bias else None
    need = C.load().efm_linear_workspace_bytes(m, k, n)
    ws = torch.full((max(need, 256),), 0x7f, dtype=torch.uint8, device=gpu)
    outs = []
    for use_ws in (True, True, False, False):
        y = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=gpu)
        if use_ws:
            C.call("efm_linear_ws", m, k, n, ptr(x), ptr(w), ptr(b), ptr(y), C.EFM_DTYPE_BF16, ptr(ws), need,
                   stream())
        else:
            C.call("efm_linear", m, k, n, ptr(x), ptr(w), ptr(b), ptr(y), C.EFM_DTYPE_BF16, stream())
        torch.cuda.synchronize()
        outs.append(y)
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[2], outs[3]), "GEMM is not deterministic"
    scale = float(outs[2].float().abs().max())
    assert torch.isfinite(outs[0].float()).all()
    assert float((outs[0].float() - outs[2].float()).abs().max()) <= scale * 2 ** -7
    rows = torch.tensor([0, m // 2, m - 1])
    exp = O.linear(x[rows].cpu(), w.cpu(), None if b is None else b.cpu())
    assert_close_bf16(outs[0][rows], exp)
    assert_close_bf16(outs[2][rows], exp)


def test_linear_workspace_plan_ignores_spare_capacity(gpu):
    """A caller whose grow-only scratch is larger than a shape needs gets the same bits as
    one passing exactly the shape's figure: the split-K plan depends on the shape alone."""
    torch.manual_seed(3)
    m, k, n = 512, 8960, 1536
    x = torch.randn(m, k, dtype=torch.bfloat16, device=gpu)
    w = (torch.randn(n, k, device=gpu) * 0.02).to(torch.bfloat16)
    need = C.load().efm_linear_workspace_bytes(m, k, n)
    big = 3 * need
    assert need > 0
    ws = torch.zeros(big, dtype=torch.uint8, device=gpu)
    a = torch.empty(m, n, dtype=torch.bfloat16, device=gpu)
    b = torch.empty_like(a)
    C.call("efm_linear_ws", m, k, n, ptr(x), ptr(w), None, ptr(a), C.EFM_DTYPE_BF16, ptr(ws), need, stream())
    C.call("efm_linear_ws", m, k, n, ptr(x), ptr(w), None, ptr(b), C.EFM_DTYPE_BF16, ptr(ws), big, stream())
    torch.cuda.synchronize()
    assert torch.equal(a, b)


def test_linear_unaligned_output(gpu):
    """An output pointer that is only 2-byte aligned is written correctly."""
    torch.manual_seed(8)
    m, k, n = 64, 1024, 1000
    x = torch.randn(m, k, dtype=torch.bfloat16, device=gpu)
    w = (torch.randn(n, k, device=gpu) * 0.02).to(torch.bfloat16)
    buf = torch.zeros(m * n + 8, dtype=torch.bfloat16, device=gpu)
    out = buf[1:1 + m * n]                       # 2-byte offset
    assert out.data_ptr() % 16 != 0
    C.call("efm_linear", m, k, n, ptr(x), ptr(w), None, ptr(out), C.EFM_DTYPE_BF16, stream())
    aligned = torch.empty(m, n, dtype=torch.bfloat16, device=gpu)
    C.call("efm_linear", m, k, n, ptr(x), ptr(w), None, ptr(aligned), C.EFM_DTYPE_BF16, stream())
    torch.cuda.synchronize()
    assert torch.equal(out.reshape(m, n), aligned)
    assert float(buf[0]) == 0.0 and float(buf[1 + m * n]) == 0.0
    assert_close_bf16(aligned[:3], O.linear(x[:3].cpu(), w.cpu()))


@pytest.mark.parametrize("m,k,n,kind", [
    pytest.param(300, 256, 1000, "bias", id="slab"),
    pytest.param(300, 256, 1000, "f32", id="slab_f32"),
    pytest.param(70, 192, 200, "swiglu", id="slab_swiglu"),
    pytest.param(20, 1536, 1000, "bias", id="k_split"),
    pytest.param(20, 1536, 1000, "f32", id="k_split_f32"),
    pytest.param(20, 896, 200, "swiglu", id="k_split_swiglu"),
])
def test_gemm_output_one_element_off(gpu, m, k, n, kind):
    """Every epilogue stores whole segments at any alignment: an output one element behind a
    16-byte boundary holds the aligned call's bits, and its neighbours are untouched."""
    torch.manual_seed(m + n)
    x = torch.randn(m, k, dtype=torch.bfloat16, device=gpu)
    w = (torch.randn((2 if kind == "swiglu" else 1) * n, k, device=gpu) * 0.05).to(torch.bfloat16)
    b = (torch.randn(n, device=gpu) * 0.05).to(torch.bfloat16) if kind == "bias" else None
    buf = [torch.full((m * n + 16,), -7.0, dtype=torch.float32 if kind == "f32" else torch.bfloat16, device=gpu)
           for _ in range(2)]
    for t, at in zip(buf, (8, 1)):
        _gemm_call(kind, m, k, n, x, w, b, t[at:])
        assert (t[:at] == -7.0).all() and (t[at + m * n:] == -7.0).all()
    assert torch.equal(buf[0][8:8 + m * n], buf[1][1:1 + m * n])


def test_linear_under_graph_capture(gpu):
    """A prefill GEMM captured into a HIP graph: every replay equals the eager call bit for
    bit, with eager calls between replays."""
    torch.manual_seed(5)
    m, k, n = 96, 1536, 2048
    x = torch.randn(m, k, dtype=torch.bfloat16, device=gpu)
    w = (torch.randn(n, k, device=gpu) * 0.02).to(torch.bfloat16)
    b = (torch.randn(n, device=gpu) * 0.05).to(torch.bfloat16)
    own = torch.empty(m, n, dtype=torch.bfloat16, device=gpu)
    C.call("efm_linear", m, k, n, ptr(x), ptr(w), ptr(b), ptr(own), C.EFM_DTYPE_BF16, stream())
    torch.cuda.synchronize()
    y = torch.empty(m, n, dtype=torch.bfloat16, device=gpu)
    st = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=st, capture_error_mode="thread_local"):
        C.call("efm_linear", m, k, n, ptr(x), ptr(w), ptr(b), ptr(y), C.EFM_DTYPE_BF16, st.cuda_stream)
    for rep in range(3):
        y.fill_(float("nan"))
        eager = torch.empty(m, n, dtype=torch.bfloat16, device=gpu)
        C.call("efm_linear", m, k, n, ptr(x), ptr(w), ptr(b), ptr(eager), C.EFM_DTYPE_BF16, stream())
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, own), f"replay {rep}"
        assert torch.equal(eager, own)


@pytest.mark.parametrize("m,hidden,inter", [(1344, 2048, 11008), (512, 1536, 8960), (33, 896, 4864)])
def test_gate_up_swiglu_ws_is_fused_kernel(gpu, m, hidden, inter):
    """efm_fused_gate_up_swiglu_ws needs no workspace and equals efm_fused_gate_up_swiglu bit
    for bit; it agrees with efm_linear into [m, 2 inter] + efm_act_and_mul (the reference's
    two-stage path) to bf16 rounding, and with the oracle on sampled rows."""
    torch.manual_seed(m)
    x = torch.randn(m, hidden, dtype=torch.bfloat16, device=gpu)
    w = (torch.randn(2 * inter, hidden, device=gpu) * 0.03).to(torch.bfloat16)
    assert C.load().efm_fused_gate_up_swiglu_workspace_bytes(m, hidden, inter) == 0
    out = torch.empty(m, inter, dtype=torch.bfloat16, device=gpu)
    C.call("efm_fused_gate_up_swiglu_ws", m, hidden, inter, ptr(x), ptr(w), ptr(out), None, 0, stream())
    fused = torch.empty_like(out)
    C.call("efm_fused_gate_up_swiglu", m, hidden, inter, ptr(x), ptr(w), ptr(fused), stream())
    gu = torch.empty(m, 2 * inter, dtype=torch.bfloat16, device=gpu)
    C.call("efm_linear", m, hidden, 2 * inter, ptr(x), ptr(w), None, ptr(gu), C.EFM_DTYPE_BF16, stream())
    two = torch.empty_like(out)
    C.call("efm_act_and_mul", m, inter, C.EFM_LAYOUT_UP_GATE, ptr(gu), ptr(two), stream())
    torch.cuda.synchronize()
    assert torch.equal(out, fused)
    diff = (two.float() - fused.float()).abs()
    assert float(diff.max()) <= float(fused.float().abs().max()) * 2 ** -6
    rows = torch.tensor([0, m - 1])
    assert_close_bf16(out[rows], O.gate_up_swiglu(x[rows].cpu(), w.cpu()), rtol=2e-2, atol=2e-2)


def test_sampler_greedy_ties(gpu):
    torch.manual_seed(0)
    rows, vocab = 4, 151936
    logits = torch.randn(rows, vocab)
    logits[0, 17] = logits[0, 9000] = 50.0
    logits[1, vocab - 1] = 60.0
    logits[2, :] = 1.0
    logits[3, 123456] = 7.0
    logits[3, 123455] = 7.0
    ws = torch.zeros(C.load().efm_sampler_greedy_workspace_bytes(rows, vocab), dtype=torch.uint8, device=gpu)
    out = torch.empty(rows, dtype=torch.int32, device=gpu)
    lg = logits.to(gpu)
    C.call("efm_sampler_greedy", rows, vocab, ptr(lg), ptr(out), ptr(ws), ws.numel(), stream())
    torch.cuda.synchronize()
    assert out.cpu().tolist() == O.argmax_lowest(logits).tolist() == [17, vocab - 1, 0, 123455]


def test_embedding_lookup_with_insertion(gpu):
    torch.manual_seed(0)
    V, H = 1000, 1536
    table = torch.randn(V, H).to(torch.bfloat16)
    custom = torch.randn(5, H).to(torch.bfloat16)
    ids = torch.tensor([3, 999, -1, 1000, 700, 701, 704, 705, 0], dtype=torch.int32)
    out = torch.empty(ids.numel(), H, dtype=torch.bfloat16, device=gpu)
    idg, tg, cg = ids.to(gpu), table.to(gpu), custom.to(gpu)
    C.call("efm_embedding_lookup", ids.numel(), H, V, ptr(idg), ptr(tg), ptr(cg), 5, 700, ptr(out), stream())
    torch.cuda.synchronize()
    assert torch.equal(out.cpu(), O.embedding(ids, table, custom, 700))


def test_decode_runtime_kernels(gpu):
    kdim, vdim, rows = 256, 256, 10
    kc = torch.zeros(rows, kdim, dtype=torch.bfloat16, device=gpu)
    vc = torch.zeros(rows, vdim, dtype=torch.bfloat16, device=gpu)
    ks = torch.randn(kdim).to(torch.bfloat16).to(gpu)
    vs = torch.randn(vdim).to(torch.bfloat16).to(gpu)
    d_len = torch.tensor([4], dtype=torch.int32, device=gpu)
    C.call("efm_copy_decode_kv_cache_slots", ptr(ks), ptr(vs), ptr(kc), ptr(vc), kdim, vdim, ptr(d_len), stream())
    sampled = torch.tensor([42], dtype=torch.int32, device=gpu)
    resp = torch.zeros(3, dtype=torch.int32, device=gpu)
    C.call("efm_finalize_decode_token", ptr(sampled), resp[1:].data_ptr(), ptr(d_len), stream())
    trip = torch.tensor([5, 6, 7], dtype=torch.int32, device=gpu)
    C.call("efm_increment_int32_triplet", ptr(trip), stream())
    torch.cuda.synchronize()
    assert torch.equal(kc[3], ks) and torch.equal(vc[3], vs)
    assert kc[:3].abs().sum() == 0 and kc[4:].abs().sum() == 0
    assert resp.cpu().tolist() == [0, 42, 0] and int(d_len.item()) == 5
    assert trip.cpu().tolist() == [6, 7, 8]


@pytest.mark.parametrize("hidden,hq,hkv,hd", [(1536, 12, 2, 128), (896, 14, 2, 64), (3584, 28, 4, 128)])
@pytest.mark.parametrize("layer0", [True, False])
def test_decode_norm_qkv_matches_unfused(gpu, hidden, hq, hkv, hd, layer0):
    torch.manual_seed(0)
    eps = 1e-6
    qd, kvd = hq * hd, hkv * hd
    h = torch.randn(1, hidden, dtype=torch.bfloat16)
    r = torch.randn(1, hidden, dtype=torch.bfloat16)
    nw = (1 + 0.1 * torch.randn(hidden)).to(torch.bfloat16)
    W = (torch.randn(qd + 2 * kvd, hidden) * 0.02).to(torch.bfloat16)
    b = (torch.randn(qd + 2 * kvd) * 0.02).to(torch.bfloat16)
    rows = 20
    kc = torch.zeros(rows, kvd, dtype=torch.bfloat16, device=gpu)
    vc = torch.zeros(rows, kvd, dtype=torch.bfloat16, device=gpu)
    d_len = torch.tensor([13], dtype=torch.int32, device=gpu)
    q_out = torch.empty(1, qd, dtype=torch.bfloat16, device=gpu)
    r_out = torch.empty(1, hidden, dtype=torch.bfloat16, device=gpu)
    hg, rg, nwg, Wg, bg = h.to(gpu), r.to(gpu), nw.to(gpu), W.to(gpu), b.to(gpu)
    C.call("efm_decode_norm_qkv", hidden, qd, kvd, eps, ptr(hg), None if layer0 else ptr(rg), ptr(r_out), ptr(nwg),
           ptr(Wg), ptr(bg), ptr(q_out), ptr(kc), ptr(vc), ptr(d_len), stream())
    torch.cuda.synchronize()
    if layer0:
        n, res = O.rms_norm(h, nw, eps), h
    else:
        n, res = O.fused_add_rms_norm(h, r, nw, eps)
    qkv = O.linear(n, W, b)
    assert torch.equal(r_out.cpu(), res)
    assert_close_bf16(q_out, qkv[:, :qd], what="q")
    assert_close_bf16(kc[12:13], qkv[:, qd:qd + kvd], what="k slot")
    assert_close_bf16(vc[12:13], qkv[:, qd + kvd:], what="v slot")
    assert kc[:12].abs().sum() == 0 and kc[13:].abs().sum() == 0


@pytest.mark.parametrize("hidden,hq,hkv,hd", [(1536, 12, 2, 128), (896, 14, 2, 64), (3584, 28, 4, 128)])
@pytest.mark.parametrize("layer0", [True, False])
@pytest.mark.parametrize("pos_off", [0, 5])
def test_decode_norm_qkv_rope_matches_oracle(gpu, hidden, hq, hkv, hd, layer0, pos_off):
    """efm_decode_norm_qkv_rope: the projection of efm_decode_norm_qkv with q and the new
    key rotated at position L - 1 (+ offset) in the epilogue: q_out and the K slot equal
    the oracle's rope_llama of the bf16 projection (one bf16 rounding), V and the residual
    are exact; no other cache row is written. Then decode attention with pos NONE over
    that cache equals the oracle's RoPE-on-read attention over the un-rotated keys."""
    torch.manual_seed(1 + hd)
    eps, theta, L = 1e-6, 1.0e6, 300
    qd, kvd = hq * hd, hkv * hd
    h = torch.randn(1, hidden, dtype=torch.bfloat16)
    r = torch.randn(1, hidden, dtype=torch.bfloat16)
    nw = (1 + 0.1 * torch.randn(hidden)).to(torch.bfloat16)
    W = (torch.randn(qd + 2 * kvd, hidden) * 0.02).to(torch.bfloat16)
    b = (torch.randn(qd + 2 * kvd) * 0.02).to(torch.bfloat16)
    k_prev = torch.randn(L - 1, hkv, hd, dtype=torch.bfloat16)
    v_prev = torch.randn(L - 1, hkv, hd, dtype=torch.bfloat16)
    rows = L + 20
    kc = torch.zeros(rows, kvd, dtype=torch.bfloat16)
    vc = torch.zeros(rows, kvd, dtype=torch.bfloat16)
    kc[: L - 1] = O.rope_llama(k_prev, torch.arange(L - 1) + pos_off, theta).to(torch.bfloat16).reshape(L - 1, kvd)
    vc[: L - 1] = v_prev.reshape(L - 1, kvd)
    kc, vc = kc.to(gpu), vc.to(gpu)
    d_len = torch.tensor([L], dtype=torch.int32, device=gpu)
    q_out = torch.empty(1, qd, dtype=torch.bfloat16, device=gpu)
    r_out = torch.empty(1, hidden, dtype=torch.bfloat16, device=gpu)
    ctx = C.make_attention_ctx(hq, hkv, hd, rope_theta=theta, q_rope_pos_offset=pos_off, k_rope_pos_offset=pos_off)
    hg, rg, nwg, Wg, bg = h.to(gpu), r.to(gpu), nw.to(gpu), W.to(gpu), b.to(gpu)
    C.call("efm_decode_norm_qkv_rope", ctx, hidden, eps, ptr(hg), None if layer0 else ptr(rg), ptr(r_out), ptr(nwg),
           ptr(Wg), ptr(bg), ptr(q_out), ptr(kc), ptr(vc), ptr(d_len), stream())
    torch.cuda.synchronize()
    if layer0:
        n, res = O.rms_norm(h, nw, eps), h
    else:
        n, res = O.fused_add_rms_norm(h, r, nw, eps)
    qkv = O.linear(n, W, b)
    pos = torch.tensor([L - 1 + pos_off])
    q_ref = O.rope_llama(qkv[:, :qd].reshape(1, hq, hd), pos, theta).to(torch.bfloat16).reshape(1, qd)
    k_new = qkv[:, qd:qd + kvd].reshape(1, hkv, hd)
    k_ref = O.rope_llama(k_new, pos, theta).to(torch.bfloat16).reshape(1, kvd)
    assert torch.equal(r_out.cpu(), res)
    assert_close_bf16(q_out, q_ref, what="rotated q")
    assert_close_bf16(kc[L - 1:L], k_ref, what="rotated k slot")
    assert_close_bf16(vc[L - 1:L], qkv[:, qd + kvd:], what="v slot")
    assert kc[L:].abs().sum() == 0 and vc[L:].abs().sum() == 0
    # attention over the rotated cache without RoPE == RoPE-on-read over un-rotated keys
    k_all = torch.cat([k_prev, k_new.to(torch.bfloat16)])
    v_all = torch.cat([v_prev, qkv[:, qd + kvd:].reshape(1, hkv, hd)])
    ref = O.attention_decode(qkv[:, :qd].reshape(1, hq, hd), k_all, v_all, L,
                             O.AttnCtx(hq, hkv, hd, rope_theta=theta, q_rope_pos_offset=pos_off,
                                       k_rope_pos_offset=pos_off))
    actx = C.make_attention_ctx(hq, hkv, hd, rope=False)
    ws = torch.zeros(C.load().efm_attention_decode_workspace_bytes(actx, rows), dtype=torch.uint8, device=gpu)
    o = torch.empty(1, hq, hd, dtype=torch.bfloat16, device=gpu)
    C.call("efm_attention_decode", actx, ptr(q_out), ptr(kc), ptr(vc), ptr(o), 0, ptr(d_len), rows, ptr(ws),
           ws.numel(), stream())
    torch.cuda.synchronize()
    assert_close_bf16(o, ref, what="attention over the rotated cache")


def test_decode_front_half_7b_16k_engine_chain(gpu):
    """The decode front half of one Qwen2.5-7B-shaped layer at C5's context, through the
    C-ABI chain the engine runs: norm + QKV with q and the new key rotated in the epilogue
    (slot 16447), decode attention over 16,448 rotated cache rows (28/4 heads: the 8-wave
    kernel, 58 splits of 288 keys of a 16,512-row cache, then the split merge kernel), and
    the o_proj GEMV; against the oracle's layer with RoPE on read over the un-rotated keys
    (Appendix-A rounding points)."""
    torch.manual_seed(21)
    hidden, hq, hkv, hd, eps, theta = 3584, 28, 4, 128, 1e-6, 1.0e6
    L, max_kv = 16448, 16512
    qd, kvd = hq * hd, hkv * hd
    h = torch.randn(1, hidden, dtype=torch.bfloat16)
    r = torch.randn(1, hidden, dtype=torch.bfloat16)
    nw = (1 + 0.1 * torch.randn(hidden)).to(torch.bfloat16)
    W = (torch.randn(qd + 2 * kvd, hidden) * 0.02).to(torch.bfloat16)
    b = (torch.randn(qd + 2 * kvd) * 0.02).to(torch.bfloat16)
    Wo = (torch.randn(hidden, qd) * 0.02).to(torch.bfloat16)
    k_prev = torch.randn(L - 1, hkv, hd, dtype=torch.bfloat16)
    v_prev = torch.randn(L - 1, hkv, hd, dtype=torch.bfloat16)
    kc = torch.full((max_kv, kvd), float("nan"), dtype=torch.bfloat16)
    vc = torch.full((max_kv, kvd), float("nan"), dtype=torch.bfloat16)
    kc[: L - 1] = O.rope_llama(k_prev, torch.arange(L - 1), theta).to(torch.bfloat16).reshape(L - 1, kvd)
    vc[: L - 1] = v_prev.reshape(L - 1, kvd)
    kc, vc = kc.to(gpu), vc.to(gpu)
    d_len = torch.tensor([L], dtype=torch.int32, device=gpu)
    hg, rg, nwg, Wg, bg, Wog = (t.to(gpu) for t in (h, r, nw, W, b, Wo))
    q = torch.empty(1, qd, dtype=torch.bfloat16, device=gpu)
    r_out = torch.empty(1, hidden, dtype=torch.bfloat16, device=gpu)
    attn = torch.empty(1, qd, dtype=torch.bfloat16, device=gpu)
    a = torch.empty(1, hidden, dtype=torch.bfloat16, device=gpu)
    cq = C.make_attention_ctx(hq, hkv, hd, rope_theta=theta)
    ca = C.make_attention_ctx(hq, hkv, hd, rope=False)
    ws = torch.zeros(C.load().efm_attention_decode_workspace_bytes(ca, max_kv), dtype=torch.uint8, device=gpu)
    C.call("efm_decode_norm_qkv_rope", cq, hidden, eps, ptr(hg), ptr(rg), ptr(r_out), ptr(nwg), ptr(Wg), ptr(bg),
           ptr(q), ptr(kc), ptr(vc), ptr(d_len), stream())
    C.call("efm_attention_decode", ca, ptr(q), ptr(kc), ptr(vc), ptr(attn), 0, ptr(d_len), max_kv, ptr(ws), ws.numel(),
           stream())
    C.call("efm_linear", 1, qd, hidden, ptr(attn), ptr(Wog), None, ptr(a), C.EFM_DTYPE_BF16, stream())
    torch.cuda.synchronize()
    n, res = O.fused_add_rms_norm(h, r, nw, eps)
    qkv = O.linear(n, W, b)
    k_all = torch.cat([k_prev, qkv[:, qd:qd + kvd].reshape(1, hkv, hd)])
    v_all = torch.cat([v_prev, qkv[:, qd + kvd:].reshape(1, hkv, hd)])
    o_ref = O.attention_decode(qkv[:, :qd].reshape(1, hq, hd), k_all, v_all, L,
                               O.AttnCtx(hq, hkv, hd, rope_theta=theta)).reshape(1, qd)
    a_ref = O.linear(o_ref, Wo)
    assert torch.equal(r_out.cpu(), res)
    assert torch.isfinite(attn.float()).all()
    assert_close_bf16(attn, o_ref, what="attention over 16,448 rows")
    assert_close_bf16(a, a_ref, what="o_proj of the attention output")
    assert torch.isnan(kc[L:].float()).all(), "rows past the newest must not be written"
    assert_close_bf16(vc[L - 1:L], qkv[:, qd + kvd:], what="v slot")


@pytest.mark.parametrize("hidden,inter", [(1536, 8960), (896, 4864), (3584, 18944)])
def test_decode_norm_gate_up_swiglu_matches_unfused(gpu, hidden, inter):
    torch.manual_seed(0)
    eps = 1e-6
    a = torch.randn(1, hidden, dtype=torch.bfloat16)
    r = torch.randn(1, hidden, dtype=torch.bfloat16)
    nw = (1 + 0.1 * torch.randn(hidden)).to(torch.bfloat16)
    W = (torch.randn(2 * inter, hidden) * 0.05).to(torch.bfloat16)
    out = torch.empty(1, inter, dtype=torch.bfloat16, device=gpu)
    r_out = torch.empty(1, hidden, dtype=torch.bfloat16, device=gpu)
    ag, rg, nwg, Wg = a.to(gpu), r.to(gpu), nw.to(gpu), W.to(gpu)
    C.call("efm_decode_norm_gate_up_swiglu", hidden, inter, eps, ptr(ag), ptr(rg), ptr(r_out), ptr(nwg), ptr(Wg),
           ptr(out), stream())
    torch.cuda.synchronize()
    n2, res = O.fused_add_rms_norm(a, r, nw, eps)
    assert torch.equal(r_out.cpu(), res)
    assert_close_bf16(out, O.gate_up_swiglu(n2, W), rtol=2e-2, atol=2e-2)


@pytest.mark.parametrize("hidden,vocab", [(1536, 151936), (896, 151936)])
def test_decode_norm_lm_head_top1_matches_unfused(gpu, hidden, vocab):
    torch.manual_seed(2)
    eps = 1e-6
    h = torch.randn(1, hidden, dtype=torch.bfloat16)
    r = torch.randn(1, hidden, dtype=torch.bfloat16)
    nw = (1 + 0.1 * torch.randn(hidden)).to(torch.bfloat16)
    W = (torch.randn(vocab, hidden) * 0.02).to(torch.bfloat16)
    ws = torch.zeros(C.load().efm_lm_head_top1_workspace_bytes(vocab), dtype=torch.uint8, device=gpu)
    tok = torch.full((1,), -1, dtype=torch.int32, device=gpu)
    hg, rg, nwg, Wg = h.to(gpu), r.to(gpu), nw.to(gpu), W.to(gpu)
    C.call("efm_decode_norm_lm_head_top1", hidden, vocab, eps, ptr(hg), ptr(rg), ptr(nwg), ptr(Wg), ptr(tok),
           ptr(ws), ws.numel(), stream())
    torch.cuda.synchronize()
    x, _ = O.fused_add_rms_norm(h, r, nw, eps)
    assert _top1_ref_ok(O.linear(x, W, out_f32=True)[0], int(tok.item()))


PREFILL_CASES = [
    pytest.param(12, 2, 128, 512, 512, id="1p5b_s512"),
    pytest.param(12, 2, 128, 37, 37, id="1p5b_s37"),
    pytest.param(14, 2, 64, 200, 200, id="0p5b_s200"),
    pytest.param(16, 2, 128, 300, 1100, id="3b_prefix800"),
    pytest.param(28, 4, 128, 1, 65, id="7b_s1_prefix64"),
    pytest.param(16, 2, 128, 1344, 1344, id="vl3b_s1344"),
]


@pytest.mark.parametrize("hq,hkv,hd,S,L", PREFILL_CASES)
def test_attention_prefill_matches_oracle(gpu, hq, hkv, hd, S, L):
    torch.manual_seed(0)
    q = torch.randn(S, hq, hd, dtype=torch.bfloat16)
    k = torch.randn(L, hkv, hd, dtype=torch.bfloat16)
    v = torch.randn(L, hkv, hd, dtype=torch.bfloat16)
    ref = O.attention_prefill(q, k, v, O.AttnCtx(hq, hkv, hd, q_rope_pos_offset=L - S), causal=True)
    ctx = C.make_attention_ctx(hq, hkv, hd, q_rope_pos_offset=L - S)
    qg, kg, vg = q.to(gpu), k.to(gpu), v.to(gpu)
    o = torch.empty(S, hq * hd, dtype=torch.bfloat16, device=gpu)
    C.call("efm_attention_prefill", ctx, ptr(qg), ptr(kg), ptr(vg), ptr(o), S, L, 1, stream())
    torch.cuda.synchronize()
    # P is rounded to bf16 before the PV product (as in FlashAttention-2 / FlashInfer)
    assert_close_bf16(o.reshape(S, hq, hd), ref, rtol=2e-2, atol=2e-2, what=f"prefill S={S} L={L}")


def test_attention_prefill_strided_qkv_no_rope_and_noncausal(gpu):
    """q taken from a fused QKV buffer (q_stride_n = qkv_total), pos NONE (M-RoPE models),
    and the non-causal mode."""
    torch.manual_seed(1)
    hq, hkv, hd, S = 16, 2, 128, 130
    tot = (hq + 2 * hkv) * hd
    qkv = torch.randn(S, tot, dtype=torch.bfloat16)
    q = qkv[:, : hq * hd].reshape(S, hq, hd)
    k = qkv[:, hq * hd: (hq + hkv) * hd].reshape(S, hkv, hd).contiguous()
    v = qkv[:, (hq + hkv) * hd:].reshape(S, hkv, hd).contiguous()
    for causal in (1, 0):
        ref = O.attention(q, k, v, torch.arange(S), O.AttnCtx(hq, hkv, hd, rope=False),
                          causal_offset=0 if causal else None)
        ctx = C.make_attention_ctx(hq, hkv, hd, rope=False, q_stride_n=tot, q_stride_h=hd)
        qkvg, kg, vg = qkv.to(gpu), k.to(gpu), v.to(gpu)
        o = torch.empty(S, hq * hd, dtype=torch.bfloat16, device=gpu)
        C.call("efm_attention_prefill", ctx, ptr(qkvg), ptr(kg), ptr(vg), ptr(o), S, S, causal, stream())
        torch.cuda.synchronize()
        assert_close_bf16(o.reshape(S, hq, hd), ref, rtol=2e-2, atol=2e-2, what=f"causal={causal}")


PIPE_CASES = [
    pytest.param(12, 2, 1, 1, 1, "none", id="s1"),
    pytest.param(12, 2, 77, 77, 1, "prerot", id="s77_prerot"),
    pytest.param(16, 2, 300, 1100, 1, "prerot", id="3b_prefix800_prerot"),
    pytest.param(28, 4, 513, 513, 0, "none", id="7b_s513_noncausal"),
    pytest.param(28, 4, 1000, 1000, 1, "none", id="7b_s1000"),
    pytest.param(16, 2, 1344, 1344, 1, "none", id="vl3b_s1344"),
    pytest.param(12, 2, 255, 1025, 0, "prerot", id="noncausal_prefix"),
    pytest.param(12, 2, 512, 512, 1, "none", id="1p5b_s512"),
]


@pytest.mark.parametrize("shape", ["2", "4", "8"])
@pytest.mark.parametrize("hq,hkv,S,L,causal,mode", PIPE_CASES)
def test_attention_prefill_pipelined_matches_oracle(gpu, knob, shape, hq, hkv, S, L, causal, mode):
    """head_dim 128 with keys already rotated (pos NONE, or RoPE on q only with
    k_already_prerotated) runs the global_load_lds ring kernel, in every workgroup shape
    (2 or 4 waves over a 2-deep ring, 8 waves over a 4-deep ring)."""
    knob(C.EFM_KNOB_PREFILL_SHAPE, int(shape))
    torch.manual_seed(S + L)
    hd = 128
    q = torch.randn(S, hq, hd, dtype=torch.bfloat16)
    k = torch.randn(L, hkv, hd, dtype=torch.bfloat16)
    v = torch.randn(L, hkv, hd, dtype=torch.bfloat16)
    if mode == "none":
        octx = O.AttnCtx(hq, hkv, hd, rope=False)
        ctx = C.make_attention_ctx(hq, hkv, hd, rope=False)
        kin = k
    else:
        octx = O.AttnCtx(hq, hkv, hd, q_rope_pos_offset=L - S)
        ctx = C.make_attention_ctx(hq, hkv, hd, q_rope_pos_offset=L - S, k_already_prerotated=True)
        kin = O.rope_llama(k, torch.arange(L), 1.0e6).to(torch.bfloat16)
    ref = O.attention(q, k, v, torch.arange(S) + (L - S), octx, causal_offset=(L - S) if causal else None)
    qg, kg, vg = q.to(gpu), kin.to(gpu), v.to(gpu)
    o = torch.empty(S, hq * hd, dtype=torch.bfloat16, device=gpu)
    C.call("efm_attention_prefill", ctx, ptr(qg), ptr(kg), ptr(vg), ptr(o), S, L, causal, stream())
    torch.cuda.synchronize()
    assert_close_bf16(o.reshape(S, hq, hd), ref, rtol=2e-2, atol=2e-2, what=f"pipelined S={S} L={L} {mode}")


@pytest.mark.parametrize("shape", ["2", "4", "8"])
def test_attention_prefill_pipelined_matches_register_kernel_c4(gpu, knob, shape):
    """BASELINE C4 shape (28/4 heads, S = 4096, causal): the pipelined kernel (every
    workgroup shape) against the register-staged one (EFM_KNOB_PREFILL_REGISTER)."""
    knob(C.EFM_KNOB_PREFILL_SHAPE, int(shape))
    torch.manual_seed(44)
    hq, hkv, hd, S = 28, 4, 128, 4096
    q = torch.randn(S, hq, hd, dtype=torch.bfloat16, device=gpu)
    k = torch.randn(S, hkv, hd, dtype=torch.bfloat16, device=gpu)
    v = torch.randn(S, hkv, hd, dtype=torch.bfloat16, device=gpu)
    ctx = C.make_attention_ctx(hq, hkv, hd, rope=False)
    outs = []
    for pipe in ("1", "0"):
        knob(C.EFM_KNOB_PREFILL_REGISTER, 1 if pipe == "0" else 0)
        o = torch.empty(S, hq * hd, dtype=torch.bfloat16, device=gpu)
        C.call("efm_attention_prefill", ctx, ptr(q), ptr(k), ptr(v), ptr(o), S, S, 1, stream())
        torch.cuda.synchronize()
        outs.append(o)
    assert torch.isfinite(outs[0].float()).all()
    assert_close_bf16(outs[0], outs[1], rtol=2e-2, atol=2e-2, what="pipelined vs register kernel")
    # spot rows against the oracle (first, middle, last query rows of every head)
    for r in (0, 1, 2047, 4095):
        ref = O.attention(q[r:r + 1].cpu(), k[:r + 1].cpu(), v[:r + 1].cpu(), torch.tensor([r]),
                          O.AttnCtx(hq, hkv, hd, rope=False), causal_offset=None)
        assert_close_bf16(outs[0][r].reshape(1, hq, hd), ref, rtol=2e-2, atol=2e-2, what=f"C4 row {r} vs oracle")


SPLIT_CASES = [
    # hq, hkv, hd, S, L, causal, rope: tile and block edges, one key, one row behind a prefix,
    # grids by XCD (1, 2, 4, 8 KV heads) and plain (3); w8 / w4 / w2: waves per block at 256 CUs
    # (8 up to half a block per CU, or a block per CU and 1024 keys; 2 past 5 blocks per CU where
    # nothing is rotated inside)
    pytest.param(12, 2, 128, 1, 1, 1, "none", id="w8_one_key"),
    pytest.param(12, 2, 128, 32, 32, 1, "none", id="w8_one_block"),
    pytest.param(12, 2, 128, 33, 2050, 1, "read", id="w8_rope"),
    pytest.param(28, 4, 128, 1, 8193, 1, "prerot", id="w8_row_behind_8k"),
    pytest.param(6, 3, 128, 65, 161, 1, "none", id="w8_plain_grid"),
    pytest.param(8, 8, 128, 900, 900, 1, "read", id="w4_rope_8_kv_heads"),
    pytest.param(28, 4, 128, 1472, 1475, 1, "prerot", id="w4_prerot_many_blocks"),
    pytest.param(28, 4, 128, 1472, 1475, 1, "none", id="w2"),
    pytest.param(28, 4, 128, 1489, 1600, 0, "none", id="w2_noncausal"),
    pytest.param(12, 2, 128, 130, 97 + 130, 0, "read", id="w8_noncausal_rope"),
    pytest.param(12, 2, 128, 509, 509, 1, "none", id="w4"),
    pytest.param(16, 2, 128, 1343, 1345, 1, "none", id="w4_two_behind"),
    pytest.param(9, 3, 128, 451, 613, 0, "none", id="w4_plain_grid_noncausal"),
    pytest.param(12, 2, 128, 400, 613, 0, "prerot", id="w4_noncausal_prerot"),
    pytest.param(14, 2, 64, 1, 1, 1, "read", id="hd64_w8_one_key"),
    pytest.param(14, 2, 64, 31, 95, 1, "none", id="hd64_w8_half_tile"),
    pytest.param(14, 2, 64, 19, 1531, 1, "prerot", id="hd64_w8"),
    pytest.param(7, 1, 64, 1200, 1200, 1, "read", id="hd64_w4_rope"),
    pytest.param(16, 8, 64, 97, 128, 0, "none", id="hd64_w8_noncausal"),
    pytest.param(14, 2, 64, 700, 700, 1, "none", id="hd64_w4"),
    pytest.param(14, 2, 64, 613, 650, 0, "none", id="hd64_w4_noncausal"),
    pytest.param(14, 2, 64, 320, 1001, 1, "prerot", id="hd64_w4_behind_prefix"),
]


@pytest.mark.parametrize("hq,hkv,hd,S,L,causal,mode", SPLIT_CASES)
def test_attention_prefill_split_matches_oracle(gpu, knob, hq, hkv, hd, S, L, causal, mode):
    """The kernel that splits a 32-row block's keys over the waves of a workgroup, against
    the oracle and the register-staged kernel, on strided q, k and v (a padded row each)."""
    torch.manual_seed(S + L + hd)
    q = torch.randn(S, hq, hd, dtype=torch.bfloat16)
    k = torch.randn(L, hkv, hd, dtype=torch.bfloat16)
    v = torch.randn(L, hkv, hd, dtype=torch.bfloat16)
    octx = O.AttnCtx(hq, hkv, hd, rope=mode != "none", q_rope_pos_offset=L - S)
    ref = O.attention(q, k, v, torch.arange(S) + (L - S), octx, causal_offset=(L - S) if causal else None)
    kin = O.rope_llama(k, torch.arange(L), 1.0e6).to(torch.bfloat16) if mode == "prerot" else k

    def padded(t, extra):   # rows of t with `extra` elements of NaN behind each
        rows = torch.full((t.shape[0], t.shape[1] * hd + extra), float("nan"), dtype=torch.bfloat16)
        rows[:, : t.shape[1] * hd] = t.reshape(t.shape[0], -1)
        return rows.to(gpu)

    qg, kg, vg = padded(q, 8), padded(kin, 16), padded(v, 24)
    ctx = C.make_attention_ctx(hq, hkv, hd, rope=mode != "none", q_rope_pos_offset=L - S,
                               k_already_prerotated=mode == "prerot", q_stride_n=hq * hd + 8, q_stride_h=hd,
                               k_stride_n=hkv * hd + 16, k_stride_h=hd, kv_stride_n=hkv * hd + 24, kv_stride_h=hd)
    outs = []
    for register in (0, 1):
        knob(C.EFM_KNOB_PREFILL_REGISTER, register)
        o = torch.full((S + 1, hq * hd), -7.0, dtype=torch.bfloat16, device=gpu)
        C.call("efm_attention_prefill", ctx, ptr(qg), ptr(kg), ptr(vg), ptr(o), S, L, causal, stream())
        torch.cuda.synchronize()
        assert (o[S] == -7.0).all()
        outs.append(o[:S].reshape(S, hq, hd))
    # P is rounded to bf16 before the PV product
    assert_close_bf16(outs[0], ref, rtol=2e-2, atol=2e-2, what="split vs oracle")
    assert_close_bf16(outs[0], outs[1], rtol=2e-2, atol=2e-2, what="split vs register-staged")


@pytest.mark.parametrize("op,hq,hkv,hd,S,L,causal,rope", [
    pytest.param("bf16", 14, 2, 64, 1259, 2371, 1, True, id="hd64_rope_behind_prefix"),
    pytest.param("bf16", 14, 2, 64, 31, 1459, 0, True, id="hd64_rope_not_causal"),
    pytest.param("bf16", 9, 9, 64, 600, 1800, 1, False, id="hd64_no_rope"),
    pytest.param("bf16", 12, 2, 128, 388, 388, 0, True, id="rope_not_causal"),
    pytest.param("bf16", 28, 4, 128, 35, 1295, 1, True, id="rope_behind_prefix"),
    pytest.param("sage", 14, 2, 64, 803, 1079, 0, False, id="sage_hd64_not_causal"),
    pytest.param("sage", 14, 2, 64, 74, 713, 1, False, id="sage_hd64_behind_prefix"),
])
def test_attention_split_error_against_64_bits(gpu, knob, op, hq, hkv, hd, S, L, causal, rope):
    """Where the split kernels took over calls of the register-staged ones, they are as close to
    64 bits (over the int8 operands for Sage): both round each p once, so their relative errors
    over a whole output are equal but for the sample (within 0.2 % over 160 shapes; 0.5 %
    allowed). Shapes where rows see many keys: there the heaviest weight counts most, which is
    exact only with the true running max as the reference point."""
    g = torch.Generator(device=gpu).manual_seed(S + L)
    q, k, v = (torch.empty(n, h, hd, dtype=torch.bfloat16, device=gpu).normal_(generator=g)
               for n, h in ((S, hq), (L, hkv), (L, hkv)))
    ctx = C.make_attention_ctx(hq, hkv, hd, rope=rope, q_rope_pos_offset=L - S)
    qf, kf = q.double(), k.double()
    if op == "sage":
        q8, k8 = torch.empty(q.shape, dtype=torch.int8, device=gpu), torch.empty(k.shape, dtype=torch.int8, device=gpu)
        sq, sk = torch.empty((S + 127) // 128, hq, device=gpu), torch.empty((L + 127) // 128, hkv, device=gpu)
        km = torch.empty(hkv, hd, device=gpu)
        C.call("efm_sage_quantize", ctx, ptr(q), ptr(k), S, L, ptr(q8), ptr(sq), ptr(k8), ptr(sk), ptr(km), stream())
        qf, kf = (x.double() * sc.double()[torch.arange(x.shape[0], device=gpu) // 128][..., None]
                  for x, sc in ((q8, sq), (k8, sk)))
    elif rope:
        half = hd // 2
        freq = 1.0e6 ** (-torch.arange(half, device=gpu, dtype=torch.float64) / half)
        rot = lambda x, pos: (lambda a, b, c, s: torch.cat([a * c - b * s, b * c + a * s], -1))(
            x[..., :half], x[..., half:], *(f(pos.double()[:, None] * freq)[:, None] for f in (torch.cos, torch.sin)))
        pos = torch.arange(L, device=gpu)
        qf, kf = rot(qf, pos[L - S:]), rot(kf, pos)
    ref = torch.empty_like(qf)
    for h in range(hq):
        s = qf[:, h] @ kf[:, h * hkv // hq].T.contiguous() / math.sqrt(hd)
        if causal:
            s.masked_fill_(torch.ones(S, L, dtype=torch.bool, device=gpu).triu(L - S + 1), -math.inf)
        ref[:, h] = torch.softmax(s, -1) @ v[:, h * hkv // hq].double()
    errs = []
    ws = torch.empty(C.load().efm_attention_prefill_sage_int8_workspace_bytes(ctx, S, L), dtype=torch.uint8, device=gpu)
    for register in (0, 1):
        knob(C.EFM_KNOB_PREFILL_REGISTER, register)
        o = torch.empty_like(q)
        args = (ctx, ptr(q), ptr(k), ptr(v), ptr(o), S, L, causal)
        if op == "sage":
            C.call("efm_attention_prefill_sage_int8", *args, ptr(ws), ws.numel(), stream())
        else:
            C.call("efm_attention_prefill", *args, stream())
        torch.cuda.synchronize()
        errs.append(float((o.double() - ref).norm() / ref.norm()))
    assert errs[0] <= 1.005 * errs[1], errs


@pytest.mark.parametrize("hd,mode,off", [
    pytest.param(128, "prerot", 3, id="hd128_prerotated"),
    pytest.param(128, "read", 3, id="hd128_rope"),
    pytest.param(64, "read", 70000, id="hd64_rope_far"),
    pytest.param(64, "prerot", 3, id="hd64_prerotated"),
])
def test_attention_prefill_split_query_rotation(gpu, knob, hd, mode, off):
    """The query's sine and cosine in the split kernel are those of fp32 (sincosf), once per row.
    Row i holds one pair (x0, x1) of bf16 values whose rotated x0 nearly cancels (1 to 3e-5 of
    the pair), so that an error e of the sine or cosine is one of e / 2e-5 in its score; key 0 is
    that channel alone, the other keys are zero, and the output is key 0's weight. Bound on the
    rotated value: sine and cosine within an ulp (2^-24) and one product rounded to fp32, 2 x
    2^-24 of the pair in all, and 2^-9 of itself where it is rounded to bf16; the weight's slope
    in the score is p (1 - p), and it is rounded to bf16 twice. (Hardware sine and cosine: 1.6 to
    1.9 times the bound.)"""
    S, d, half = 512, 1, hd // 2
    freq = np.float32(math.exp(-2.0 * d / hd * math.log(1.0e6)))
    ang = (np.arange(S, dtype=np.float32) + np.float32(off)) * freq
    c, s = np.cos(ang.astype(np.float64)), np.sin(ang.astype(np.float64))
    pair, y0 = np.zeros((S, 2)), np.zeros(S)
    x0 = np.arange(128, 256) / 128.0   # bf16 mantissas, and the largest bf16 x1 of no more than x0 |c / s|
    for i in range(S):
        x1 = x0 * abs(c[i] / s[i])
        ulp = 2.0 ** (np.floor(np.log2(x1)) - 7)
        x1 = np.floor(x1 / ulp) * ulp
        y = x0 * abs(c[i]) - x1 * abs(s[i])
        j = np.argmin(np.abs(y / np.hypot(x0, x1) - 2e-5))
        pair[i], y0[i] = (x0[j] * np.sign(c[i]), x1[j] * np.sign(s[i])), y[j]
    scale = 2.0 ** np.round(np.log2(4.1 * math.sqrt(hd) / y0) - 8)   # times key 0's 2^8
    pair, y0 = pair * scale[:, None], y0 * scale
    q = torch.zeros(S, 1, hd, dtype=torch.float64)
    q[:, 0, d], q[:, 0, d + half] = torch.from_numpy(pair[:, 0]), torch.from_numpy(pair[:, 1])
    assert torch.equal(q.bfloat16().double(), q)
    k, v = torch.zeros(S, 1, hd), torch.zeros(S, 1, hd)
    k[0, 0, d], v[0] = 256.0, 1.0
    sc = y0 * 256.0 / math.sqrt(hd)
    ref = np.exp(sc) / (np.exp(sc) + S - 1)
    use = (y0 / np.hypot(*pair.T) > 1e-5) & (y0 / np.hypot(*pair.T) < 3e-5)
    assert use.sum() > 100
    err_s = 256.0 / math.sqrt(hd) * (2 * 2.0 ** -24 * np.hypot(*pair.T) + 2.0 ** -9 * y0)
    bound = ref * (1 - ref) * err_s * 1.1 + 2.0 ** -8 * ref
    qg, kg, vg = (t.to(torch.bfloat16).to(gpu) for t in (q, k, v))
    ctx = C.make_attention_ctx(1, 1, hd, rope=True, q_rope_pos_offset=off, k_already_prerotated=mode == "prerot")
    for register in (1, 0):
        knob(C.EFM_KNOB_PREFILL_REGISTER, register)
        o = torch.empty_like(qg)
        C.call("efm_attention_prefill", ctx, ptr(qg), ptr(kg), ptr(vg), ptr(o), S, S, 0, stream())
        torch.cuda.synchronize()
        got = o[:, 0, 0].double().cpu().numpy()
        over = np.abs(got - ref)[use] / bound[use]
        assert over.max() <= 1, (register, float(over.max()))


@pytest.mark.parametrize("op,hq,hkv,hd,L,mode", [
    pytest.param("bf16", 14, 2, 64, 200, "none", id="hd64"),
    pytest.param("bf16", 14, 2, 64, 1100, "read", id="hd64_rope_eight_waves"),
    pytest.param("bf16", 12, 2, 128, 200, "read", id="rope"),
    pytest.param("sage", 14, 2, 64, 200, "none", id="sage_hd64"),
    pytest.param("sage", 14, 2, 64, 2100, "none", id="sage_hd64_eight_waves"),
])
def test_attention_split_rows_without_weight(gpu, knob, op, hq, hkv, hd, L, mode):
    """Rows whose visible scores all overflow to -inf are 0, as in the register-staged kernel;
    rows that also see a key of finite score (bf16: key L / 2 and later are 0) are its value."""
    q, k = torch.zeros(L, hq, hd), torch.zeros(L, hkv, hd)
    q[:, :, hd // 2 - 1] = 2.0 ** 100   # the pair of the lowest frequency
    k[: L // 2, :, hd // 2 - 1] = -(2.0 ** 100)
    if op == "sage":   # K less its mean: both signs, so only the first half of the rows is finite
        k[L // 2:, :, hd // 2 - 1] = 2.0 ** 100
    v = torch.randn(L, hkv, hd, generator=torch.Generator().manual_seed(L))
    qg, kg, vg = (t.to(torch.bfloat16).to(gpu) for t in (q, k, v))
    ctx = C.make_attention_ctx(hq, hkv, hd, rope=mode == "read")
    ws = torch.zeros(C.load().efm_attention_prefill_sage_int8_workspace_bytes(ctx, L, L), dtype=torch.uint8, device=gpu)
    for register in (1, 0):
        knob(C.EFM_KNOB_PREFILL_REGISTER, register)
        o = torch.full_like(qg, -7.0)
        args = (ctx, ptr(qg), ptr(kg), ptr(vg), ptr(o), L, L, 1)
        if op == "sage":
            C.call("efm_attention_prefill_sage_int8", *args, ptr(ws), ws.numel(), stream())
        else:
            C.call("efm_attention_prefill", *args, stream())
        torch.cuda.synchronize()
        assert (o[: L // 2] == 0).all(), register
        if op == "bf16":
            h = torch.arange(hq, device=gpu) * hkv // hq
            assert torch.equal(o[L // 2], vg[L // 2, h]), register
            ref = (vg[L // 2:, h].double().cumsum(0) / torch.arange(1, L - L // 2 + 1, device=gpu)[:, None, None])
            assert_close_bf16(o[L // 2:], ref.to(torch.bfloat16), rtol=2e-2, atol=2e-2)


def test_attention_prefill_unaligned_rows(gpu):
    """head_dim 64 rows at an 8-byte (not 16-byte) aligned address: accepted as before."""
    torch.manual_seed(5)
    hq, hkv, hd, S = 14, 2, 64, 70
    q, k, v = (torch.randn(S, h, hd, dtype=torch.bfloat16) for h in (hq, hkv, hkv))
    off = [torch.zeros(t.numel() + 4, dtype=torch.bfloat16, device=gpu) for t in (q, k, v)]
    for d, t in zip(off, (q, k, v)):
        d[4:] = t.reshape(-1).to(gpu)
    o = torch.empty(S, hq * hd, dtype=torch.bfloat16, device=gpu)
    C.call("efm_attention_prefill", C.make_attention_ctx(hq, hkv, hd), *(d.data_ptr() + 8 for d in off), ptr(o), S, S, 1,
           stream())
    torch.cuda.synchronize()
    ref = O.attention_prefill(q, k, v, O.AttnCtx(hq, hkv, hd), causal=True)
    assert_close_bf16(o.reshape(S, hq, hd), ref, rtol=2e-2, atol=2e-2)


@pytest.mark.parametrize("S", [70, 1500])
@pytest.mark.parametrize("op,rope", [("bf16", False), ("bf16", True), ("sage", False)])
@pytest.mark.parametrize("how", ["offset", "stride"])
def test_attention_prefill_operands_without_dma(gpu, knob, op, rope, how, S):
    """head_dim 128 operands that the tile loads cannot take (rows 8 bytes off a 16-byte
    boundary; rows so far apart that a tile spans more than 32-bit offsets) run the
    register-staged kernel, at row counts where aligned ones run the split and the pipelined
    kernel: the same bits as the same rows through that kernel, packed."""
    hq, hkv, hd = 28, 4, 128
    L = 66 if how == "stride" else S
    S = min(S, L)
    g = torch.Generator(device=gpu).manual_seed(S)
    q, k, v = (torch.empty(n, h, hd, dtype=torch.bfloat16, device=gpu).normal_(generator=g)
               for n, h in ((S, hq), (L, hkv), (L, hkv)))
    moved, kw = [q, k, v], {}
    only_v = op == "sage"   # its q and k are quantised by another kernel
    if how == "offset":
        for i in (2,) if only_v else (0, 1, 2):
            t = moved[i]
            moved[i] = torch.zeros(t.numel() + 4, dtype=torch.bfloat16, device=gpu)[4:].view_as(t).copy_(t)
            assert moved[i].data_ptr() % 16 == 8
    else:   # one buffer of L rows, K and V side by side in each
        sn = 1 << 25
        rows = torch.empty(L, sn, dtype=torch.bfloat16, device=gpu)
        kw = dict(kv_stride_n=sn, kv_stride_h=hd)
        moved[2] = rows[:, hkv * hd:2 * hkv * hd].copy_(v.reshape(L, -1))
        if not only_v:
            kw.update(k_stride_n=sn, k_stride_h=hd)
            moved[1] = rows[:, :hkv * hd].copy_(k.reshape(L, -1))
    outs = []
    for register, ts, c in ((1, (q, k, v), {}), (0, moved, kw)):
        knob(C.EFM_KNOB_PREFILL_REGISTER, register)
        ctx = C.make_attention_ctx(hq, hkv, hd, rope=rope, k_already_prerotated=rope, **c)
        ws = torch.zeros(C.load().efm_attention_prefill_sage_int8_workspace_bytes(ctx, S, L), dtype=torch.uint8, device=gpu)
        o = torch.empty_like(q)
        args = (ctx, *(ptr(t) for t in ts), ptr(o), S, L, 1)
        if op == "sage":
            C.call("efm_attention_prefill_sage_int8", *args, ptr(ws), ws.numel(), stream())
        else:
            C.call("efm_attention_prefill", *args, stream())
        torch.cuda.synchronize()
        outs.append(o)
    assert torch.equal(*outs)


def test_attention_prefill_last_row_equals_decode(gpu):
    """The last prefill row equals single-query decode over the same cache (the
    reference's prefill/decode consistency)."""
    torch.manual_seed(2)
    hq, hkv, hd, L = 12, 2, 128, 700
    q = torch.randn(L, hq, hd, dtype=torch.bfloat16, device=gpu)
    k = torch.randn(L, hkv, hd, dtype=torch.bfloat16, device=gpu)
    v = torch.randn(L, hkv, hd, dtype=torch.bfloat16, device=gpu)
    o = torch.empty(L, hq * hd, dtype=torch.bfloat16, device=gpu)
    C.call("efm_attention_prefill", C.make_attention_ctx(hq, hkv, hd), ptr(q), ptr(k), ptr(v), ptr(o), L, L, 1,
           stream())
    dec, _ = _decode(C.make_attention_ctx(hq, hkv, hd), q[-1:].contiguous(), k, v, L)
    assert_close_bf16(o[-1].reshape(1, hq, hd), dec, rtol=2e-2, atol=2e-2)


def test_mrope_matches_oracle(gpu):
    torch.manual_seed(0)
    S, hq, hkv, hd = 70, 16, 2, 128
    sections = (16, 24, 24)
    q = torch.randn(S, hq, hd, dtype=torch.bfloat16)
    k = torch.randn(S, hkv, hd, dtype=torch.bfloat16)
    pos = torch.stack([torch.zeros(S, dtype=torch.int32), torch.arange(S, dtype=torch.int32) // 7,
                       torch.arange(S, dtype=torch.int32) % 7]) + 3
    qg, kg, pg = q.to(gpu), k.to(gpu), pos.to(gpu)
    C.call("efm_mrope", ptr(qg), ptr(kg), ptr(pg), S, S, hq, hkv, hd, 0, 0, *sections, 1.0e6, 1.0, stream())
    torch.cuda.synchronize()
    assert_close_bf16(qg, O.mrope(q, pos, sections, 1.0e6), what="mrope q")
    assert_close_bf16(kg, O.mrope(k, pos, sections, 1.0e6), what="mrope k")


def test_decode_mrope_write_kv(gpu):
    torch.manual_seed(0)
    hq, hkv, hd = 16, 2, 128
    sections = (16, 24, 24)
    qkv = torch.randn(1, (hq + 2 * hkv) * hd, dtype=torch.bfloat16)
    pos = torch.tensor([40, 41, 45], dtype=torch.int32)
    rows = 50
    qkvg, pg = qkv.to(gpu), pos.to(gpu)
    kc = torch.zeros(rows, hkv * hd, dtype=torch.bfloat16, device=gpu)
    vc = torch.zeros(rows, hkv * hd, dtype=torch.bfloat16, device=gpu)
    qd = torch.empty(1, hq * hd, dtype=torch.bfloat16, device=gpu)
    d_len = torch.tensor([31], dtype=torch.int32, device=gpu)
    base = qkvg.data_ptr()
    C.call("efm_decode_mrope_write_kv", base, base + hq * hd * 2, base + (hq + hkv) * hd * 2, ptr(qd), ptr(kc),
           ptr(vc), hq, hkv, hd, ptr(pg), *sections, 1.0e6, 1.0, ptr(d_len), stream())
    torch.cuda.synchronize()
    q = qkv[:, : hq * hd].reshape(1, hq, hd)
    k = qkv[:, hq * hd: (hq + hkv) * hd].reshape(1, hkv, hd)
    p3 = pos.reshape(3, 1)
    assert_close_bf16(qd.reshape(1, hq, hd), O.mrope(q, p3, sections, 1.0e6))
    assert_close_bf16(kc[30].reshape(1, hkv, hd), O.mrope(k, p3, sections, 1.0e6))
    assert torch.equal(vc[30].cpu(), qkv[0, (hq + hkv) * hd:])
    assert kc[:30].abs().sum() == 0 and kc[31:].abs().sum() == 0


def test_finalize_indexed(gpu):
    resp = torch.full((8,), -1, dtype=torch.int32, device=gpu)
    step = torch.zeros(1, dtype=torch.int32, device=gpu)
    d_len = torch.tensor([10], dtype=torch.int32, device=gpu)
    tok = torch.zeros(1, dtype=torch.int32, device=gpu)
    for i in range(10):
        tok.fill_(100 + i)
        C.call("efm_finalize_decode_token_indexed", ptr(tok), ptr(resp), ptr(step), ptr(d_len), 8, stream())
    torch.cuda.synchronize()
    assert resp.cpu().tolist() == [100 + i for i in range(8)]
    assert int(step.item()) == 10 and int(d_len.item()) == 20


@pytest.mark.parametrize("hq,hkv,hd,hidden", [pytest.param(12, 2, 128, 1536, id="1p5b"),
                                               pytest.param(14, 2, 64, 896, id="0p5b"),
                                               pytest.param(16, 2, 128, 2048, id="vl3b")])
@pytest.mark.parametrize("max_kv,kv_len,rope", [(768, 1, True), (768, 100, True), (768, 640, True),
                                                (768, 767, True), (768, 640, False), (1024, 1024, False),
                                                (1024, 129, True)])
def test_decode_attention_partials_merge_o_proj(gpu, hq, hkv, hd, hidden, max_kv, kv_len, rope):
    """Split partials + merge folded into the o_proj GEMV == attention then o_proj, on
    rotate-on-read and rotated caches, up to the 1024 rows (8 splits) it takes."""
    torch.manual_seed(0)
    q = torch.randn(1, hq, hd, dtype=torch.bfloat16)
    k = torch.randn(max_kv, hkv, hd, dtype=torch.bfloat16)
    v = torch.randn(max_kv, hkv, hd, dtype=torch.bfloat16)
    wo = (torch.randn(hidden, hq * hd) * 0.02).to(torch.bfloat16)
    ctx = C.make_attention_ctx(hq, hkv, hd, rope=rope)
    qg, kg, vg, wg = q.to(gpu), k.to(gpu), v.to(gpu), wo.to(gpu)
    d_len = torch.tensor([kv_len], dtype=torch.int32, device=gpu)
    ws = torch.zeros(C.load().efm_attention_decode_workspace_bytes(ctx, max_kv), dtype=torch.uint8, device=gpu)
    out = torch.empty(1, hidden, dtype=torch.bfloat16, device=gpu)
    for _ in range(2):
        C.call("efm_decode_attention_partials", ctx, ptr(qg), ptr(kg), ptr(vg), ptr(d_len), max_kv, ptr(ws),
               ws.numel(), stream())
        C.call("efm_decode_attention_merge_o_proj", ctx, ptr(d_len), max_kv, ptr(ws), ws.numel(), ptr(wg), hidden,
               ptr(out), stream())
    torch.cuda.synchronize()
    att = O.attention_decode(q, k, v, kv_len, O.AttnCtx(hq, hkv, hd, rope=rope))
    ref = O.linear(att.reshape(1, hq * hd), wo)
    assert_close_bf16(out, ref, rtol=2e-2, atol=2e-2, what=f"partials+merge max={max_kv} kv={kv_len}")


@pytest.mark.parametrize("hq,hkv,hidden", [pytest.param(14, 2, 896, id="0p5b"), pytest.param(16, 2, 1024, id="w1024"),
                                            pytest.param(8, 8, 512, id="mha")])
@pytest.mark.parametrize("max_kv,kv_len", [(1, 1), (40, 17), (1025, 1025), (1025, 1), (1025, 64), (1025, 65),
                                           (1536, 1536), (1536, 700)])
def test_decode_attention_partials_merge_o_proj_narrow(gpu, hq, hkv, hidden, max_kv, kv_len):
    """head_dim 64 with query widths up to 1024: one-wave partials of 32 / 64 keys (up to
    24 splits, caches up to 1536 rows) merged in the narrow o_proj prologue == the oracle's
    attention then o_proj, and == efm_attention_decode + efm_linear to rounding. Rows past
    the length hold Inf / NaN and must not leak in; two calls in a row agree bit for bit."""
    hd = 64
    torch.manual_seed(1)
    q = torch.randn(1, hq, hd, dtype=torch.bfloat16)
    k = torch.randn(max_kv, hkv, hd, dtype=torch.bfloat16)
    v = torch.randn(max_kv, hkv, hd, dtype=torch.bfloat16)
    wo = (torch.randn(hidden, hq * hd) * 0.02).to(torch.bfloat16)
    ctx = C.make_attention_ctx(hq, hkv, hd, rope=False)
    lib = C.load()
    assert lib.efm_decode_attention_merge_o_proj_supported(ctx, max_kv) == C.EFM_OK
    qg, kg, vg, wg = q.to(gpu), k.to(gpu), v.to(gpu), wo.to(gpu)
    kg[kv_len:] = float("inf")
    vg[kv_len:] = float("nan")
    d_len = torch.tensor([kv_len], dtype=torch.int32, device=gpu)
    ws = torch.zeros(lib.efm_attention_decode_workspace_bytes(ctx, max_kv), dtype=torch.uint8, device=gpu)
    outs = []
    for _ in range(2):
        out = torch.empty(1, hidden, dtype=torch.bfloat16, device=gpu)
        C.call("efm_decode_attention_partials", ctx, ptr(qg), ptr(kg), ptr(vg), ptr(d_len), max_kv, ptr(ws),
               ws.numel(), stream())
        C.call("efm_decode_attention_merge_o_proj", ctx, ptr(d_len), max_kv, ptr(ws), ws.numel(), ptr(wg), hidden,
               ptr(out), stream())
        outs.append(out)
    att = torch.empty(1, hq * hd, dtype=torch.bfloat16, device=gpu)
    ref_gpu = torch.empty(1, hidden, dtype=torch.bfloat16, device=gpu)
    C.call("efm_attention_decode", ctx, ptr(qg), ptr(kg), ptr(vg), ptr(att), 0, ptr(d_len), max_kv, ptr(ws),
           ws.numel(), stream())
    C.call("efm_linear", 1, hq * hd, hidden, ptr(att), ptr(wg), None, ptr(ref_gpu), C.EFM_DTYPE_BF16, stream())
    torch.cuda.synchronize()
    assert torch.equal(outs[0], outs[1])
    assert torch.isfinite(outs[0].float()).all()
    ref = O.linear(O.attention_decode(q, k[:kv_len], v[:kv_len], kv_len, O.AttnCtx(hq, hkv, hd, rope=False))
                   .reshape(1, hq * hd), wo)
    what = f"narrow partials+merge {hq}/{hkv} max={max_kv} kv={kv_len}"
    assert_close_bf16(outs[0], ref, rtol=2e-2, atol=2e-2, what=what)
    assert_close_bf16(outs[0], ref_gpu, rtol=2e-2, atol=2e-2, what=what + " vs attention_decode + linear")


@pytest.mark.parametrize("hq,hkv,hidden", [pytest.param(12, 2, 1536, id="1p5b"), pytest.param(16, 2, 2048, id="vl3b"),
                                            pytest.param(16, 4, 2048, id="g4")])
@pytest.mark.parametrize("max_kv,kv_len", [(96, 96), (256, 1), (384, 200), (1025, 1025), (1280, 700), (1536, 1536),
                                           (1536, 1)])
def test_decode_attention_partials_merge_o_proj_head_dim_128_plans(gpu, hq, hkv, hidden, max_kv, kv_len):
    """head_dim 128 beyond the 8-split merge: one-tile (32-key) partials up to 12 splits at
    short caches, and 9-12 splits of 128 keys (the 12-slot prologue) at 1025-1536 rows, ==
    the oracle's attention then o_proj, and == efm_attention_decode + efm_linear to rounding.
    Rows past the length hold Inf / NaN; two calls in a row agree bit for bit."""
    hd = 128
    torch.manual_seed(4)
    q = torch.randn(1, hq, hd, dtype=torch.bfloat16)
    k = torch.randn(max_kv, hkv, hd, dtype=torch.bfloat16)
    v = torch.randn(max_kv, hkv, hd, dtype=torch.bfloat16)
    wo = (torch.randn(hidden, hq * hd) * 0.02).to(torch.bfloat16)
    ctx = C.make_attention_ctx(hq, hkv, hd, rope=False)
    lib = C.load()
    assert lib.efm_decode_attention_merge_o_proj_supported(ctx, max_kv) == C.EFM_OK
    qg, kg, vg, wg = q.to(gpu), k.to(gpu), v.to(gpu), wo.to(gpu)
    kg[kv_len:] = float("inf")
    vg[kv_len:] = float("nan")
    d_len = torch.tensor([kv_len], dtype=torch.int32, device=gpu)
    ws = torch.zeros(lib.efm_attention_decode_workspace_bytes(ctx, max_kv), dtype=torch.uint8, device=gpu)
    outs = []
    for _ in range(2):
        out = torch.empty(1, hidden, dtype=torch.bfloat16, device=gpu)
        C.call("efm_decode_attention_partials", ctx, ptr(qg), ptr(kg), ptr(vg), ptr(d_len), max_kv, ptr(ws),
               ws.numel(), stream())
        C.call("efm_decode_attention_merge_o_proj", ctx, ptr(d_len), max_kv, ptr(ws), ws.numel(), ptr(wg), hidden,
               ptr(out), stream())
        outs.append(out)
    att = torch.empty(1, hq * hd, dtype=torch.bfloat16, device=gpu)
    ref_gpu = torch.empty(1, hidden, dtype=torch.bfloat16, device=gpu)
    C.call("efm_attention_decode", ctx, ptr(qg), ptr(kg), ptr(vg), ptr(att), 0, ptr(d_len), max_kv, ptr(ws),
           ws.numel(), stream())
    C.call("efm_linear", 1, hq * hd, hidden, ptr(att), ptr(wg), None, ptr(ref_gpu), C.EFM_DTYPE_BF16, stream())
    torch.cuda.synchronize()
    assert torch.equal(outs[0], outs[1])
    assert torch.isfinite(outs[0].float()).all()
    ref = O.linear(O.attention_decode(q, k[:kv_len], v[:kv_len], kv_len, O.AttnCtx(hq, hkv, hd, rope=False))
                   .reshape(1, hq * hd), wo)
    what = f"head_dim 128 partials+merge {hq}/{hkv} max={max_kv} kv={kv_len}"
    assert_close_bf16(outs[0], ref, rtol=2e-2, atol=2e-2, what=what)
    assert_close_bf16(outs[0], ref_gpu, rtol=2e-2, atol=2e-2, what=what + " vs attention_decode + linear")


def _sage_inputs(S, L, hq, hkv, hd, seed=0, gpu=None):
    g = torch.Generator().manual_seed(seed)
    q = torch.randn(S, hq, hd, generator=g).to(torch.bfloat16)
    k = (torch.randn(L, hkv, hd, generator=g) + 0.5).to(torch.bfloat16)  # non-zero channel means
    v = torch.randn(L, hkv, hd, generator=g).to(torch.bfloat16)
    return q, k, v


@pytest.mark.parametrize("S,L,hq,hkv,hd", [(300, 300, 28, 4, 128), (129, 257, 4, 2, 64), (1, 40, 8, 1, 128)])
def test_sage_quantize_bit_exact(gpu, S, L, hq, hkv, hd):
    """The int8 path is exact: Q8 / K8 / scales equal the oracle bit for bit (K8 and its
    scales recomputed from the GPU's float64-accumulated K mean)."""
    q, k, v = _sage_inputs(S, L, hq, hkv, hd)
    ctx = C.make_attention_ctx(hq, hkv, hd, rope=False)
    qg, kg = q.to(gpu), k.to(gpu)
    nbq, nbk = (S + 127) // 128, (L + 127) // 128
    q8 = torch.empty(S, hq, hd, dtype=torch.int8, device=gpu)
    k8 = torch.empty(L, hkv, hd, dtype=torch.int8, device=gpu)
    sq = torch.empty(nbq, hq, dtype=torch.float32, device=gpu)
    sk = torch.empty(nbk, hkv, dtype=torch.float32, device=gpu)
    km = torch.empty(hkv, hd, dtype=torch.float32, device=gpu)
    C.call("efm_sage_quantize", ctx, ptr(qg), ptr(kg), S, L, ptr(q8), ptr(sq), ptr(k8), ptr(sk), ptr(km), stream())
    torch.cuda.synchronize()
    ref_km = O.sage_kmean(k)
    torch.testing.assert_close(km.cpu(), ref_km, rtol=2e-7, atol=1e-7)
    rq8, rsq = O.sage_quant_blocks(q.float())
    rk8, rsk = O.sage_quant_blocks(k.float() - km.cpu()[None])
    assert torch.equal(q8.cpu(), rq8) and torch.equal(sq.cpu(), rsq)
    assert torch.equal(k8.cpu(), rk8) and torch.equal(sk.cpu(), rsk)


@pytest.mark.parametrize("S,L,hq,hkv,hd", [(300, 300, 28, 4, 128), (129, 257, 4, 2, 64), (1, 40, 8, 1, 128),
                                           (4096, 4096, 28, 4, 128), (700, 1003, 8, 2, 128)])
def test_sage_attention_quantisation_equals_quantize_entry(gpu, S, L, hq, hkv, hd):
    """The attention entry point takes its K mean from float64 row-slice sums added up by
    the quantisation kernel; its K8 / K scales / K mean (left in the workspace) must equal
    efm_sage_quantize's (one workgroup per channel group) bit for bit."""
    q, k, v = _sage_inputs(S, L, hq, hkv, hd, seed=3)
    ctx = C.make_attention_ctx(hq, hkv, hd, rope=False)
    qg, kg, vg = q.to(gpu), k.to(gpu), v.to(gpu)
    nbq, nbk = (S + 127) // 128, (L + 127) // 128
    q8 = torch.empty(S, hq, hd, dtype=torch.int8, device=gpu)
    k8 = torch.empty(L, hkv, hd, dtype=torch.int8, device=gpu)
    sq = torch.empty(nbq, hq, dtype=torch.float32, device=gpu)
    sk = torch.empty(nbk, hkv, dtype=torch.float32, device=gpu)
    km = torch.empty(hkv, hd, dtype=torch.float32, device=gpu)
    C.call("efm_sage_quantize", ctx, ptr(qg), ptr(kg), S, L, ptr(q8), ptr(sq), ptr(k8), ptr(sk), ptr(km), stream())
    ws = torch.zeros(C.load().efm_attention_prefill_sage_int8_workspace_bytes(ctx, S, L), dtype=torch.uint8,
                     device=gpu)
    o = torch.empty(S, hq * hd, dtype=torch.bfloat16, device=gpu)
    C.call("efm_attention_prefill_sage_int8", ctx, ptr(qg), ptr(kg), ptr(vg), ptr(o), S, L, 1, ptr(ws), ws.numel(),
           stream())
    torch.cuda.synchronize()
    al = lambda x: (x + 255) // 256 * 256
    off_k8 = al(S * hq * hd)
    off_sk = off_k8 + al(L * hkv * hd) + al(nbq * hq * 4)
    off_km = off_sk + al(nbk * hkv * 4)
    w = ws.cpu()
    assert torch.equal(w[off_k8:off_k8 + L * hkv * hd].view(torch.int8).reshape(L, hkv, hd), k8.cpu())
    assert torch.equal(w[off_sk:off_sk + nbk * hkv * 4].view(torch.float32).reshape(nbk, hkv), sk.cpu())
    assert torch.equal(w[off_km:off_km + hkv * hd * 4].view(torch.float32).reshape(hkv, hd), km.cpu())
    torch.testing.assert_close(km.cpu(), O.sage_kmean(k), rtol=2e-7, atol=1e-7)


@pytest.mark.parametrize("S,L,hq,hkv,hd", [(512, 512, 28, 4, 128), (300, 700, 8, 2, 128), (200, 200, 14, 2, 64)])
def test_sage_attention_matches_oracle(gpu, S, L, hq, hkv, hd):
    q, k, v = _sage_inputs(S, L, hq, hkv, hd, seed=1)
    ctx = C.make_attention_ctx(hq, hkv, hd, rope=False)
    qg, kg, vg = q.to(gpu), k.to(gpu), v.to(gpu)
    o = torch.empty(S, hq * hd, dtype=torch.bfloat16, device=gpu)
    ws = torch.zeros(C.load().efm_attention_prefill_sage_int8_workspace_bytes(ctx, S, L), dtype=torch.uint8,
                     device=gpu)
    C.call("efm_attention_prefill_sage_int8", ctx, ptr(qg), ptr(kg), ptr(vg), ptr(o), S, L, 1, ptr(ws), ws.numel(),
           stream())
    torch.cuda.synchronize()
    ref = O.sage_attention(q, k, v, hkv, causal=True)
    assert_close_bf16(o.reshape(S, hq, hd), ref, rtol=2e-2, atol=2e-2, what="sage vs int8 oracle")
    bf = O.attention_prefill(q, k, v, O.AttnCtx(hq, hkv, hd, rope=False), causal=True)
    err = (o.reshape(S, hq, hd).float().cpu() - bf.float()).abs()
    assert float(err.mean()) < 5e-3 and float(err.max()) < 0.1, (float(err.mean()), float(err.max()))


def test_sage_attention_c4_shape_vs_bf16_kernel(gpu):
    """BASELINE config 4 at full size (28/4 heads, hd 128, S 4096, causal): int8 path vs
    the bf16 MFMA prefill kernel on the same inputs (size-independent error bounds)."""
    S, hq, hkv, hd = 4096, 28, 4, 128
    g = torch.Generator(device=gpu).manual_seed(7)
    q = torch.randn(S, hq, hd, generator=g, device=gpu).to(torch.bfloat16)
    k = torch.randn(S, hkv, hd, generator=g, device=gpu).to(torch.bfloat16)
    v = torch.randn(S, hkv, hd, generator=g, device=gpu).to(torch.bfloat16)
    ctx = C.make_attention_ctx(hq, hkv, hd, rope=False)
    o8 = torch.empty(S, hq * hd, dtype=torch.bfloat16, device=gpu)
    ob = torch.empty(S, hq * hd, dtype=torch.bfloat16, device=gpu)
    ws = torch.zeros(C.load().efm_attention_prefill_sage_int8_workspace_bytes(ctx, S, S), dtype=torch.uint8,
                     device=gpu)
    C.call("efm_attention_prefill_sage_int8", ctx, ptr(q), ptr(k), ptr(v), ptr(o8), S, S, 1, ptr(ws), ws.numel(),
           stream())
    C.call("efm_attention_prefill", ctx, ptr(q), ptr(k), ptr(v), ptr(ob), S, S, 1, stream())
    torch.cuda.synchronize()
    err = (o8.float() - ob.float()).abs()
    cos = torch.nn.functional.cosine_similarity(o8.float().flatten(), ob.float().flatten(), dim=0)
    assert float(err.mean()) < 5e-3 and float(cos) > 0.999, (float(err.mean()), float(cos))


@pytest.mark.parametrize("shape", ["4", "8"])
@pytest.mark.parametrize("S,L,causal", [(4096, 4096, 1), (1000, 1300, 1), (77, 77, 0)])
def test_sage_attention_pipelined_matches_register_kernel(gpu, knob, shape, S, L, causal):
    """head_dim 128 runs the global_load_lds ring kernel (both workgroup shapes); it must
    agree with the register-staged kernel (EFM_KNOB_PREFILL_REGISTER) on the same inputs."""
    knob(C.EFM_KNOB_PREFILL_SHAPE, int(shape))
    hq, hkv, hd = 28, 4, 128
    g = torch.Generator(device=gpu).manual_seed(S + L)
    q = torch.randn(S, hq, hd, generator=g, device=gpu).to(torch.bfloat16)
    k = torch.randn(L, hkv, hd, generator=g, device=gpu).to(torch.bfloat16)
    v = torch.randn(L, hkv, hd, generator=g, device=gpu).to(torch.bfloat16)
    ctx = C.make_attention_ctx(hq, hkv, hd, rope=False)
    ws = torch.zeros(C.load().efm_attention_prefill_sage_int8_workspace_bytes(ctx, S, L), dtype=torch.uint8,
                     device=gpu)
    outs = []
    for pipe in ("1", "0"):
        knob(C.EFM_KNOB_PREFILL_REGISTER, 1 if pipe == "0" else 0)
        o = torch.empty(S, hq * hd, dtype=torch.bfloat16, device=gpu)
        C.call("efm_attention_prefill_sage_int8", ctx, ptr(q), ptr(k), ptr(v), ptr(o), S, L, causal, ptr(ws),
               ws.numel(), stream())
        torch.cuda.synchronize()
        outs.append(o)
    assert torch.isfinite(outs[0].float()).all()
    assert_close_bf16(outs[0], outs[1], rtol=2e-2, atol=2e-2, what="sage pipelined vs register kernel")


@pytest.mark.parametrize("hq,hkv,hd,S,L,causal", [
    pytest.param(14, 2, 64, 1, 1, 1, id="hd64_one_row"),
    pytest.param(14, 2, 64, 33, 64, 1, id="hd64_whole_tile"),
    pytest.param(6, 3, 64, 129, 193, 1, id="hd64_three_kv_heads"),
    pytest.param(14, 2, 64, 200, 2111, 1, id="hd64_eight_waves"),
    pytest.param(14, 2, 64, 300, 333, 0, id="hd64_not_causal"),
    pytest.param(12, 2, 128, 97, 97, 1, id="first_split_length"),
    pytest.param(12, 2, 128, 5, 1025, 1, id="few_rows_one_key_past"),
    pytest.param(6, 3, 128, 129, 255, 1, id="three_kv_heads"),
    pytest.param(16, 16, 128, 40, 300, 0, id="sixteen_kv_heads"),
    pytest.param(12, 2, 128, 130, 2049, 1, id="eight_waves"),
    pytest.param(12, 2, 128, 700, 901, 0, id="not_causal"),
])
def test_sage_attention_split_matches_register_kernel(gpu, knob, hq, hkv, hd, S, L, causal):
    """Launches that split their keys over waves (head_dim 64, or few query blocks), q, k and v
    strided out of one row: against the register-staged kernel, which quantises the same. Both
    round p to bf16 before the products; its row sums are over p before that rounding and its
    reference point for p is the true maximum, so a p differs by 2^-8 of itself at most."""
    g = torch.Generator(device=gpu).manual_seed(S + L)
    rows = torch.empty(L, (hq + 2 * hkv) * hd, dtype=torch.bfloat16, device=gpu).normal_(generator=g)
    rows[0, :hq * hd] *= 6   # one 128-row block with a larger scale than the others
    q, k, v = (rows[:, a * hd:] for a in (0, hq, hq + hkv))
    tot = rows.shape[1]
    ctx = C.make_attention_ctx(hq, hkv, hd, rope=False, q_stride_n=tot, q_stride_h=hd, k_stride_n=tot, k_stride_h=hd,
                               kv_stride_n=tot, kv_stride_h=hd)
    ws = torch.zeros(C.load().efm_attention_prefill_sage_int8_workspace_bytes(ctx, S, L), dtype=torch.uint8, device=gpu)
    outs = []
    for register in (0, 1):
        knob(C.EFM_KNOB_PREFILL_REGISTER, register)
        o = torch.full((S + 1, hq * hd), -7.0, dtype=torch.bfloat16, device=gpu)
        C.call("efm_attention_prefill_sage_int8", ctx, ptr(q), ptr(k), ptr(v), ptr(o), S, L, causal, ptr(ws),
               ws.numel(), stream())
        torch.cuda.synchronize()
        assert (o[S] == -7.0).all() and torch.isfinite(o.float()).all()
        outs.append(o[:S])
    assert_close_bf16(outs[0], outs[1], rtol=2e-2, atol=2e-2, what="sage split vs register kernel")


@pytest.mark.parametrize("amp", [1.0, 8.0, 16.0, 64.0])
def test_sage_head_dim_64_scores_are_exact(gpu, amp):
    """The int8 scores of head_dim 64 enter the softmax as exact integers times the scale, at
    any amplitude of q and k: against float64 over the quantised operands. Queries are one
    quantum in one channel, so that the scores of a row stay within a few octaves, and V is
    +-1 per 64-key tile, so that an offset common to a tile shows. Bound: a p is rounded to
    bf16 (2^-9 of it, in the weights and in their sum at most), the output too."""
    g = torch.Generator(device=gpu).manual_seed(int(amp))
    hq, hkv, hd, S, L = 14, 2, 64, 300, 1500
    q = torch.zeros(S, hq, hd, device=gpu)
    ch = torch.randint(0, hd, (S, hq, 1), device=gpu, generator=g)
    q.scatter_(2, ch, amp * 4.0 / 127)
    q[torch.arange(0, S, 128)] = amp * 4.0   # one row of every 128-row block sets its scale
    q = q.bfloat16()
    blk = torch.arange(L, device=gpu) // 128
    k = (torch.empty(L, hkv, hd, device=gpu).normal_(generator=g) * (amp * (1 + 0.13 * blk))[:, None, None]).bfloat16()
    v = (torch.randint(0, 2, ((L + 63) // 64, hkv, hd), device=gpu, generator=g) * 2 - 1)[torch.arange(L, device=gpu) // 64].bfloat16()
    ctx = C.make_attention_ctx(hq, hkv, hd, rope=False)
    q8, k8 = torch.empty(q.shape, dtype=torch.int8, device=gpu), torch.empty(k.shape, dtype=torch.int8, device=gpu)
    sq, sk = torch.empty((S + 127) // 128, hq, device=gpu), torch.empty((L + 127) // 128, hkv, device=gpu)
    km = torch.empty(hkv, hd, device=gpu)
    C.call("efm_sage_quantize", ctx, ptr(q), ptr(k), S, L, ptr(q8), ptr(sq), ptr(k8), ptr(sk), ptr(km), stream())
    ws = torch.zeros(C.load().efm_attention_prefill_sage_int8_workspace_bytes(ctx, S, L), dtype=torch.uint8, device=gpu)
    o = torch.empty(S, hq, hd, dtype=torch.bfloat16, device=gpu)
    C.call("efm_attention_prefill_sage_int8", ctx, ptr(q), ptr(k), ptr(v), ptr(o), S, L, 0, ptr(ws), ws.numel(), stream())
    torch.cuda.synchronize()
    rows = torch.arange(S, device=gpu)
    qd = q8.double() * sq.double()[rows // 128][..., None]
    kd = (k8.double() * sk.double()[blk][..., None]).repeat_interleave(hq // hkv, 1)
    worst = 0.0
    for h in range(hq):
        w = torch.softmax(qd[:, h] @ kd[:, h].T.contiguous() / 8.0, -1)
        ref = w @ v[:, h // (hq // hkv)].double()
        err = (o[:, h].double() - ref).abs() - (2.0 ** -8 + 2.0 ** -9 * ref.abs() + 1e-4)
        worst = max(worst, float(err.max()))
    assert worst <= 0, worst


@pytest.mark.parametrize("hq,hkv", [(12, 2), (28, 4), (16, 2), (8, 8)])
@pytest.mark.parametrize("kv_len,max_kv", [(1, 1), (100, 128), (767, 768), (1025, 2000), (16385, 16513)])
def test_decode_attention_lds_kernel_matches_register_kernel(gpu, knob, hq, hkv, kv_len, max_kv):
    """head_dim 128 with a rotated cache runs the LDS-staged kernel; it must agree with
    the register kernel (EFM_KNOB_DECODE_REGISTER) on the same cache, through both the merged
    entry point and the partials + fused o_proj merge, and store the same rotated newest
    row. Rows past the length hold NaN."""
    _lds_vs_register(gpu, knob, hq, hkv, kv_len, max_kv)


@pytest.mark.parametrize("hq,hkv,kv_len,max_kv", [
    pytest.param(64, 64, 1057, 1100, id="288keys-partial-last-split"),
    pytest.param(64, 64, 1, 1100, id="288keys-one-row"),
    pytest.param(128, 64, 900, 1100, id="288keys-g2"),
    pytest.param(448, 64, 1100, 1100, id="288keys-g7-full"),
    pytest.param(256, 256, 257, 300, id="256keys-8-tiles"),
    pytest.param(28, 4, 16448, 16512, id="c5-58-splits"),
    pytest.param(28, 4, 16390, 16512, id="c5-short-last-split"),
    pytest.param(28, 4, 18432, 18432, id="c5-64-splits-9-tiles"),
])
def test_decode_attention_wide_kernel_matches_register_kernel(gpu, knob, hq, hkv, kv_len, max_kv):
    """Plans past 512 splits of 128 keys run the 8-wave kernel (one workgroup per CU, splits
    of 256-288 keys, every tile in LDS; wave 0 takes a ninth tile): same checks as the 4-wave kernel, including a split whose last tiles lie past the
    length and waves without a tile."""
    _lds_vs_register(gpu, knob, hq, hkv, kv_len, max_kv)


@pytest.mark.parametrize("hq,hkv,kv_len,max_kv,k_off", [
    pytest.param(64, 64, 1057, 1100, 0, id="288keys-partial-last-split"),
    pytest.param(64, 64, 1, 1100, 0, id="288keys-one-row"),
    pytest.param(128, 64, 900, 1100, 3, id="288keys-g2-koff"),
    pytest.param(448, 64, 1100, 1100, 0, id="288keys-g7-full"),
    pytest.param(256, 256, 257, 300, 0, id="256keys-8-tiles"),
    pytest.param(28, 4, 16448, 16512, 0, id="c5-7b-16k"),
    pytest.param(28, 4, 18400, 18432, 5, id="288keys-9-tiles-koff"),
])
def test_decode_attention_wide_kernel_rotate_on_read(gpu, knob, hq, hkv, kv_len, max_kv, k_off):
    """The reference's un-rotated cache (k_already_prerotated 0: every key rotated on read
    at j + k_rope_pos_offset, qwen2_5.cpp:602,624-638 and attention.cu:135-139) on plans
    that take the 8-wave kernel: against the oracle and the register-staged kernel, rows
    past the length NaN, and the cache left as it was (nothing is stored back)."""
    torch.manual_seed(kv_len + hq + 7)
    hd = 128
    q = torch.randn(1, hq, hd, dtype=torch.bfloat16)
    k0 = torch.randn(max_kv, hkv, hd, dtype=torch.bfloat16)
    v0 = torch.randn(max_kv, hkv, hd, dtype=torch.bfloat16)
    ref = O.attention_decode(q, k0, v0, kv_len, O.AttnCtx(hq, hkv, hd, k_rope_pos_offset=k_off))
    k0[kv_len:] = float("nan")
    v0[kv_len:] = float("nan")
    ctx = C.make_attention_ctx(hq, hkv, hd, k_rope_pos_offset=k_off)
    assert ctx.k_already_prerotated == 0
    qg, vg = q.reshape(1, hq * hd).to(gpu), v0.to(gpu)
    d_len = torch.tensor([kv_len], dtype=torch.int32, device=gpu)
    ws = torch.zeros(C.load().efm_attention_decode_workspace_bytes(ctx, max_kv), dtype=torch.uint8, device=gpu)
    outs = []
    for reg in (0, 1):
        knob(C.EFM_KNOB_DECODE_REGISTER, reg)
        k = k0.to(gpu)
        o = torch.empty_like(qg)
        C.call("efm_attention_decode", ctx, ptr(qg), ptr(k), ptr(vg), ptr(o), 0, ptr(d_len), max_kv, ptr(ws),
               ws.numel(), stream())
        torch.cuda.synchronize()
        outs.append(o)
        assert torch.equal(k[:kv_len].cpu(), k0[:kv_len]), "rotate-on-read must not store keys"
    assert torch.isfinite(outs[0].float()).all()
    assert_close_bf16(outs[0].reshape(1, hq, hd), ref, what=f"wide rotate-on-read L={kv_len}")
    assert_close_bf16(outs[0], outs[1], what="wide rotate-on-read vs register kernel")


def _lds_vs_register(gpu, knob, hq, hkv, kv_len, max_kv):
    torch.manual_seed(kv_len + hq)
    hd = 128
    q = torch.randn(1, hq * hd, dtype=torch.bfloat16, device=gpu)
    k0 = torch.randn(max_kv, hkv, hd, dtype=torch.bfloat16, device=gpu)
    v = torch.randn(max_kv, hkv, hd, dtype=torch.bfloat16, device=gpu)
    k0[kv_len:] = float("nan")
    v[kv_len:] = float("nan")
    ctx = C.make_attention_ctx(hq, hkv, hd)
    ctx.k_already_prerotated = C.EFM_K_PREROTATED_EXCEPT_NEWEST
    d_len = torch.tensor([kv_len], dtype=torch.int32, device=gpu)
    ws = torch.zeros(C.load().efm_attention_decode_workspace_bytes(ctx, max_kv), dtype=torch.uint8, device=gpu)
    outs, caches = [], []
    for lds in ("1", "0"):
        knob(C.EFM_KNOB_DECODE_REGISTER, 1 if lds == "0" else 0)
        k = k0.clone()
        o = torch.empty_like(q)
        C.call("efm_attention_decode", ctx, ptr(q), ptr(k), ptr(v), ptr(o), 0, ptr(d_len), max_kv, ptr(ws),
               ws.numel(), stream())
        torch.cuda.synchronize()
        outs.append(o)
        caches.append(k)
    assert torch.isfinite(outs[0].float()).all()
    assert_close_bf16(outs[0], outs[1], what="lds vs register decode kernel")
    assert torch.equal(caches[0][: kv_len - 1], k0[: kv_len - 1])
    # the newest row: both rotate with the same cos/sin table and rounding
    assert torch.equal(caches[0][kv_len - 1], caches[1][kv_len - 1])


@pytest.mark.parametrize("lds", ["0", "1"])
@pytest.mark.parametrize("kv_len,max_kv", [(161, 40000), (321, 70000), (1025, 40000), (129, 40000)])
def test_decode_newest_row_owned_by_one_split(gpu, knob, lds, kv_len, max_kv):
    """With keys-per-split not a multiple of 128 (large max_kv_len) a split's last round has
    idle tiles that lie in the next split; they must not touch the newest row, which only
    its owning split rotates and stores (regression: the idle tile stored zeros)."""
    knob(C.EFM_KNOB_DECODE_REGISTER, 1 if lds == "0" else 0)
    torch.manual_seed(0)
    hq, hkv, hd = 12, 2, 128
    q = torch.randn(1, hq * hd, dtype=torch.bfloat16, device=gpu)
    k = torch.randn(max_kv, hkv, hd, dtype=torch.bfloat16, device=gpu)
    v = torch.randn(max_kv, hkv, hd, dtype=torch.bfloat16, device=gpu)
    raw = k[kv_len - 1].clone().cpu()
    ctx = C.make_attention_ctx(hq, hkv, hd)
    ctx.k_already_prerotated = C.EFM_K_PREROTATED_EXCEPT_NEWEST
    d_len = torch.tensor([kv_len], dtype=torch.int32, device=gpu)
    ws = torch.zeros(C.load().efm_attention_decode_workspace_bytes(ctx, max_kv), dtype=torch.uint8, device=gpu)
    C.call("efm_decode_attention_partials", ctx, ptr(q), ptr(k), ptr(v), ptr(d_len), max_kv, ptr(ws), ws.numel(),
           stream())
    torch.cuda.synchronize()
    want = O.rope_llama(raw.unsqueeze(0), torch.tensor([kv_len - 1]), 1.0e6).to(torch.bfloat16)[0]
    assert_close_bf16(k[kv_len - 1], want, rtol=1e-2, atol=1e-2, what="newest row")
