"""Fused decode-step kernels (include/qwen2_decode.h) against the torch
restatement of src/qwen_int4/model.py they replace, and the fused decode step
of the whole decoder against the module-level decode path.

Tolerances: the residual sum and the rotated cache rows repeat the
reference's bf16 roundings exactly (bit-exact); RMSNorm differs from torch
only in the order of the fp32 sum of squares (>= 99% of outputs bit-identical,
the rest one bf16 ulp); attention differs in fp32 summation order (normwise
max error <= 1e-2 of the largest output, cosine >= 0.99999); model logits
cosine >= 0.9999 (the model-level gate).
"""

from __future__ import annotations

import ctypes
from types import SimpleNamespace

import pytest
import torch

from qwen_int4_hip import _lib
from qwen_int4_hip.model import QwenInt4ForCausalLM, RMSNorm, RotaryEmbedding, attend, rotate_half

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a ROCm GPU")]


def _p(t):
    return None if t is None else ctypes.c_void_p(t.data_ptr())


def _stream():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


@pytest.mark.parametrize("rows,hidden", [(1, 1536), (3, 1536), (2, 896), (1, 8192), (4, 104), (2, 2056)])
@pytest.mark.parametrize("delta_dtype", [None, torch.bfloat16, torch.float32])
def test_add_rmsnorm_matches_torch(rows, hidden, delta_dtype):
    lib = _lib.load()
    g = _gen(rows * 7 + hidden)
    x = (torch.randn((rows, hidden), generator=g, device="cuda") * 3).to(torch.bfloat16)
    delta = None if delta_dtype is None else (torch.randn((rows, hidden), generator=g, device="cuda") * 2).to(delta_dtype)
    norm = RMSNorm(hidden, 1e-6).cuda()
    with torch.no_grad():
        norm.weight.copy_((torch.rand(hidden, generator=g, device="cuda") + 0.5).to(torch.bfloat16))
    want_sum = x if delta is None else x + delta.to(torch.bfloat16)
    want = norm(want_sum)
    out_sum = torch.empty_like(x)
    out = torch.empty_like(x)
    code = {None: 0, torch.bfloat16: _lib.DTYPE_BF16, torch.float32: _lib.DTYPE_F32}[delta_dtype]
    _lib.check(lib.qwen2_add_rmsnorm(_p(x), _p(delta), code, _p(norm.weight), ctypes.c_float(1e-6), _p(out_sum),
                                     _p(out), rows, hidden, _stream()))
    torch.cuda.synchronize()
    assert torch.equal(out_sum, want_sum)
    same = (out == want).float().mean().item()
    rel = ((out.float() - want.float()).abs() / want.float().abs().clamp_min(1e-30)).max().item()
    assert same >= 0.99 and rel <= 2.0 ** -7, (same, rel)
    # in place on the residual stream (out_sum aliases x)
    x2 = x.clone()
    _lib.check(lib.qwen2_add_rmsnorm(_p(x2), _p(delta), code, _p(norm.weight), ctypes.c_float(1e-6), _p(x2),
                                     _p(out), rows, hidden, _stream()))
    torch.cuda.synchronize()
    assert torch.equal(x2, want_sum)


@pytest.mark.parametrize("delta_dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("form,n,k", [("linear", 2048, 1536), ("linear", 200, 640), ("planes", 8960, 1536),
                                      ("planes", 72, 192), ("planes", 256, 256), ("planes", 2064, 640),
                                      ("planes", 17920, 1536), ("planes", 512, 2048)])
def test_linear_rmsnorm_matches_norm_then_linear(delta_dtype, form, n, k):
    """w4g64_linear_rmsnorm (one row) = qwen2_add_rmsnorm followed by the
    plain linear (or the gate|up planes entry): the residual sum bit-exact
    (torch's bf16 add), the activation to the norm's own bar (the fp32 sum of
    squares runs in another order), so the outputs agree to the bf16 rounding
    that can flip (normwise 1e-2; most outputs identical)."""
    lib = _lib.load()
    g = _gen(n + k + (1 if delta_dtype == torch.float32 else 0))
    x = (torch.randn((1, k), generator=g, device="cuda") * 3).to(torch.bfloat16)
    delta = (torch.randn((1, k), generator=g, device="cuda") * 2).to(delta_dtype)
    norm = RMSNorm(k, 1e-6).cuda()
    with torch.no_grad():
        norm.weight.copy_((torch.rand(k, generator=g, device="cuda") + 0.5).to(torch.bfloat16))
    qw, sc, z = _weights(n, k, 23, asymmetric=True)
    bias = (torch.randn(n, generator=g, device="cuda") * 0.3).to(torch.bfloat16) if form == "linear" else None
    dcode = _lib.DTYPE_BF16 if delta_dtype == torch.bfloat16 else _lib.DTYPE_F32
    planes = form == "planes"
    y = (torch.empty((3, 1, n // 2), dtype=torch.bfloat16, device="cuda") if planes
         else torch.empty((1, n), dtype=torch.bfloat16, device="cuda"))
    out_sum = torch.empty_like(x)
    ws = torch.zeros(1 << 20, dtype=torch.uint8, device="cuda")
    _lib.check(lib.w4g64_linear_rmsnorm(_p(x), _p(delta), dcode, _p(norm.weight), ctypes.c_float(1e-6), _p(out_sum),
                                        _p(qw), _p(sc), _p(z), _p(bias), _lib.DTYPE_BF16 if bias is not None else 0,
                                        _p(y), 1 if planes else 0, 1, n, k, _p(ws), ws.numel(), _stream()))
    # the separate kernels
    ref_sum, normed = torch.empty_like(x), torch.empty_like(x)
    _lib.check(lib.qwen2_add_rmsnorm(_p(x), _p(delta), dcode, _p(norm.weight), ctypes.c_float(1e-6), _p(ref_sum),
                                     _p(normed), 1, k, _stream()))
    want = torch.empty_like(y)
    if planes:
        _lib.check(lib.w4g64_linear_gate_up_planes(_p(normed), _p(qw), _p(sc), _p(z), None, 0, _p(want), 1, n, k,
                                                   _p(ws), ws.numel(), _stream()))
    else:
        _lib.check(lib.w4g64_linear(_p(normed), _lib.DTYPE_BF16, _p(qw), _p(sc), _p(z), _p(bias), _lib.DTYPE_BF16,
                                    _p(want), 1, n, k, _p(ws), ws.numel(), _stream()))
    torch.cuda.synchronize()
    assert torch.equal(out_sum, x + delta.to(torch.bfloat16)) and torch.equal(out_sum, ref_sum)
    got = y.float().sum(0) if planes else y.float()
    ref = want.float().sum(0) if planes else want.float()
    assert bool(torch.isfinite(got).all())
    assert _normwise(got, ref) <= 1e-2
    assert (got == ref).float().mean().item() >= 0.9


def _torch_attention(qkv, cos, sin, k_cache, v_cache, pos, heads, kv_heads):
    """The module path of one cached token: rotary in bf16, cache write,
    fp32 attention over positions 0..pos (qwen_int4_hip.model, which restates
    model.py:61-122)."""
    batch = qkv.shape[0]
    d = 128
    q = qkv[:, : heads * d].view(batch, heads, 1, d)
    k = qkv[:, heads * d:(heads + kv_heads) * d].view(batch, kv_heads, 1, d)
    v = qkv[:, (heads + kv_heads) * d:].view(batch, kv_heads, 1, d)
    c, s = cos.view(batch, 1, 1, d), sin.view(batch, 1, 1, d)
    q = q * c + rotate_half(q) * s
    k = k * c + rotate_half(k) * s
    k_cache = k_cache.clone()
    v_cache = v_cache.clone()
    k_cache[:, :, pos] = k[:, :, 0]
    v_cache[:, :, pos] = v[:, :, 0]
    group = heads // kv_heads
    allowed = (torch.arange(k_cache.shape[2], device="cuda") <= pos).view(1, 1, 1, -1)
    out = attend(q.reshape(batch, kv_heads, group, d), k_cache, v_cache, allowed, d ** -0.5)
    return out.reshape(batch, heads * d), k_cache, v_cache


@pytest.mark.parametrize("batch,heads,kv_heads,max_length,positions", [
    (1, 12, 2, 640, (0, 1, 63, 64, 65, 200, 511, 639)),
    (3, 12, 2, 130, (0, 64, 127, 129)),
    (2, 8, 1, 64, (0, 31, 63)),
    (1, 4, 4, 700, (5, 699)),
    (1, 12, 2, 2048, (1000, 2047)),  # 32 chunks merged
    (1, 12, 2, 2200, (0, 64, 2199)),  # a partial last chunk; early positions leave most chunks empty
])
def test_decode_attention_matches_torch(batch, heads, kv_heads, max_length, positions):
    lib = _lib.load()
    g = _gen(batch * 1000 + heads * 10 + kv_heads)
    d = 128
    rot = RotaryEmbedding(d, 1_000_000.0).cuda()
    k_cache = (torch.randn((batch, kv_heads, max_length, d), generator=g, device="cuda")).to(torch.bfloat16)
    v_cache = (torch.randn((batch, kv_heads, max_length, d), generator=g, device="cuda")).to(torch.bfloat16)
    ws = torch.zeros(lib.qwen2_decode_attention_workspace_bytes(batch, kv_heads, max_length), dtype=torch.uint8,
                     device="cuda")
    for pos in positions:
        qkv = (torch.randn((batch, (heads + 2 * kv_heads) * d), generator=g, device="cuda") * 2).to(torch.bfloat16)
        position = torch.tensor([pos], dtype=torch.long, device="cuda")
        cos, sin = rot(position.view(1, 1).expand(batch, 1), torch.bfloat16)
        cos, sin = cos.reshape(batch, d).contiguous(), sin.reshape(batch, d).contiguous()
        want, want_k, want_v = _torch_attention(qkv, cos, sin, k_cache, v_cache, pos, heads, kv_heads)
        out = torch.empty((batch, heads * d), dtype=torch.bfloat16, device="cuda")
        for _ in range(2):  # a second call on the same workspace: counters were left at zero
            _lib.check(lib.qwen2_decode_attention(
                _p(qkv), _p(cos), _p(sin), _p(k_cache), _p(v_cache), _p(position), _p(out), batch, heads, kv_heads,
                d, max_length, ctypes.c_float(d ** -0.5), _p(ws), ws.numel(), _stream()))
            torch.cuda.synchronize()
            assert torch.equal(k_cache, want_k) and torch.equal(v_cache, want_v)
            err = (out.float() - want.float()).abs().max().item()
            cos_sim = torch.nn.functional.cosine_similarity(out.double().flatten(), want.double().flatten(), dim=0)
            assert err <= 1e-2 * want.float().abs().max().item(), (pos, err)
            assert cos_sim.item() >= 0.99999, (pos, cos_sim.item())


@pytest.mark.parametrize("batch,heads,kv_heads,max_length,positions", [
    (2, 12, 2, 64, (0, 1, 30, 31, 32, 63)),         # one split: no merge launch
    (3, 8, 1, 129, (0, 15, 16, 127, 128)),          # two splits, the cache ends one row into a block
    (2, 3, 3, 1000, (3, 126, 511, 512, 999)),       # one query head per key/value head, a ragged last block
    (33, 14, 2, 300, (0, 200, 299)),                # seven per head; fewer splits than the cache has room for
    (1, 16, 2, 17408, (31, 4095, 17407)),           # the longest cache, the most splits
    (2, 12, 2, 640, (-5, 640, 10_000)),             # clamped to the cache
    (24, 16, 2, 129, (0, 127, 128)),                # past 96 chunks: two splits of the split kernel
    (3, 3, 3, 1000, (3, 126, 511, 512, 999)),
    (6, 12, 2, 640, (-5, 640, 10_000)),
])
def test_decode_attention_split_over_workgroups(batch, heads, kv_heads, max_length, positions):
    """qwen2_decode_attention past one sequence or 1024 positions (the split
    kernel and its merge) against the same in fp64 from the rounded rotary
    step: the fp32 result differs from it by a few fp32 ulp of the sums, so
    the bf16 output by at most one rounding (2^-8 of the value) plus 2^-16 of
    the largest one.  Rows past the position are NaN and must not be read into
    the result; the workspace starts as NaN."""
    lib = _lib.load()
    g = _gen(batch * 100 + heads + max_length)
    d = 128
    rot = RotaryEmbedding(d, 1_000_000.0).cuda()
    base = torch.randn((2, batch, kv_heads, max_length, d), generator=g, device="cuda").to(torch.bfloat16)
    wbytes = lib.qwen2_decode_attention_workspace_bytes(batch, kv_heads, max_length)
    counters = (batch * kv_heads * 4 + 255) // 256 * 256
    for at in positions:
        pos = min(max(at, 0), max_length - 1)
        k_cache, v_cache = base.clone().unbind(0)
        k_cache[:, :, pos:], v_cache[:, :, pos:] = float("nan"), float("nan")
        qkv = (torch.randn((batch, (heads + 2 * kv_heads) * d), generator=g, device="cuda") * 2).to(torch.bfloat16)
        cos, sin = rot(torch.tensor([[pos]], device="cuda").expand(batch, 1), torch.bfloat16)
        cos, sin = cos.reshape(batch, d).contiguous(), sin.reshape(batch, d).contiguous()
        ws = torch.full((wbytes,), 0xFF, dtype=torch.uint8, device="cuda")
        ws[:counters] = 0
        out = torch.empty((batch, heads * d), dtype=torch.bfloat16, device="cuda")
        position = torch.tensor([at], dtype=torch.long, device="cuda")
        _lib.check(lib.qwen2_decode_attention(
            _p(qkv), _p(cos), _p(sin), _p(k_cache), _p(v_cache), _p(position), _p(out), batch, heads, kv_heads,
            d, max_length, ctypes.c_float(d ** -0.5), _p(ws), ws.numel(), _stream()))
        torch.cuda.synchronize()
        q, k, v = (t.view(batch, -1, 1, d) for t in qkv.split([heads * d, kv_heads * d, kv_heads * d], dim=1))
        c, s = cos.view(batch, 1, 1, d), sin.view(batch, 1, 1, d)
        q, k = q * c + rotate_half(q) * s, k * c + rotate_half(k) * s
        want_k, want_v = base.clone().unbind(0)
        want_k[:, :, pos], want_v[:, :, pos] = k[:, :, 0], v[:, :, 0]
        assert torch.equal(k_cache[:, :, : pos + 1], want_k[:, :, : pos + 1])
        assert torch.equal(v_cache[:, :, : pos + 1], want_v[:, :, : pos + 1])
        assert bool(torch.isnan(k_cache[:, :, pos + 1:]).all()) and bool(torch.isnan(v_cache[:, :, pos + 1:]).all())
        keys, values = want_k[:, :, : pos + 1].double(), want_v[:, :, : pos + 1].double()
        scores = (q.view(batch, kv_heads, -1, 1, d).double() * keys.unsqueeze(2)).sum(-1) * d ** -0.5
        probs = torch.softmax(scores, dim=-1)
        want = (probs @ values).reshape(batch, heads * d)
        err = (out.double() - want).abs()
        assert bool((err <= want.abs() * 2.0 ** -8 + want.abs().max() * 2.0 ** -16).all()), (at, err.max().item())


@pytest.mark.parametrize("heads,kv_heads,max_length,positions,n,with_bias", [
    (12, 2, 640, (0, 1, 63, 64, 65, 511, 639), 1536, False),
    (12, 2, 1024, (0, 700, 1023), 1536, True),  # 16 chunks: the most the merge form takes
    (8, 1, 100, (3, 99), 200, False),            # 8 query heads per key/value head, a partial last chunk
    (2, 2, 64, (0, 63), 96, False),              # one query head per key/value head, one chunk
    (4, 2, 200, (130,), 1536, True),
])
def test_attention_merged_in_o_proj_equals_attention_then_o_proj(heads, kv_heads, max_length, positions, n,
                                                                 with_bias):
    """qwen2_decode_attention_partials + w4g64_linear_attention_merge against
    qwen2_decode_attention + w4g64_linear on the same inputs: the same cache
    writes and, bit for bit, the same o_proj output (the merge in the GEMV's
    staging repeats the attention's own merge operation for operation).  The
    unmerged path's workspace starts as NaN, so chunks past the position must
    be written (as empty partials), not assumed."""
    lib = _lib.load()
    g = _gen(heads * 100 + kv_heads + max_length)
    d = 128
    k = heads * d
    rot = RotaryEmbedding(d, 1_000_000.0).cuda()
    k_cache = torch.randn((1, kv_heads, max_length, d), generator=g, device="cuda").to(torch.bfloat16)
    v_cache = torch.randn((1, kv_heads, max_length, d), generator=g, device="cuda").to(torch.bfloat16)
    k_part, v_part = k_cache.clone(), v_cache.clone()
    qw, sc, z = _weights(n, k, heads + n, asymmetric=True)
    bias = (torch.randn(n, generator=g, device="cuda") * 0.1).to(torch.bfloat16) if with_bias else None
    bias_code = _lib.DTYPE_BF16 if with_bias else _lib.DTYPE_NONE
    wbytes = lib.qwen2_decode_attention_workspace_bytes(1, kv_heads, max_length)
    ws = torch.zeros(wbytes, dtype=torch.uint8, device="cuda")
    ws_part = torch.full((wbytes,), 0xFF, dtype=torch.uint8, device="cuda")  # NaN partials
    lws = torch.zeros(max(lib.w4g64_linear_workspace_bytes(1, n, k, _lib.DTYPE_BF16), 1), dtype=torch.uint8,
                      device="cuda")
    attended = torch.empty((1, k), dtype=torch.bfloat16, device="cuda")
    want = torch.empty((1, n), dtype=torch.bfloat16, device="cuda")
    got = torch.empty((1, n), dtype=torch.bfloat16, device="cuda")
    for pos in positions:
        qkv = (torch.randn((1, (heads + 2 * kv_heads) * d), generator=g, device="cuda") * 2).to(torch.bfloat16)
        position = torch.tensor([pos], dtype=torch.long, device="cuda")
        cos, sin = rot(position.view(1, 1), torch.bfloat16)
        cos, sin = cos.reshape(1, d).contiguous(), sin.reshape(1, d).contiguous()
        _lib.check(lib.qwen2_decode_attention(
            _p(qkv), _p(cos), _p(sin), _p(k_cache), _p(v_cache), _p(position), _p(attended), 1, heads, kv_heads, d,
            max_length, ctypes.c_float(d ** -0.5), _p(ws), ws.numel(), _stream()))
        _lib.check(lib.w4g64_linear(_p(attended), _lib.DTYPE_BF16, _p(qw), _p(sc), _p(z), _p(bias), bias_code,
                                    _p(want), 1, n, k, _p(lws), lws.numel(), _stream()))
        _lib.check(lib.qwen2_decode_attention_partials(
            _p(qkv), _p(cos), _p(sin), _p(k_part), _p(v_part), _p(position), 1, heads, kv_heads, d, max_length,
            ctypes.c_float(d ** -0.5), _p(ws_part), ws_part.numel(), _stream()))
        _lib.check(lib.w4g64_linear_attention_merge(_p(ws_part), ws_part.numel(), max_length, heads, kv_heads,
                                                    _p(qw), _p(sc), _p(z), _p(bias), bias_code, _p(got), 1, n,
                                                    _stream()))
        torch.cuda.synchronize()
        assert torch.equal(k_part, k_cache) and torch.equal(v_part, v_cache), pos
        assert torch.isfinite(want.float()).all(), pos
        assert torch.equal(got, want), (pos, (got.float() - want.float()).abs().max().item())


def test_fused_decode_step_merged_in_o_proj_is_bit_identical():
    """The batch-1 decode step with the attention merged in the o_proj GEMV
    against the same step with the attention's own merge: identical logits,
    greedy tokens and caches over 70 steps (across a 64-position chunk
    boundary)."""
    from qwen_int4_hip.decode import FusedDecodeStep
    from qwen_int4_hip.generation import StaticGreedyDecoder

    model = _build(SMALL128, 21)
    prompt = torch.randint(0, SMALL128.vocab_size, (1, 13), generator=torch.Generator().manual_seed(7)).cuda()
    merged = StaticGreedyDecoder(model, 1, 96, use_graph=False, fused=True)
    plain = StaticGreedyDecoder(model, 1, 96, use_graph=False, fused=True)
    plain.fused = FusedDecodeStep(model, 1, 96, merge_attention_in_o_proj=False)
    assert merged.fused.merge_in_o_proj and not plain.fused.merge_in_o_proj
    merged.prefill(prompt)
    plain.prefill(prompt)
    for step in range(70):
        token = plain.token.clone()
        want = plain.step(token).clone()
        got = merged.step(token).clone()
        assert torch.equal(got, want), step
        assert torch.equal(merged.token, plain.token), step
    for (k0, v0), (k1, v1) in zip(plain.caches, merged.caches):
        assert torch.equal(k0, k1) and torch.equal(v0, v1)


@pytest.mark.parametrize("batch,hidden,vocab", [(1, 1536, 151936), (3, 256, 512)])
def test_decode_prologue_matches_embedding_and_rotary(batch, hidden, vocab):
    """qwen2_decode_prologue = the embedding lookup and RotaryEmbedding.forward
    of one position (model.py:22-31, :182, :190), bit for bit, at positions up
    to a 17408-position cache, and the first layer's RMSNorm to its bar; an id
    outside [0, vocab) gives a NaN row."""
    lib = _lib.load()
    g = _gen(batch * 31 + hidden)
    embed = (torch.randn((vocab, hidden), generator=g, device="cuda") * 0.02).to(torch.bfloat16)
    rot = RotaryEmbedding(128, 1_000_000.0).cuda()
    x = torch.empty((batch, hidden), dtype=torch.bfloat16, device="cuda")
    normed = torch.empty_like(x)
    norm = RMSNorm(hidden, 1e-6).cuda()
    with torch.no_grad():
        norm.weight.copy_((torch.rand(hidden, generator=g, device="cuda") + 0.5).to(torch.bfloat16))
    cos = torch.empty((batch, 128), dtype=torch.bfloat16, device="cuda")
    sin = torch.empty_like(cos)
    for pos in (0, 1, 63, 511, 640, 4095, 17407):
        ids = torch.randint(0, vocab, (batch,), generator=g, device="cuda", dtype=torch.int64)
        position = torch.tensor([pos], dtype=torch.int64, device="cuda")
        _lib.check(lib.qwen2_decode_prologue(_p(ids), _p(embed), _p(position), _p(rot.inv_freq), _p(x), _p(cos),
                                             _p(sin), _p(norm.weight), ctypes.c_float(1e-6), _p(normed), batch,
                                             hidden, vocab, 128, _stream()))
        want_cos, want_sin = rot(position.view(1, 1).expand(batch, 1), torch.bfloat16)
        want_x = embed[ids]
        want_n = norm(want_x)
        torch.cuda.synchronize()
        assert torch.equal(x, want_x), pos
        assert torch.equal(cos, want_cos.reshape(batch, 128)), pos
        assert torch.equal(sin, want_sin.reshape(batch, 128)), pos
        # the norm to RMSNorm's bar (the fp32 sum of squares runs in another order)
        rel = ((normed.float() - want_n.float()).abs() / want_n.float().abs().clamp_min(1e-30)).max().item()
        assert (normed == want_n).float().mean().item() >= 0.99 and rel <= 2.0 ** -7, (pos, rel)
    # without the norm: x, cos and sin only
    _lib.check(lib.qwen2_decode_prologue(_p(ids), _p(embed), _p(position), _p(rot.inv_freq), _p(x), _p(cos), _p(sin),
                                         None, ctypes.c_float(1e-6), None, batch, hidden, vocab, 128, _stream()))
    torch.cuda.synchronize()
    assert torch.equal(x, embed[ids])
    bad = torch.full((batch,), vocab, dtype=torch.int64, device="cuda")
    _lib.check(lib.qwen2_decode_prologue(_p(bad), _p(embed), _p(position), _p(rot.inv_freq), _p(x), _p(cos), _p(sin),
                                         None, ctypes.c_float(1e-6), None, batch, hidden, vocab, 128, _stream()))
    torch.cuda.synchronize()
    assert bool(torch.isnan(x.float()).all())


@pytest.mark.parametrize("batch,heads,kv_heads,length,max_length", [
    (1, 12, 2, 512, 640),  # the prefill of the model's workload
    (2, 8, 1, 100, 128),   # a partial last block; group 8
    (3, 4, 4, 65, 70),     # one query row past a block boundary; no grouping
    (1, 12, 2, 1, 8),      # a single position
])
def test_prefill_attention_matches_torch(batch, heads, kv_heads, length, max_length):
    """Rotary, cache update and causal attention over a prompt against the
    module path's torch restatement (rotary in bf16, fp32 attention)."""
    lib = _lib.load()
    g = _gen(batch * 100 + length)
    d = 128
    rows = batch * length
    qkv = (torch.randn((rows, (heads + 2 * kv_heads) * d), generator=g, device="cuda") * 2).to(torch.bfloat16)
    k_cache = torch.randn((batch, kv_heads, max_length, d), generator=g, device="cuda").to(torch.bfloat16)
    v_cache = torch.randn((batch, kv_heads, max_length, d), generator=g, device="cuda").to(torch.bfloat16)
    positions = torch.arange(length, device="cuda").view(1, -1).expand(batch, length)
    cos, sin = RotaryEmbedding(d, 1_000_000.0).cuda()(positions, torch.bfloat16)
    q = qkv[:, : heads * d].view(batch, length, heads, d).transpose(1, 2)
    k = qkv[:, heads * d:(heads + kv_heads) * d].view(batch, length, kv_heads, d).transpose(1, 2)
    v = qkv[:, (heads + kv_heads) * d:].view(batch, length, kv_heads, d).transpose(1, 2)
    c, s = cos.unsqueeze(1), sin.unsqueeze(1)
    q = q * c + rotate_half(q) * s
    k = k * c + rotate_half(k) * s
    want_k, want_v = k_cache.clone(), v_cache.clone()
    want_k[:, :, :length] = k
    want_v[:, :, :length] = v
    allowed = torch.ones((length, length), dtype=torch.bool, device="cuda").tril().view(1, 1, length, length)
    group = heads // kv_heads
    want = attend(q, k.repeat_interleave(group, dim=1), v.repeat_interleave(group, dim=1), allowed, d ** -0.5)
    want = want.transpose(1, 2).reshape(rows, heads * d)
    out = torch.empty((rows, heads * d), dtype=torch.bfloat16, device="cuda")
    ws = torch.empty(lib.qwen2_prefill_attention_workspace_bytes(batch, heads, length), dtype=torch.uint8,
                     device="cuda")
    _lib.check(lib.qwen2_prefill_attention(
        _p(qkv), _p(cos.reshape(rows, d).contiguous()), _p(sin.reshape(rows, d).contiguous()), _p(k_cache),
        _p(v_cache), _p(out), batch, length, heads, kv_heads, d, max_length, ctypes.c_float(d ** -0.5), _p(ws),
        ws.numel(), _stream()))
    torch.cuda.synchronize()
    assert torch.equal(k_cache, want_k) and torch.equal(v_cache, want_v)  # rows past the prompt untouched
    err = (out.float() - want.float()).abs().max().item()
    cos_sim = torch.nn.functional.cosine_similarity(out.double().flatten(), want.double().flatten(), dim=0)
    assert err <= 1e-2 * want.float().abs().max().item(), err
    assert cos_sim.item() >= 0.99999, cos_sim.item()


@pytest.mark.parametrize("batch,heads,kv_heads,length,max_length,scale,shift", [
    (1, 12, 2, 31, 31, 128 ** -0.5, 0),    # the cache ends with the prompt, a partial block
    (2, 3, 3, 32, 40, 128 ** -0.5, 1),     # exactly one block; factors and output only 2-byte aligned
    (1, 8, 1, 33, 64, -0.05, 0),           # one row past a block; a negative scale
    (1, 2, 2, 160, 161, 128 ** -0.5, 0),   # five blocks: one wave takes two
    (1, 14, 2, 1021, 1024, 1.0, 3),        # sharp softmax: rows rescaled late, many blocks per wave
])
def test_prefill_attention_block_edges(batch, heads, kv_heads, length, max_length, scale, shift):
    """qwen2_prefill_attention at the edges of its 32-row tiles and 32-key
    blocks against the same in fp64 from the rounded rotary step: fp32 scores
    of magnitude up to s carry an error of about 128 2^-24 s into the
    exponent, so an output differs by at most its bf16 rounding (2^-8 of the
    value) plus (2^-16 + 2^-16 s) of the largest one."""
    lib = _lib.load()
    g = _gen(batch * 100 + length)
    d, rows = 128, batch * length
    qkv = torch.randn((rows, (heads + 2 * kv_heads) * d), generator=g, device="cuda").to(torch.bfloat16)
    caches = torch.randn((2, batch, kv_heads, max_length, d), generator=g, device="cuda").to(torch.bfloat16)
    k_cache, v_cache = caches.clone().unbind(0)
    positions = torch.arange(length, device="cuda").repeat(batch)

    def shifted(cols):  # a tensor that starts `shift` elements into its storage
        return torch.empty(rows * cols + shift, dtype=torch.bfloat16, device="cuda")[shift:].view(rows, cols)

    cos, sin, out = shifted(d), shifted(d), shifted(heads * d)
    for to, value in zip((cos, sin), RotaryEmbedding(d, 1_000_000.0).cuda()(positions, torch.bfloat16)):
        to.copy_(value)
    ws = torch.empty(lib.qwen2_prefill_attention_workspace_bytes(batch, heads, length), dtype=torch.uint8,
                     device="cuda")
    _lib.check(lib.qwen2_prefill_attention(
        _p(qkv), _p(cos), _p(sin), _p(k_cache), _p(v_cache), _p(out), batch, length, heads, kv_heads, d, max_length,
        ctypes.c_float(scale), _p(ws), ws.numel(), _stream()))
    torch.cuda.synchronize()
    q, k, v = (t.view(batch, length, -1, d).transpose(1, 2)
               for t in qkv.split([heads * d, kv_heads * d, kv_heads * d], dim=1))
    c, s = cos.view(batch, 1, length, d), sin.view(batch, 1, length, d)
    q, k = q * c + rotate_half(q) * s, k * c + rotate_half(k) * s
    want_k, want_v = caches.clone().unbind(0)
    want_k[:, :, :length], want_v[:, :, :length] = k, v
    assert torch.equal(k_cache, want_k) and torch.equal(v_cache, want_v)
    group = heads // kv_heads
    k, v = (t.double().repeat_interleave(group, dim=1) for t in (k, v))
    scores = torch.matmul(q.double(), k.transpose(-1, -2).contiguous()) * scale
    causal = torch.ones((length, length), dtype=torch.bool, device="cuda").tril()
    probs = torch.softmax(scores.masked_fill(~causal, float("-inf")), dim=-1)
    want = torch.matmul(probs, v).transpose(1, 2).reshape(rows, heads * d)
    err = (out.double() - want).abs()
    bound = want.abs() * 2.0 ** -8 + want.abs().max() * 2.0 ** -16 * (1 + scores.abs().max())
    assert bool((err <= bound).all()), (err - bound).max().item()


@pytest.mark.parametrize("length,low", [(70, ((0, 32),)), (200, ((0, 32), (96, 128), (160, 165)))])
def test_prefill_attention_keys_of_infinite_score(length, low):
    """Keys whose scores overflow to -inf in fp32 take no part, also where they
    fill a wave's first 32-key block (bound as in the block edges' test)."""
    lib = _lib.load()
    g = _gen(length)
    d, heads, kv_heads = 128, 4, 2
    q, k, v = (torch.randn((length, h, d), generator=g, device="cuda").to(torch.bfloat16)
               for h in (heads, kv_heads, kv_heads))
    q[:, :, 0] = 100.0
    dead = torch.zeros(length, dtype=torch.bool, device="cuda")
    for begin, end in low:
        dead[begin:end] = True
    k[dead, :, 0] = -3e38
    qkv = torch.cat((q, k, v), dim=1).reshape(length, -1).contiguous()
    cos, sin = torch.ones((length, d), dtype=torch.bfloat16, device="cuda"), torch.zeros((length, d), dtype=torch.bfloat16, device="cuda")
    caches = torch.zeros((2, 1, kv_heads, length, d), dtype=torch.bfloat16, device="cuda")
    out = torch.empty((length, heads * d), dtype=torch.bfloat16, device="cuda")
    ws = torch.empty(lib.qwen2_prefill_attention_workspace_bytes(1, heads, length), dtype=torch.uint8, device="cuda")
    _lib.check(lib.qwen2_prefill_attention(
        _p(qkv), _p(cos), _p(sin), _p(caches[0]), _p(caches[1]), _p(out), 1, length, heads, kv_heads, d, length,
        ctypes.c_float(d ** -0.5), _p(ws), ws.numel(), _stream()))
    kk, vv = (t.double().repeat_interleave(heads // kv_heads, dim=1).transpose(0, 1).contiguous() for t in (k, v))
    scores = torch.matmul(q.double().transpose(0, 1).contiguous(), kk.transpose(-1, -2).contiguous()) * d ** -0.5
    causal = torch.ones((length, length), dtype=torch.bool, device="cuda").tril()
    allowed = causal & ~dead
    live = allowed.any(-1)  # rows with a finite score
    probs = torch.softmax(scores.masked_fill(~allowed, float("-inf"))[:, live], dim=-1)
    want = torch.matmul(probs, vv).transpose(0, 1).reshape(-1, heads * d)
    err = (out[live].double() - want).abs()
    bound = want.abs() * 2.0 ** -8 + want.abs().max() * 2.0 ** -16 * (1 + scores[:, live][:, :, ~dead].abs().max())
    assert bool((err <= bound).all()), (err - bound).max().item()


@pytest.mark.parametrize("max_length,pos,dead", [(64, 60, 32), (64, 63, 63), (1100, 1000, 900), (4096, 4095, 4000)])
def test_decode_attention_keys_of_infinite_score(max_length, pos, dead):
    """The split kernel where whole waves and splits meet nothing but scores of -inf."""
    lib = _lib.load()
    g = _gen(max_length + pos)
    d, heads, kv_heads, batch = 128, 4, 2, 2
    k_cache, v_cache = (torch.randn((batch, kv_heads, max_length, d), generator=g, device="cuda").to(torch.bfloat16)
                        for _ in range(2))
    k_cache[:, :, :dead, 0] = float("-inf")
    qkv = torch.randn((batch, heads + 2 * kv_heads, d), generator=g, device="cuda").to(torch.bfloat16)
    qkv[:, :heads, 0] = 100.0
    cos, sin = torch.ones((batch, d), dtype=torch.bfloat16, device="cuda"), torch.zeros((batch, d), dtype=torch.bfloat16, device="cuda")
    out = torch.empty((batch, heads * d), dtype=torch.bfloat16, device="cuda")
    ws = torch.zeros(lib.qwen2_decode_attention_workspace_bytes(batch, kv_heads, max_length), dtype=torch.uint8, device="cuda")
    _lib.check(lib.qwen2_decode_attention(
        _p(qkv), _p(cos), _p(sin), _p(k_cache), _p(v_cache), _p(torch.tensor([pos], device="cuda")), _p(out), batch,
        heads, kv_heads, d, max_length, ctypes.c_float(d ** -0.5), _p(ws), ws.numel(), _stream()))
    keys = torch.cat((k_cache[:, :, :pos], qkv[:, heads:heads + kv_heads, None]), dim=2)[:, :, dead:].double()
    values = torch.cat((v_cache[:, :, :pos], qkv[:, heads + kv_heads:, None]), dim=2)[:, :, dead:].double()
    q = qkv[:, :heads].reshape(batch, kv_heads, -1, 1, d).double()
    scores = (q * keys.unsqueeze(2)).sum(-1) * d ** -0.5
    want = (torch.softmax(scores, dim=-1) @ values).reshape(batch, heads * d)
    err = (out.double() - want).abs()
    bound = want.abs() * 2.0 ** -8 + want.abs().max() * 2.0 ** -16 * (1 + scores.abs().max())
    assert bool((err <= bound).all()), (err - bound).max().item()


@pytest.mark.parametrize("batch,heads,kv_heads,length", [(1, 12, 2, 100), (3, 4, 4, 33)])
def test_prefill_attention_into_the_projections(batch, heads, kv_heads, length):
    """The output over qkv's own memory, and qkv as the workspace of an output
    elsewhere: the same bits."""
    lib = _lib.load()
    d, rows = 128, batch * length
    qkv = torch.randn((rows, (heads + 2 * kv_heads) * d), generator=_gen(length), device="cuda").to(torch.bfloat16)
    positions = torch.arange(length, device="cuda").repeat(batch)
    cos, sin = RotaryEmbedding(d, 1_000_000.0).cuda()(positions, torch.bfloat16)
    ws = torch.empty(lib.qwen2_prefill_attention_workspace_bytes(batch, heads, length), dtype=torch.uint8, device="cuda")
    size = rows * heads * d
    outs = []
    for at in (None, "workspace", 0, qkv.numel() - size, qkv.numel() - 64):
        memory = torch.cat((qkv.flatten(), torch.zeros(size, dtype=torch.bfloat16, device="cuda")))
        elsewhere = at in (None, "workspace")
        out = torch.empty(size, dtype=torch.bfloat16, device="cuda") if elsewhere else memory[at: at + size]
        caches = torch.zeros((2, batch, kv_heads, length, d), dtype=torch.bfloat16, device="cuda")
        _lib.check(lib.qwen2_prefill_attention(
            _p(memory), _p(cos), _p(sin), _p(caches[0]), _p(caches[1]), _p(out), batch, length, heads, kv_heads, d,
            length, ctypes.c_float(d ** -0.5), _p(memory if at == "workspace" else ws), ws.numel(), _stream()))
        outs.append(torch.cat((out, caches.flatten())))
    assert all(torch.equal(o, outs[0]) for o in outs)


@pytest.mark.parametrize("scale", [0.0, -0.0, 1e-42])
@pytest.mark.parametrize("length", [5, 70])
def test_prefill_attention_without_scale(length, scale):
    """A scale of zero (or too small for a normal number) is the mean of the
    values so far: exact bf16 weights of one, fp32 sums."""
    lib = _lib.load()
    d, heads, kv_heads = 128, 4, 2
    qkv = torch.randn((length, (heads + 2 * kv_heads) * d), generator=_gen(length), device="cuda").to(torch.bfloat16)
    cos, sin = RotaryEmbedding(d, 1_000_000.0).cuda()(torch.arange(length, device="cuda"), torch.bfloat16)
    caches = torch.zeros((2, 1, kv_heads, length, d), dtype=torch.bfloat16, device="cuda")
    out = torch.empty((length, heads * d), dtype=torch.bfloat16, device="cuda")
    ws = torch.empty(lib.qwen2_prefill_attention_workspace_bytes(1, heads, length), dtype=torch.uint8, device="cuda")
    _lib.check(lib.qwen2_prefill_attention(
        _p(qkv), _p(cos), _p(sin), _p(caches[0]), _p(caches[1]), _p(out), 1, length, heads, kv_heads, d, length,
        ctypes.c_float(scale), _p(ws), ws.numel(), _stream()))
    values = qkv[:, (heads + kv_heads) * d:].double().view(length, kv_heads, 1, d).expand(-1, -1, heads // kv_heads, d)
    count = torch.arange(1, length + 1, device="cuda").double().view(-1, 1, 1, 1)
    want = (values.cumsum(0) / count).reshape(length, heads * d)
    err = (out.double() - want).abs()
    assert bool((err <= want.abs() * 2.0 ** -8 + want.abs().max() * 2.0 ** -16).all()), err.max().item()


@pytest.mark.parametrize("batch,heads,kv_heads,length,past,masking", [
    (1, 12, 2, 1, 0, "none"),        # one row, its own key only
    (4, 12, 2, 33, 0, "left"),       # left-padded prompts: rows without an allowed key
    (3, 12, 2, 1, 127, "left"),      # a cached step; the new key starts a block
    (2, 3, 3, 40, 29, "random"),     # rows cross block boundaries at an offset; any key may be excluded
    (2, 16, 1, 65, 70, "random"),    # sixteen query heads per key/value head
    (1, 4, 2, 300, 500, "none"),     # many blocks per wave
    (2, 4, 4, 5, 31, "all"),         # every key excluded for one sequence
])
def test_cached_attention_matches_torch(batch, heads, kv_heads, length, past, masking):
    """qwen2_cached_attention against the module path's torch restatement in
    fp64 (bound as in the prompt attention's edge test); the cache is the
    past followed by the rotated keys and the values, bit for bit."""
    from qwen_int4_hip.kernels import cached_attention_hip

    g = _gen(batch * 1000 + length + past)
    d, total = 128, past + length
    q = torch.randn((batch, length, heads * d), generator=g, device="cuda").to(torch.bfloat16)
    k, v = (torch.randn((batch, length, kv_heads * d), generator=g, device="cuda").to(torch.bfloat16) for _ in range(2))
    cache = None
    if past:
        cache = tuple(torch.randn((2, batch, kv_heads, past, d), generator=g, device="cuda").to(torch.bfloat16))
    mask = torch.ones((batch, total), dtype=torch.bool, device="cuda")
    if masking == "left":
        for b in range(1, batch):
            mask[b, : total * b // (batch + 1)] = False
    elif masking == "random":
        mask = torch.rand((batch, total), generator=g, device="cuda") < 0.7
    elif masking == "all":
        mask[-1] = False
    positions = (mask.long().cumsum(-1) - 1).clamp_min(0)[:, -length:]
    cos, sin = RotaryEmbedding(d, 1_000_000.0).cuda()(positions, torch.bfloat16)
    out, (new_k, new_v) = cached_attention_hip(q, k, v, cos, sin, cache, mask, num_heads=heads, num_kv_heads=kv_heads)

    def split(t):
        return t.view(batch, length, -1, d).transpose(1, 2)

    c, s = cos.unsqueeze(1), sin.unsqueeze(1)
    qr = split(q) * c + rotate_half(split(q)) * s
    kr = split(k) * c + rotate_half(split(k)) * s
    want_k, want_v = (kr, split(v)) if cache is None else (torch.cat((cache[0], kr), 2), torch.cat((cache[1], split(v)), 2))
    assert torch.equal(new_k, want_k) and torch.equal(new_v, want_v)
    assert new_k.is_contiguous() and new_v.is_contiguous()
    allowed = torch.ones((length, total), dtype=torch.bool, device="cuda").tril(past) & mask[:, None, None, :]
    kk, vv = (t.double().repeat_interleave(heads // kv_heads, dim=1) for t in (want_k, want_v))
    scores = torch.matmul(qr.double(), kk.transpose(-1, -2).contiguous()) * d ** -0.5
    probs = torch.softmax(scores.masked_fill(~allowed, float("-inf")), dim=-1)
    probs = torch.where(allowed.any(-1, keepdim=True), probs, torch.zeros_like(probs))
    want = torch.matmul(probs, vv).transpose(1, 2).reshape(batch, length, heads * d)
    err = (out.double() - want).abs()
    bound = want.abs() * 2.0 ** -8 + want.abs().max() * 2.0 ** -16 * (1 + scores.abs().max())
    assert bool((err <= bound).all()), (err - bound).max().item()
    blind = ~allowed.any(-1).expand(batch, 1, length).squeeze(1)
    assert bool((out[blind] == 0).all())


@pytest.mark.parametrize("batch,length,past", [(4, 300, 0), (6, 1, 1500)])
def test_cached_attention_keeps_the_probabilities_bits(batch, length, past):
    """Probabilities of fp32: sums of some hundred products then err by about
    2^-21 of the value, and an output is another bf16 value (spacing 2^-8 or
    more) than the exact result's for one in 2^12 of them.  Of 16 bits (2^-17)
    it would be one in 2^9."""
    from qwen_int4_hip.kernels import cached_attention_hip

    g = _gen(length + past)
    d, heads, kv_heads, total = 128, 12, 2, length + past
    q, k, v = (torch.randn((batch, length, h * d), generator=g, device="cuda").to(torch.bfloat16)
               for h in (heads, kv_heads, kv_heads))
    cache = None
    if past:
        cache = tuple(torch.randn((2, batch, kv_heads, past, d), generator=g, device="cuda").to(torch.bfloat16))
    mask = torch.ones((batch, total), dtype=torch.bool, device="cuda")
    positions = torch.arange(past, total, device="cuda").expand(batch, length)
    cos, sin = RotaryEmbedding(d, 1_000_000.0).cuda()(positions, torch.bfloat16)
    out, (keys, values) = cached_attention_hip(q, k, v, cos, sin, cache, mask, num_heads=heads, num_kv_heads=kv_heads)
    qr = q.view(batch, length, heads, d).transpose(1, 2)
    qr = qr * cos.unsqueeze(1) + rotate_half(qr) * sin.unsqueeze(1)
    keys, values = (t.double().repeat_interleave(heads // kv_heads, dim=1) for t in (keys, values))
    allowed = torch.ones((length, total), dtype=torch.bool, device="cuda").tril(past)
    scores = torch.matmul(qr.double(), keys.transpose(-1, -2).contiguous()) * d ** -0.5
    probs = torch.softmax(scores.masked_fill(~allowed, float("-inf")), dim=-1)
    want = torch.matmul(probs, values).transpose(1, 2).reshape(batch, length, heads * d).to(torch.bfloat16)
    assert (out != want).float().mean().item() <= 2.0 ** -11


def test_cached_attention_takes_no_past_of_another_shape():
    """A past that the kernels would read out of its bounds, and states in which
    torch's operators are followed, are left to torch."""
    from torch.autograd import forward_ad
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode

    from qwen_int4_hip.kernels import cached_attention_hip

    q, kv = (torch.randn((2, 3, h * 128), device="cuda").to(torch.bfloat16) for h in (4, 2))
    cos = torch.ones((2, 3, 128), device="cuda", dtype=torch.bfloat16)
    mask = torch.ones((2, 10), device="cuda", dtype=torch.bool)

    def past(*shape):
        return torch.zeros(shape, device="cuda", dtype=torch.bfloat16)

    def call(*caches):
        return cached_attention_hip(q, kv, kv, cos, cos, caches, mask, num_heads=4, num_kv_heads=2)

    whole = past(2, 2, 7, 128)
    for caches in ((past(2, 1, 7, 128), whole), (whole, past(2, 1, 7, 128)), (past(2, 2, 7, 64),) * 2,
                   (whole, past(2, 2, 6, 128)), (past(1, 2, 7, 128),) * 2, (past(2, 2, 7),) * 2, (whole,) * 3,
                   (past(2, 4, 7, 128),) * 2):
        assert call(*caches) is None, [tuple(t.shape) for t in caches]
    for mode in (TorchFunctionMode(), TorchDispatchMode(), forward_ad.dual_level()):
        with mode:
            assert call(whole, whole) is None, type(mode)
    assert call(whole, whole) is not None


def test_cached_attention_leaves_other_tensors_to_torch():
    from qwen_int4_hip.kernels import cached_attention_hip

    q = torch.randn((2, 3, 256), device="cuda").to(torch.bfloat16)
    cos = torch.ones((2, 3, 128), device="cuda", dtype=torch.bfloat16)
    mask = torch.ones((2, 3), device="cuda", dtype=torch.bool)
    base = dict(q=q, k=q, v=q, cos=cos, sin=cos, past=None, mask=mask)
    past = (torch.zeros((2, 2, 4, 128), device="cuda", dtype=torch.bfloat16),) * 2

    def call(**other):
        return cached_attention_hip(**{**base, **other}, num_heads=2, num_kv_heads=2)

    assert call() is not None
    for name, other in {"fp16": dict(q=q.half()), "host": dict(k=q.cpu()), "mask": dict(mask=mask[:, :2]),
                        "uncovered past": dict(past=past), "head": dict(cos=cos[..., :64]),
                        "gradient": dict(past=(past[0].clone().requires_grad_(), past[1]),
                                         mask=torch.ones((2, 7), device="cuda", dtype=torch.bool))}.items():
        assert call(**other) is None, name
    strided = q.repeat(1, 1, 2)[..., :256]
    got, want = call(q=strided, mask=mask.to(torch.int64)), call()
    assert torch.equal(got[0], want[0])


@pytest.mark.parametrize("rows,inter", [(1, 8960), (4, 8960), (16, 100)])
def test_silu_mul_matches_torch(rows, inter):
    lib = _lib.load()
    g = _gen(rows + inter)
    gate_up = (torch.randn((rows, 2 * inter), generator=g, device="cuda") * 4).to(torch.bfloat16)
    want = torch.nn.functional.silu(gate_up[:, :inter].float()) * gate_up[:, inter:].float()
    out = torch.empty((rows, inter), dtype=torch.float32, device="cuda")
    _lib.check(lib.qwen2_silu_mul(_p(gate_up), _p(out), rows, inter, _stream()))
    torch.cuda.synchronize()
    assert torch.allclose(out, want, rtol=2e-6, atol=1e-30)
    assert (out == want).float().mean().item() >= 0.99


def _weights(n, k, seed, asymmetric=False):
    from oracle import oracle as O

    q, sc, z = (O.asymmetric_weights(n, k, seed) if asymmetric else O.symmetric_weights(n, k, seed))
    return tuple(torch.from_numpy(t).cuda() for t in (q, sc, z))


def _normwise(got, want):
    return ((got.float() - want.float()).abs().max() / want.float().abs().max()).item()


@pytest.mark.parametrize("rows", [1, 4, 9, 16])
@pytest.mark.parametrize("n,k", [(1536, 8960), (100, 128), (256, 1536)])
def test_linear_swiglu_matches_silu_then_reference_linear(rows, n, k):
    """w4g64_linear_swiglu = fp32 silu(gate) * up (torch) followed by the
    reference torch backend's fp32 linear (the oracle); the fp32 activations
    run exactly (three bf16 parts), so the output agrees to fp32 summation
    order (normwise 1e-5)."""
    from oracle import oracle as O

    lib = _lib.load()
    g = _gen(rows * 17 + n + k)
    gate_up = (torch.randn((rows, 2 * k), generator=g, device="cuda") * 3).to(torch.bfloat16)
    h = torch.nn.functional.silu(gate_up[:, :k].float()) * gate_up[:, k:].float()
    qw, sc, z = _weights(n, k, 9)
    want = O.reference_linear_torch(h, qw, sc, z, None, out_features=n, in_features=k)
    ws = torch.zeros(max(1, lib.w4g64_linear_workspace_bytes(rows, n, k, _lib.DTYPE_BF16_SWIGLU)),
                     dtype=torch.uint8, device="cuda")
    y = torch.empty((rows, n), dtype=torch.float32, device="cuda")
    _lib.check(lib.w4g64_linear_swiglu(_p(gate_up), _p(qw), _p(sc), _p(z), None, 0, _p(y), rows, n, k, _p(ws),
                                       ws.numel(), _stream()))
    torch.cuda.synchronize()
    assert bool(torch.isfinite(y).all()) and _normwise(y, want) <= 1e-5


def _split3(h):
    """Exact three-way bf16 split of fp32 h by truncation: planes [3, ...]
    with hi + mid + lo == h (the decomposition the GEMV kernels stage)."""
    mask = torch.tensor(-65536, dtype=torch.int32, device=h.device)  # 0xFFFF0000
    hi = (h.contiguous().view(torch.int32) & mask).view(torch.float32)
    r1 = h - hi
    mid = (r1.view(torch.int32) & mask).view(torch.float32)
    lo = r1 - mid
    top = lambda t: (t.view(torch.int32) >> 16).to(torch.int16).view(torch.bfloat16)
    return torch.stack([top(hi), top(mid), top(lo)])


@pytest.mark.parametrize("rows", [1, 4, 9, 16])
@pytest.mark.parametrize("n,k", [(1536, 8960), (100, 128), (256, 1536)])
def test_linear_planes_form_matches_reference_linear(rows, n, k):
    """w4g64_linear with the bf16-planes activation form = the reference torch
    backend's fp32 linear of the planes' sum (the oracle); the planes are the
    exact split, so the output agrees to fp32 summation order (normwise 1e-5)."""
    from oracle import oracle as O

    lib = _lib.load()
    g = _gen(rows * 23 + n + k)
    h = torch.randn((rows, k), generator=g, device="cuda") * 2
    planes = _split3(h)
    assert torch.equal(planes.float().sum(0), h)
    qw, sc, z = _weights(n, k, 13, asymmetric=True)
    want = O.reference_linear_torch(h, qw, sc, z, None, out_features=n, in_features=k)
    ws = torch.zeros(max(1, lib.w4g64_linear_workspace_bytes(rows, n, k, _lib.DTYPE_BF16_PLANES)),
                     dtype=torch.uint8, device="cuda")
    y = torch.empty((rows, n), dtype=torch.float32, device="cuda")
    _lib.check(lib.w4g64_linear(_p(planes), _lib.DTYPE_BF16_PLANES, _p(qw), _p(sc), _p(z), None, 0, _p(y), rows, n,
                                k, _p(ws), ws.numel(), _stream()))
    torch.cuda.synchronize()
    assert bool(torch.isfinite(y).all()) and _normwise(y, want) <= 1e-5


def _partials_and_reduced(lib, x, code, qw, sc, z, rows, n, k):
    """w4g64_linear_partials' partial sums and w4g64_linear's reduced output."""
    parts = lib.w4g64_linear_partial_count(rows, n, k, code)
    assert parts >= 1
    partials = torch.empty((parts, rows, n), dtype=torch.float32, device="cuda")
    _lib.check(lib.w4g64_linear_partials(_p(x), code, _p(qw), _p(sc), _p(z), _p(partials), partials.numel() * 4,
                                         rows, n, k, _stream()))
    ws = torch.zeros(max(1, lib.w4g64_linear_workspace_bytes(rows, n, k, code)), dtype=torch.uint8, device="cuda")
    y = torch.empty((rows, n), dtype=torch.float32, device="cuda")
    _lib.check(lib.w4g64_linear(_p(x), code, _p(qw), _p(sc), _p(z), None, 0, _p(y), rows, n, k, _p(ws), ws.numel(),
                                _stream()))
    torch.cuda.synchronize()
    return partials, y


def _sum_in_order(partials):
    total = torch.zeros_like(partials[0])
    for part in partials:
        total = total + part
    return total + 0.0


@pytest.mark.parametrize("code", [_lib.DTYPE_BF16_PLANES, _lib.DTYPE_F32])
@pytest.mark.parametrize("rows", [1, 2, 5, 16])
@pytest.mark.parametrize("n,k", [(1536, 8960), (100, 128)])
def test_linear_partials_sum_to_the_reduced_linear(code, rows, n, k):
    """w4g64_linear_partials leaves the split-K partial sums to the caller:
    their sum in order from part 0 is w4g64_linear's fp32 output bit for bit
    (the reduction kernel adds them in that order)."""
    lib = _lib.load()
    g = _gen(rows * 29 + n + k + code)
    h = torch.randn((rows, k), generator=g, device="cuda") * 2
    x = _split3(h) if code == _lib.DTYPE_BF16_PLANES else h
    qw, sc, z = _weights(n, k, 31, asymmetric=True)
    partials, y = _partials_and_reduced(lib, x, code, qw, sc, z, rows, n, k)
    assert torch.equal(_sum_in_order(partials), y)
    if n == 1536 and k == 8960 and code == _lib.DTYPE_BF16_PLANES:
        assert partials.shape[0] > 1  # the decode down projection splits K


@pytest.mark.parametrize("rows", [1, 3])
def test_add_rmsnorm_adds_partial_sums_like_the_reduced_delta(rows):
    """qwen2_add_rmsnorm with delta W4G64_DTYPE_F32_PARTIALS(count) = with the
    reduced fp32 delta, bit for bit (sum and norm)."""
    lib = _lib.load()
    hidden, k = 1536, 8960
    g = _gen(rows + 41)
    x = (torch.randn((rows, hidden), generator=g, device="cuda") * 3).to(torch.bfloat16)
    planes = _split3(torch.randn((rows, k), generator=g, device="cuda") * 2)
    qw, sc, z = _weights(hidden, k, 37, asymmetric=False)
    partials, y = _partials_and_reduced(lib, planes, _lib.DTYPE_BF16_PLANES, qw, sc, z, rows, hidden, k)
    weight = (torch.rand(hidden, generator=g, device="cuda") + 0.5).to(torch.bfloat16)
    outs = []
    for delta, code in ((y, _lib.DTYPE_F32), (partials, _lib.dtype_f32_partials(partials.shape[0]))):
        out_sum, out = torch.empty_like(x), torch.empty_like(x)
        _lib.check(lib.qwen2_add_rmsnorm(_p(x), _p(delta), code, _p(weight), ctypes.c_float(1e-6), _p(out_sum),
                                         _p(out), rows, hidden, _stream()))
        outs.append((out_sum, out))
    torch.cuda.synchronize()
    assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])


@pytest.mark.parametrize("form,n", [("linear", 2048), ("planes", 17920)])
def test_linear_rmsnorm_adds_partial_sums_like_the_reduced_delta(form, n):
    """w4g64_linear_rmsnorm with the down projection's partial sums as delta =
    with their reduced fp32 output: residual sum and linear output bit for bit."""
    lib = _lib.load()
    hidden, inter = 1536, 8960
    g = _gen(n + 43)
    x = (torch.randn((1, hidden), generator=g, device="cuda") * 3).to(torch.bfloat16)
    planes = _split3(torch.randn((1, inter), generator=g, device="cuda") * 2)
    dq, ds, dz = _weights(hidden, inter, 47, asymmetric=True)
    partials, y = _partials_and_reduced(lib, planes, _lib.DTYPE_BF16_PLANES, dq, ds, dz, 1, hidden, inter)
    assert 1 < partials.shape[0] <= 8
    qw, sc, z = _weights(n, hidden, 53, asymmetric=True)
    weight = (torch.rand(hidden, generator=g, device="cuda") + 0.5).to(torch.bfloat16)
    pl = form == "planes"
    ws = torch.zeros(1 << 20, dtype=torch.uint8, device="cuda")
    outs = []
    for delta, code in ((y, _lib.DTYPE_F32), (partials, _lib.dtype_f32_partials(partials.shape[0]))):
        out_sum = torch.empty_like(x)
        out = (torch.empty((3, 1, n // 2), dtype=torch.bfloat16, device="cuda") if pl
               else torch.empty((1, n), dtype=torch.bfloat16, device="cuda"))
        _lib.check(lib.w4g64_linear_rmsnorm(_p(x), _p(delta), code, _p(weight), ctypes.c_float(1e-6), _p(out_sum),
                                            _p(qw), _p(sc), _p(z), None, 0, _p(out), 1 if pl else 0, 1, n, hidden,
                                            _p(ws), ws.numel(), _stream()))
        outs.append((out_sum, out))
    torch.cuda.synchronize()
    assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])


@pytest.mark.parametrize("rows", [1, 4, 9, 16])
@pytest.mark.parametrize("inter,k", [(8960, 1536), (100, 128), (72, 192)])
@pytest.mark.parametrize("with_bias", [False, True])
def test_gate_up_planes_matches_reference_swiglu_product(rows, inter, k, with_bias):
    """w4g64_linear_gate_up_planes over a stacked [gate; up] weight writes
    h = silu(bf16(gate)) * bf16(up) (model.py:133-135) as the exact bf16
    split of its fp32 value: the planes reassemble to h exactly, and h agrees
    with the oracle's projections (bf16 outputs, as the reference's) followed
    by torch's silu and product -- to the bf16 rounding of gate and up that
    a different fp32 summation order can flip (normwise 1e-2, the GEMM bar)."""
    from oracle import oracle as O

    lib = _lib.load()
    g = _gen(rows * 31 + inter + k)
    x = (torch.randn((rows, k), generator=g, device="cuda")).to(torch.bfloat16)
    gw = _weights(inter, k, 17)
    uw = _weights(inter, k, 19, asymmetric=True)
    qw, sc, z = (torch.cat([a.reshape(-1), b.reshape(-1)]) for a, b in zip(gw, uw))
    sc = sc.view(2 * inter, k // 64)
    bias = (torch.randn(2 * inter, generator=g, device="cuda") * 0.5).to(torch.bfloat16) if with_bias else None
    ws = torch.zeros(max(1, lib.w4g64_linear_workspace_bytes(rows, 2 * inter, k, _lib.DTYPE_BF16_GATE_UP)),
                     dtype=torch.uint8, device="cuda")
    planes = torch.empty((3, rows, inter), dtype=torch.bfloat16, device="cuda")
    _lib.check(lib.w4g64_linear_gate_up_planes(_p(x), _p(qw), _p(sc), _p(z), _p(bias),
                                               _lib.DTYPE_BF16 if with_bias else _lib.DTYPE_NONE, _p(planes), rows,
                                               2 * inter, k, _p(ws), ws.numel(), _stream()))
    torch.cuda.synchronize()
    h = planes.float().sum(0)
    assert torch.equal(_split3(h), planes)
    gate = O.reference_linear_torch(x, *gw, None if bias is None else bias[:inter], out_features=inter, in_features=k)
    up = O.reference_linear_torch(x, *uw, None if bias is None else bias[inter:], out_features=inter, in_features=k)
    want = torch.nn.functional.silu(gate.float()) * up.float()
    assert bool(torch.isfinite(h).all()) and _normwise(h, want) <= 1e-2


@pytest.mark.parametrize("rows", [17, 64, 512])
@pytest.mark.parametrize("n,k", [(1536, 8960), (100, 128)])
def test_linear_swiglu_gemm_rows(rows, n, k):
    """Prefill rows: the product is written as the GEMM's bf16 hi|lo planes and
    multiplied by bf16-rounded dequantized weights -- the GEMM bar, normwise
    1e-2."""
    from oracle import oracle as O

    lib = _lib.load()
    g = _gen(rows * 13 + n + k)
    gate_up = (torch.randn((rows, 2 * k), generator=g, device="cuda") * 3).to(torch.bfloat16)
    h = torch.nn.functional.silu(gate_up[:, :k].float()) * gate_up[:, k:].float()
    qw, sc, z = _weights(n, k, 11, asymmetric=True)
    want = O.reference_linear_torch(h, qw, sc, z, None, out_features=n, in_features=k)
    ws = torch.zeros(lib.w4g64_linear_workspace_bytes(rows, n, k, _lib.DTYPE_BF16_SWIGLU), dtype=torch.uint8,
                     device="cuda")
    y = torch.empty((rows, n), dtype=torch.float32, device="cuda")
    _lib.check(lib.w4g64_linear_swiglu(_p(gate_up), _p(qw), _p(sc), _p(z), None, 0, _p(y), rows, n, k, _p(ws),
                                       ws.numel(), _stream()))
    torch.cuda.synchronize()
    assert bool(torch.isfinite(y).all()) and _normwise(y, want) <= 1e-2


def _lm_head(x, weight, with_argmax=True):
    lib = _lib.load()
    rows, hidden = x.shape
    vocab = weight.shape[0]
    logits = torch.full((rows, vocab), float("nan"), dtype=torch.bfloat16, device="cuda")
    argmax = torch.full((rows,), -1, dtype=torch.int64, device="cuda") if with_argmax else None
    nbytes = lib.qwen2_lm_head_workspace_bytes(rows, vocab, hidden)
    assert nbytes > 0
    workspace = torch.zeros(nbytes, dtype=torch.uint8, device="cuda")
    _lib.check(lib.qwen2_lm_head(_p(x), _p(weight), _p(logits), _p(argmax), rows, vocab, hidden, _p(workspace),
                                 nbytes, _stream()))
    torch.cuda.synchronize()
    return logits, argmax


def _first_argmax(logits):
    """torch.argmax's rule on bf16 rows, written out: the first index of the
    largest value, NaN largest (torch documents the first occurrence)."""
    values = logits.float()
    nan = torch.isnan(values)
    top = torch.where(nan.any(dim=1, keepdim=True), nan, values == values.max(dim=1, keepdim=True).values)
    return top.float().argmax(dim=1)  # first True


@pytest.mark.parametrize("rows,vocab,hidden", [(1, 151936, 1536), (2, 151936, 1536), (16, 4099, 1536),
                                               (5, 1000, 896), (3, 257, 128), (1, 33, 4096), (7, 2048, 3584)])
def test_lm_head_matches_fp64_and_argmax_is_torchs(rows, vocab, hidden):
    g = _gen(rows * 1000 + hidden)
    x = (torch.randn((rows, hidden), generator=g, device="cuda")).to(torch.bfloat16)
    weight = (torch.randn((vocab, hidden), generator=g, device="cuda") * 0.02).to(torch.bfloat16)
    logits, argmax = _lm_head(x, weight)
    exact = x.double() @ weight.double().T
    # fp32 sums of exact bf16 products, one bf16 rounding: within half a bf16
    # ulp of the exact value plus the fp32 summation error
    bound = exact.abs() * 2.0 ** -8 + 1e-5 * (x.double().abs() @ weight.double().abs().T)
    assert bool(((logits.double() - exact).abs() <= bound).all())
    assert torch.equal(argmax, logits.argmax(dim=1))
    assert torch.equal(argmax, _first_argmax(logits))
    # without the argmax: same logits, no workspace needed
    again, _ = _lm_head(x, weight, with_argmax=False)
    assert torch.equal(again, logits)


def test_lm_head_argmax_ties_and_nan():
    hidden, vocab = 256, 3000
    g = _gen(77)
    weight = (torch.randn((vocab, hidden), generator=g, device="cuda") * 0.02).to(torch.bfloat16)
    # rows 2900, 40 and 1999 equal the largest row: ties resolve to the first
    big = torch.full((hidden,), 0.5, dtype=torch.bfloat16, device="cuda")
    for v in (2900, 40, 1999):
        weight[v] = big
    x = torch.ones((4, hidden), dtype=torch.bfloat16, device="cuda")
    x[1] = -1.0  # all-negative ties: row 0 of the smallest weights wins instead
    x[2, 5] = float("nan")  # every logit NaN: index 0
    x[3] = 0.0  # every logit +0: index 0
    logits, argmax = _lm_head(x, weight)
    assert argmax[0].item() == 40
    assert torch.equal(argmax, _first_argmax(logits))
    assert argmax[2].item() == 0 and argmax[3].item() == 0


@pytest.mark.parametrize("rows,vocab", [(1, 1), (3, 4095), (17, 4096), (24, 4097), (5, 8200), (33, 151936)])
def test_argmax_of_any_rows(rows, vocab):
    """qwen2_argmax at the edges of its slices, aligned rows and not, with ties
    over slices, NaN, infinities and zeros of both signs."""
    lib = _lib.load()
    logits = torch.randn((rows, vocab), generator=_gen(vocab), device="cuda").to(torch.bfloat16)
    logits[0] = float("-inf")
    if rows > 2:
        logits[1, vocab // 3] = logits[1, vocab - 1] = logits[1].max() + 1  # the first of two
        logits[2] = -0.0
        logits[2, vocab // 2] = 0.0  # equal to -0: index 0
    if rows > 4:
        logits[3, vocab - 1] = float("nan")
        logits[4, vocab - 2:] = float("inf")
    need = lib.qwen2_argmax_workspace_bytes(rows, vocab)
    workspace = torch.full((need,), 0xFF, dtype=torch.uint8, device="cuda")
    got = torch.empty(rows, dtype=torch.int64, device="cuda")
    _lib.check(lib.qwen2_argmax(_p(logits), _p(got), rows, vocab, _p(workspace), need, _stream()))
    assert torch.equal(got, _first_argmax(logits))
    assert lib.qwen2_argmax(_p(logits), _p(got), rows, vocab, _p(workspace), need - 1, _stream()) != 0


def test_lm_head_repeated_calls_share_the_workspace():
    """Back-to-back calls on one stream reuse one workspace."""
    lib = _lib.load()
    g = _gen(5)
    weight = (torch.randn((151936, 1536), generator=g, device="cuda") * 0.02).to(torch.bfloat16)
    nbytes = lib.qwen2_lm_head_workspace_bytes(4, 151936, 1536)
    workspace = torch.zeros(nbytes, dtype=torch.uint8, device="cuda")
    outs = []
    for seed in range(6):
        x = torch.randn((4, 1536), generator=_gen(seed), device="cuda").to(torch.bfloat16)
        logits = torch.empty((4, 151936), dtype=torch.bfloat16, device="cuda")
        argmax = torch.empty(4, dtype=torch.int64, device="cuda")
        _lib.check(lib.qwen2_lm_head(_p(x), _p(weight), _p(logits), _p(argmax), 4, 151936, 1536, _p(workspace),
                                     nbytes, _stream()))
        outs.append((logits, argmax))
    torch.cuda.synchronize()
    for logits, argmax in outs:
        assert torch.equal(argmax, logits.argmax(dim=1))


SMALL128 = SimpleNamespace(hidden_size=256, num_attention_heads=2, num_key_value_heads=1, head_dim=128,
                           intermediate_size=512, num_hidden_layers=3, vocab_size=512, rms_norm_eps=1e-6,
                           rope_theta=1_000_000.0)


def _build(config, seed):
    from qwen_int4_hip import QuantLinear, quantize_symmetric_rtn

    gen = _gen(seed)
    model = QwenInt4ForCausalLM(config, packing="canonical", group_size=64).cuda()
    with torch.no_grad():
        emb = model.model.embed_tokens.weight
        emb.copy_(torch.randn(emb.shape, generator=gen, device="cuda") * 0.02)
        for module in model.modules():
            if isinstance(module, QuantLinear):
                w = torch.randn((module.out_features, module.in_features), generator=gen, device="cuda") * 0.02
                q, s = quantize_symmetric_rtn(w, group_size=64)
                module.qweight.copy_(q)
                module.scales.copy_(s)
                if module.bias is not None:
                    module.bias.copy_(torch.randn(module.out_features, generator=gen, device="cuda") * 0.02)
    return model.eval()


def _cos(a, b):
    return torch.nn.functional.cosine_similarity(a.double().flatten(), b.double().flatten(), dim=0).item()


def test_fuse_projections_keeps_state_dict_and_eager_outputs():
    from qwen_int4_hip.decode import fuse_projections

    model = _build(SMALL128, 3)
    tokens = torch.randint(0, SMALL128.vocab_size, (1, 9), generator=torch.Generator().manual_seed(0)).cuda()
    with torch.inference_mode():
        before = model(tokens)
        state = {k: v.clone() for k, v in model.state_dict().items()}
        fused = fuse_projections(model)
        after = model(tokens)
    assert torch.equal(before, after)
    assert state.keys() == model.state_dict().keys()
    assert all(torch.equal(state[k], v) for k, v in model.state_dict().items())
    attn = model.model.layers[0].self_attn
    assert attn.k_proj.qweight.data_ptr() == attn.q_proj.qweight.data_ptr() + attn.q_proj.qweight.numel()
    assert fused[0]["qkv"]["out_features"] == 4 * 128 and fused[0]["gate_up"]["out_features"] == 1024
    # loading a state dict writes through the views into the fused buffers
    with torch.no_grad():
        sd = model.state_dict()
        sd["model.layers.0.self_attn.v_proj.scales"] = sd["model.layers.0.self_attn.v_proj.scales"] * 2
        model.load_state_dict(sd)
    assert torch.equal(fused[0]["qkv"]["scales"][384:], sd["model.layers.0.self_attn.v_proj.scales"])


@pytest.mark.parametrize("batch", [1, 2])
def test_fused_decode_step_matches_module_decode(batch):
    from qwen_int4_hip.generation import StaticGreedyDecoder

    model = _build(SMALL128, 11 + batch)
    prompt = torch.randint(0, SMALL128.vocab_size, (batch, 13), generator=torch.Generator().manual_seed(batch)).cuda()
    module = StaticGreedyDecoder(model, batch, 96, use_graph=False, fused=False)
    fused = StaticGreedyDecoder(model, batch, 96, use_graph=False, fused=True)
    graph = StaticGreedyDecoder(model, batch, 96, use_graph=True, fused=True)
    module.prefill(prompt)
    fused.prefill(prompt)
    graph.prefill(prompt)
    for step in range(70):  # crosses the 64-position chunk boundary of the attention kernel
        token = module.token.clone()
        want = module.step(token).clone()
        got = fused.step(token).clone()
        replay = graph.step(token).clone()
        assert torch.equal(got, replay), step  # graph replays run the same kernels on the same inputs
        assert _cos(got, want) >= 0.9999, (step, _cos(got, want))
        # the fused step's greedy choice is argmax of its own logits
        assert torch.equal(fused.token, got[:, -1].argmax(dim=-1, keepdim=True)), step
        assert torch.equal(graph.token, fused.token), step
    for (k0, v0), (k1, v1) in zip(module.caches, fused.caches):
        assert _cos(k0[:, :, :83], k1[:, :, :83]) >= 0.9999 and _cos(v0[:, :, :83], v1[:, :, :83]) >= 0.9999


def test_static_decoder_rejects_out_of_vocabulary_tokens():
    """Caller-supplied ids (a prompt, or the token given to step) outside
    [0, vocab) raise the reference embedding's IndexError before anything
    runs; the decoder's state is left as it was."""
    from qwen_int4_hip.generation import StaticGreedyDecoder

    model = _build(SMALL128, 23)
    dec = StaticGreedyDecoder(model, 1, 32, use_graph=True, fused=True)
    bad_prompt = torch.tensor([[1, SMALL128.vocab_size]], device="cuda")
    with pytest.raises(IndexError, match="index out of range"):
        dec.prefill(bad_prompt)
    dec.prefill(torch.tensor([[1, 2, 3]], device="cuda"))
    before = dec.token.clone()
    for bad in (-1, SMALL128.vocab_size):
        with pytest.raises(IndexError, match="index out of range"):
            dec.step(torch.tensor([[bad]], device="cuda"))
    assert dec.length == 3 and torch.equal(dec.token, before)
    logits = dec.step(torch.tensor([[SMALL128.vocab_size - 1]], device="cuda"))
    assert bool(torch.isfinite(logits.float()).all())


@pytest.mark.parametrize("batch,length", [(1, 40), (2, 17)])
def test_fused_prefill_matches_module_forward(batch, length):
    from qwen_int4_hip.decode import FusedPrefill

    model = _build(SMALL128, 5 + batch)
    prompt = torch.randint(0, SMALL128.vocab_size, (batch, length), generator=torch.Generator().manual_seed(7)).cuda()
    with torch.inference_mode():
        want, cache = model(prompt, use_cache=True)
        caches = model.new_static_cache(batch, 64, "cuda")
        got = FusedPrefill(model)(prompt, caches)
    assert got.shape == want.shape and _cos(got, want) >= 0.9999
    for (k0, v0), (k1, v1) in zip(cache, caches):
        assert _cos(k1[:, :, :length], k0) >= 0.9999 and _cos(v1[:, :, :length], v0) >= 0.9999
        assert not bool(k1[:, :, length:].any())  # positions past the prompt untouched


def test_full_width_fused_decode_against_reference_backend():
    """Qwen2-1.5B widths at 2 layers: the fused prefill and the fused
    graph-replayed decode steps stay within cosine 0.9999 of the model whose
    linears run the reference's torch backend (the oracle's restatement,
    backends.py:73-98)."""
    from test_model import QWEN2_1_5B, with_reference_linears

    from qwen_int4_hip.generation import StaticGreedyDecoder

    config = SimpleNamespace(num_hidden_layers=2, **QWEN2_1_5B)
    model = _build(config, 20260831)
    ref = with_reference_linears(model)
    prompt = torch.randint(0, config.vocab_size, (1, 64), generator=torch.Generator().manual_seed(4)).cuda()
    decoder = StaticGreedyDecoder(model, 1, 96)
    with torch.inference_mode():
        got = decoder.prefill(prompt)
        want, cache = ref(prompt, use_cache=True)
        assert _cos(got, want) >= 0.9999  # the fused prefill
        token = want[:, -1:].argmax(dim=-1)
        for _ in range(4):
            got = decoder.step(token)
            want, cache = ref(token, past_key_values=cache, use_cache=True)
            assert _cos(got, want) >= 0.9999
            token = want[:, -1:].argmax(dim=-1)
