"""GPU parity of kernels a dispatch rule chooses, at the sizes where each can
go wrong: edges of its tiles and chunks, remainders, alignment.

Bar: max |gpu - oracle| <= 1e-3 * max |oracle| (fp32 outputs, float64 oracle),
as for every attention kernel here."""

import numpy as np
import pytest
import torch

from oracle import sunshape_oracle as O
import sunshape_mlx_amd as S
from sunshape_mlx_amd import _hip, attention
from test_gpu_kernels import REL_TOL, decode_case, rel_err, t

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,hq,t_kv,t_buf,t_q,bdt,pad", [
    (128, 8, 300, 1, 1, torch.float16, 0),      # one token
    (128, 8, 300, 127, 1, torch.bfloat16, 0),   # one short of a chunk
    (128, 8, 300, 128, 1, torch.float16, 1),    # a chunk, rows at odd addresses
    (64, 8, 300, 129, 1, torch.float16, 0),     # a chunk and one token
    (64, 8, 0, 300, 1, torch.float32, 0),       # buffer only, several chunks
    (128, 2, 70, 200, 1, torch.float32, 1),     # one row per group
    (128, 8, 300, 130, 5, torch.float16, 0),    # causal rows that see part of the buffer
])
def test_merge_attends_the_buffer(d, hq, t_kv, t_buf, t_q, bdt, pad):
    """A hybrid cache's buffered tokens attended by the split-merge launch
    (rotated TurboQuant values, and token-major values with no transform)."""
    b, hkv, bits = 2, 2, 4
    cap = max(t_kv, 1)
    cents, perm, idx, vals, q = decode_case(7 * t_buf + t_kv, b, hq, hkv, d, t_kv, t_q, cap,
                                            v_dtype=np.float32)
    rng = np.random.default_rng(t_buf)
    kb = torch.from_numpy(rng.standard_normal((b, hkv, t_buf, d + pad)).astype(np.float32)).to(bdt)
    vb = torch.from_numpy(rng.standard_normal((b, hkv, t_buf, d + pad)).astype(np.float32)).to(bdt)
    kb, vb = kb[..., pad:], vb[..., pad:]
    full_k = torch.empty((b, hkv, t_buf, d + pad), dtype=bdt, device="cuda")
    full_v = torch.empty_like(full_k)
    kd, vd = full_k[..., pad:], full_v[..., pad:]
    kd.copy_(kb)
    vd.copy_(vb)
    scale = 1.0 / np.sqrt(d)
    kw = dict(causal=t_q > 1, q_offset=t_kv + t_buf - t_q if t_q > 1 else 0,
              out_dtype=torch.float32, buf_keys=kd, buf_values=vd, buf_len=t_buf)
    codes = rng.integers(0, 1 << bits, (b, hkv, cap, d)).astype(np.uint8)
    packed = O.pack_indices(codes, bits).astype(np.uint32)
    norms = (rng.random((b, hkv, cap)) * 3 + 0.1).astype(np.float32)
    levels = (O.lloyd_max_gaussian(bits)[0] / np.sqrt(d)).astype(np.float32)
    rot = O.rotation_matrix(d, 43)
    turbo = O.turboquant_decode(packed[:, :, :t_kv], norms[:, :, :t_kv], rot, levels, d, bits) \
        if t_kv else np.zeros((b, hkv, 0, d), np.float32)
    got = {"turbo": _hip.decode_attn_turboquant(t(q), scale, t(perm), t(cents), t(idx),
                                                t(packed.view(np.int32)), t(norms), levels, t(rot),
                                                bits, t_kv, **kw),
           "dense": _hip.decode_attn_dense(t(q), scale, t(perm), t(cents), t(idx), t(vals), t_kv,
                                           **kw)}
    ref_vals = {"turbo": turbo, "dense": vals[:, :, :t_kv]}
    for name, out in got.items():
        v_all = np.concatenate([ref_vals[name], vb.float().numpy()], axis=2)
        ref = O.sdpa_two_pass(q, scale, perm, cents, idx[:, :, :t_kv], kb.float().numpy(), v_all,
                              mask="causal" if t_q > 1 else None)
        assert rel_err(out.cpu().numpy(), ref) <= REL_TOL, name


@pytest.mark.parametrize("b,hq,hkv,d,t_kv,t_buf,t_q,cap,qdt", [
    (1, 4, 1, 128, 1, 0, 1, 256, torch.bfloat16),       # one token
    (1, 8, 2, 128, 64, 0, 1, 64, torch.bfloat16),       # one whole tile, full cache
    (2, 8, 2, 128, 1089, 0, 1, 1280, torch.bfloat16),   # 17 tiles and a token, several splits
    (1, 8, 2, 64, 1023, 0, 1, 1024, torch.float16),     # head_dim 64, last tile one short
    (1, 2, 2, 64, 130, 0, 5, 130, torch.bfloat16),      # causal rows, one query head per group
    (1, 8, 2, 128, 600, 37, 3, 640, torch.bfloat16),    # buffered tokens, causal rows
    (2, 6, 2, 128, 0, 20, 1, 64, torch.bfloat16),       # buffer only, three rows per group
    (1, 8, 1, 128, 2000, 9, 1, 2048, torch.float32),    # float32 query, two row groups
])
def test_decode_bf16_values_on_the_matrix_cores(b, hq, hkv, d, t_kv, t_buf, t_q, cap, qdt):
    """ss_decode_attn_dense_mfma: token-major bfloat16 values, with and
    without buffered tokens, against the oracle over the same values."""
    cents, perm, idx, _, q = decode_case(31 * t_kv + t_buf, b, hq, hkv, d, t_kv, t_q, cap)
    rng = np.random.default_rng(t_kv + d)
    # rows past t_kv hold NaN: nothing may read them into the result
    vals = torch.full((b, hkv, cap, d), float("nan"), dtype=torch.bfloat16)
    vals[:, :, :t_kv] = torch.from_numpy(rng.standard_normal((b, hkv, t_kv, d)).astype(np.float32))
    kb = torch.from_numpy(rng.standard_normal((b, hkv, max(t_buf, 1), d)).astype(np.float32))
    vb = torch.from_numpy(rng.standard_normal((b, hkv, max(t_buf, 1), d)).astype(np.float32))
    kb, vb = kb.bfloat16(), vb.bfloat16()
    qd = torch.from_numpy(q).to(qdt).cuda()
    scale = 1.0 / np.sqrt(d)
    total = t_kv + t_buf
    # (kept alive for the plan's pointers)
    idx_d, vals_d, perm_d, cb = t(idx), vals.cuda(), t(perm), _hip.codebook_f16x2(t(cents))
    plan = _hip.prepare_decode_dense(qd, scale, perm_d, cb, d // 8, 256, idx_d, vals_d)
    out = plan(qd, t_kv, t_q > 1, total - t_q if t_q > 1 else 0, kb.cuda(), vb.cuda(), t_buf,
               out_dtype=torch.float32)
    # queries scaled and rounded in their own type, then exact
    qs = (qd * scale).float().cpu().numpy()
    v_all = np.concatenate([vals[:, :, :t_kv].float().numpy(), vb[:, :, :t_buf].float().numpy()],
                           axis=2)
    ref = O.sdpa_two_pass(qs, 1.0, perm, cents, idx[:, :, :t_kv],
                          kb[:, :, :t_buf].float().numpy() if t_buf else None, v_all,
                          mask="causal" if t_q > 1 else None)
    assert rel_err(out.cpu().numpy(), ref) <= REL_TOL


def _masked_cache(backend, bits, dtype, d, hkv, b, t_kv, buffer):
    rng = np.random.default_rng(t_kv + bits)
    codec = S.SunShapeBlockCodec(d, device="cuda")
    codec.load_state_dict({"centroids": rng.standard_normal((d // 8, 256, 8)).astype(np.float32),
                           "permutation": rng.permutation(d).astype(np.int32)})
    kw = {}
    if backend == "sunshape":
        vc = S.SunShapeBlockCodec(d, block_dim=4, device="cuda")
        vc.load_state_dict({"centroids": rng.standard_normal((d // 4, 256, 4)).astype(np.float32),
                            "permutation": rng.permutation(d).astype(np.int32)})
        kw["value_codec"] = vc
    cache = S.create_kv_cache(codec, n_kv_heads=hkv, dtype=dtype, value_backend=backend,
                              value_bits=bits or None, buffer_size=buffer, **kw)
    g = torch.Generator(device="cuda").manual_seed(t_kv)
    k = torch.randn((b, hkv, t_kv, d), generator=g, device="cuda").to(dtype)
    v = torch.randn((b, hkv, t_kv, d), generator=g, device="cuda").to(dtype)
    cache.update_and_fetch(k, v)
    return cache


@pytest.mark.parametrize("backend,bits,dtype,d,hq,hkv,t_kv,t_q,buffer", [
    ("fp16", 0, torch.float16, 128, 8, 2, 1, 1, 128),        # one key
    ("fp16", 0, torch.float16, 128, 8, 2, 1089, 1, 128),     # several splits, a ragged tile
    ("fp16", 0, torch.bfloat16, 64, 6, 2, 700, 3, 128),      # bf16 rows, three a head and query
    ("fp16", 0, torch.float16, 64, 8, 2, 300, 2, 16),        # hybrid fp16 with a buffer
    ("fp16", 0, torch.bfloat16, 128, 8, 2, 300, 1, 40),      # hybrid bf16 with a buffer
    ("grouped", 2, torch.float16, 128, 8, 2, 900, 1, 128),   # register units
    ("grouped", 4, torch.float16, 128, 8, 2, 900, 1, 20),    # loader-wave shape
    ("grouped", 3, torch.float16, 128, 8, 2, 333, 1, 20),    # packed rows on the vector ALUs
    ("turboquant", 2, torch.float16, 128, 8, 2, 600, 1, 30),
    ("turboquant", 4, torch.float16, 64, 2, 2, 333, 1, 20),
    ("sunshape", 8, torch.float16, 128, 8, 2, 1500, 1, 128),
    ("sunshape", 8, torch.float16, 64, 8, 2, 200, 2, 10),
])
def test_masked_decodes_equal_the_two_pass_path(backend, bits, dtype, d, hq, hkv, t_kv, t_q, buffer):
    """Boolean and additive masks on the fused decodes against the two-pass
    path over the same cache: broadcast forms, per-head biases, rows with
    every key hidden (they average the values), the type's lowest value,
    -inf, and a row that is -inf throughout (NaN in both)."""
    b = 2
    cache = _masked_cache(backend, bits, dtype, d, hkv, b, t_kv, buffer)
    g = torch.Generator(device="cuda").manual_seed(3)
    q = torch.randn((b, hq, t_q, d), generator=g, device="cuda").to(dtype)
    keep = torch.rand((b, 1, t_q, t_kv), generator=g, device="cuda") > 0.4
    keep[1] = False
    bias = torch.randn((1, hq, 1, t_kv), generator=g, device="cuda")
    low = torch.where(keep, 0.0, torch.finfo(dtype).min).to(dtype)
    lowest = torch.where(keep, 0.5, torch.finfo(torch.float32).min)
    inf = torch.where(torch.rand((t_q, t_kv), generator=g, device="cuda") > 0.5, 0.0, -torch.inf)
    all_inf = inf.clone()
    all_inf[0] = -torch.inf
    masks = {"bool": keep, "row": keep[0, 0, 0], "per head": bias.half(),
             "expanded": bias.expand(b, hq, t_q, t_kv), "lowest f16": low,
             "lowest f32": lowest, "inf": inf, "all inf": all_inf, "int": (bias > 0).int(),
             "transposed": torch.randn((t_kv, t_q), generator=g, device="cuda").t()}
    for name, mask in masks.items():
        ref = attention._two_pass(cache, q, 0.11, mask, torch.float32)
        before = S.get_kernel_stats().get("sunshape_block_vq_score_hip", 0)
        got = S.sunshape_sdpa(q, cache, 0.11, mask, out_dtype=torch.float32)
        assert S.get_kernel_stats().get("sunshape_block_vq_score_hip", 0) == before, name  # fused
        assert torch.equal(torch.isnan(ref), torch.isnan(got)), name
        err = (got - ref).nan_to_num().abs().max() / ref.nan_to_num().abs().max().clamp(min=1e-30)
        assert float(err) <= REL_TOL, (name, float(err))


def test_kept_plan_follows_memory_given_in_place():
    """A permutation given other memory through ``.data``: the next bf16
    decode reads it there."""
    cache = _masked_cache("fp16", 0, torch.bfloat16, 128, 2, 1, 300, 128)
    q = torch.randn((1, 8, 1, 128), device="cuda").bfloat16()
    first = S.sunshape_sdpa(q, cache, 0.11)
    perm = cache.codec.permutation
    old = perm.detach()  # the old memory stays allocated
    perm.data = old.flip(0).clone()
    got = S.sunshape_sdpa(q, cache, 0.11)
    cache._decode_prepared = None
    assert torch.equal(got, S.sunshape_sdpa(q, cache, 0.11)) and not torch.equal(got, first)


@pytest.mark.parametrize("backend,bits,buffer,stores", [
    ("fp16", 0, 128, ("_key_indices", "_values")),
    ("fp16", 0, 20, ("_key_indices", "_values_il8", "_key_buffer", "_value_buffer")),
    ("grouped", 2, 20, ("_key_indices", "_values_il", "_value_scales", "_key_buffer")),
])
@pytest.mark.parametrize("held", [True, False])
def test_steps_follow_memory_given_in_place(backend, bits, buffer, stores, held):
    """Codebook, permutation and stores given other memory through ``.data``:
    the next step (one launch, or an append and a decode) reads and writes
    there, as where they are replaced by other tensors."""
    caches = [_masked_cache(backend, bits, torch.float16, 128, 2, 1, 300, buffer) for _ in range(2)]
    g = torch.Generator(device="cuda").manual_seed(9)
    k, v = torch.randn((2, 2, 1, 2, 1, 128), generator=g, device="cuda").half()
    q = torch.randn((1, 8, 1, 128), generator=g, device="cuda").half()
    outs, old = [], []
    for i in range(2):
        for cache in caches:
            cache.fuse_steps = held
            cache.update_and_fetch(k[i], v[i])
            outs.append(S.sunshape_sdpa(q, cache, 0.11))
            assert ("step" in cache.codec.last_score_backend) == held
        for in_place, cache in enumerate(caches if i == 0 else ()):
            c = cache.codec
            for where, name, new in (
                    [(c, "permutation", c.permutation.flip(0)), (c, "centroids", c.centroids * 0.5)] +
                    [(cache, n, getattr(cache, n).clone()) for n in stores]):
                if not in_place:
                    setattr(where, name, new)
                    continue
                old.append(getattr(where, name).data)  # stays allocated, versions of its own
                getattr(where, name).data = new
                old[-1].zero_()
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[2], outs[3])
    assert not torch.equal(outs[0], outs[2])
    assert torch.equal(caches[0].key_indices, caches[1].key_indices)
    assert not any(bool(t.any()) for t in old)


@pytest.mark.parametrize("backend,bits,d,buffer", [
    ("fp16", 0, 64, 128), ("fp16", 0, 128, 20), ("grouped", 4, 128, 20)])
def test_steps_of_unaligned_rows(backend, bits, d, buffer):
    """New keys and values as slices of wider rows, at addresses and strides
    the one-launch step does not take: as contiguous ones."""
    g = torch.Generator(device="cuda").manual_seed(d)
    wide = torch.randn((2, 1, 2, 1, d + 3), generator=g, device="cuda").half()
    q = torch.randn((1, 8, 1, d), generator=g, device="cuda").half()
    outs = []
    for k, v in (wide[..., 1:d + 1], wide[..., 1:d + 1].contiguous()):
        cache = _masked_cache(backend, bits, torch.float16, d, 2, 1, 300, buffer)
        cache.update_and_fetch(k, v)
        outs += [S.sunshape_sdpa(q, cache, 0.11), cache.key_indices, cache.values]
    assert torch.equal(outs[1], outs[4]) and torch.equal(outs[2], outs[5])
    assert rel_err(outs[0].float().cpu().numpy(), outs[3].float().cpu().numpy()) <= REL_TOL


def test_masks_that_carry_gradients_keep_the_two_pass_path():
    """A learned bias gets its gradient, a dual bias its tangent and vmap its
    batch: equal to the two-pass path's, and the same values as the fused
    decode of the plain mask."""
    cache = _masked_cache("fp16", 0, torch.float16, 128, 2, 1, 300, 128)
    g = torch.Generator(device="cuda").manual_seed(4)
    q = torch.randn((1, 8, 1, 128), generator=g, device="cuda").half()
    bias, tangent = torch.randn((2, 8, 1, 300), generator=g, device="cuda")
    plain = S.sunshape_sdpa(q, cache, 0.11, bias, out_dtype=torch.float32)
    grads = []
    for fn in (lambda m: S.sunshape_sdpa(q, cache, 0.11, m, out_dtype=torch.float32),
               lambda m: attention._two_pass(cache, q, 0.11, m, torch.float32)):
        m = bias.clone().requires_grad_()
        out = fn(m)
        assert rel_err(out.detach().cpu().numpy(), plain.cpu().numpy()) <= REL_TOL
        out.square().sum().backward()
        with torch.autograd.forward_ad.dual_level():
            dual = torch.autograd.forward_ad.make_dual(bias, tangent)
            jvp = torch.autograd.forward_ad.unpack_dual(fn(dual)).tangent.clone()
        grads.append((m.grad, jvp, torch.vmap(fn)(torch.stack([bias, tangent]))))
    for got, ref in zip(*grads):
        assert torch.allclose(got, ref, rtol=1e-5, atol=1e-6 * float(ref.abs().max()))
    assert torch.allclose(grads[0][2][0], plain, rtol=0, atol=REL_TOL * float(plain.abs().max()))


@pytest.mark.parametrize("b,hq,hkv,d,t_q,past,causal,qdt,vdt,n_raw,nc,ws_heads", [
    (1, 4, 1, 128, 1, 0, True, torch.float16, torch.float16, 0, 256, 0),       # one key, one row
    (1, 8, 2, 128, 33, 0, True, torch.float16, torch.float16, 0, 256, 0),      # a sub-tile and a key
    (2, 8, 2, 128, 64, 1, True, torch.bfloat16, torch.bfloat16, 0, 100, 0),    # 65 keys
    (1, 14, 2, 128, 70, 300, True, torch.float16, torch.bfloat16, 0, 256, 1),  # groups of 7 heads
    (1, 2, 2, 64, 129, 0, True, torch.float16, torch.float16, 0, 256, 0),      # one head a group
    (1, 8, 2, 64, 40, 77, False, torch.bfloat16, torch.bfloat16, 0, 17, 1),    # no causal cut
    (2, 8, 2, 128, 50, 200, True, torch.float16, torch.float16, 90, 256, 3),   # whole keys
    (1, 8, 2, 64, 30, 64, True, torch.bfloat16, torch.bfloat16, 31, 256, 0),   # and bf16 values
    (1, 64, 16, 128, 2080, 0, True, torch.float16, torch.float16, 0, 256, 0),  # 8 x 1 waves
    (1, 64, 16, 64, 1040, 30, True, torch.float16, torch.float16, 0, 256, 0),  # 4 x 1 waves
])
def test_prompt_kernel_matches_the_definition(b, hq, hkv, d, t_q, past, causal, qdt, vdt, n_raw, nc,
                                              ws_heads):
    """ss_prefill_attn against attention over the reconstructed keys in
    float64: tile edges, ragged rows, GQA groups, both value types, whole
    (buffered) keys, and workspaces that hold a few heads at a time.  Key
    and value slots past the last token hold NaN."""
    g = torch.Generator(device="cuda").manual_seed(t_q * 7 + past)
    nb, t_kv = d // 8, past + t_q
    cap = (t_kv + 255) // 256 * 256
    cents = torch.randn((nb, nc, 8), generator=g, device="cuda")
    perm = torch.randperm(d, generator=g, device="cuda").int()
    idx = torch.randint(0, nc, (b, hkv, cap, nb), generator=g, device="cuda").to(torch.uint8)
    v = torch.randn((b, hkv, t_kv, d), generator=g, device="cuda").to(vdt)
    v8 = torch.full((b, hkv, cap // 8, d, 8), float("nan"), dtype=vdt, device="cuda")
    _hip.append_values_il8(v, v8, 0)
    q = torch.randn((b, hq, t_q, d), generator=g, device="cuda").to(qdt)
    scale, t_raw0 = 0.1, t_kv - n_raw
    raw = torch.randn((b, hkv, max(n_raw, 1), d), generator=g, device="cuda").to(qdt)
    kw = {}
    if n_raw:
        rows, fac = _hip.raw_key_rows(raw, perm)
        kw = dict(kraw=rows, kfac=fac, t_raw0=t_raw0)
    out = _hip.prefill_attn(q, scale, perm, _hip.codebook_f16x2(cents), nc, idx, v8, t_kv,
                            causal=causal, q_offset=past if causal else 0,
                            out_dtype=torch.float32, **kw)
    if ws_heads:  # the same call with room for ws_heads heads
        lib = _hip.load_library()
        cb = _hip.codebook_f16x2(cents)
        ws = torch.empty(lib.ss_prefill_workspace_bytes(1, 1, d, t_kv) * ws_heads,
                         dtype=torch.uint8, device="cuda")
        out2 = torch.empty_like(out)
        _hip.check(lib.ss_prefill_attn(
            q.data_ptr(), _hip.dtype_code(qdt), b, hq, hkv, t_q, d, scale, perm.data_ptr(),
            cb.data_ptr(), nb, nc, idx.data_ptr(), cap, v8.data_ptr(), _hip.dtype_code(vdt), cap,
            t_kv, _hip.ptr(kw.get("kraw")), _hip.ptr(kw.get("kfac")), t_raw0, int(causal),
            past if causal else 0, out2.data_ptr(), _hip.SS_F32, ws.data_ptr(), ws.numel(),
            _hip.stream_handle(q.device)))
        assert torch.equal(out, out2)
    k = cents.double()[torch.arange(nb, device="cuda"), idx[:, :, :t_kv].long()].flatten(-2)
    if n_raw:
        k[:, :, t_raw0:] = raw[:, :, :n_raw].double()[..., perm.long()]
    qs = (q * scale).double()[..., perm.long()]
    rep = hq // hkv
    pos = torch.arange(t_kv, device="cuda")
    hide = pos[None] > past + torch.arange(t_q, device="cuda")[:, None]
    worst = 0.0
    for bi in range(b):
        for h in range(0, hq, 1 if t_q < 500 else 23):
            s = qs[bi, h] @ k[bi, h // rep].t()
            if causal:
                s = s.masked_fill(hide, float("-inf"))
            ref = torch.softmax(s, dim=-1) @ v[bi, h // rep].double()
            worst = max(worst, float((out[bi, h] - ref).abs().max() / ref.abs().max()))
    assert worst <= REL_TOL


@pytest.mark.parametrize("dtype,d,hq,hkv,buffer", [
    (torch.float16, 64, 8, 2, 128), (torch.float16, 128, 14, 2, 128), (torch.bfloat16, 128, 8, 2, 128),
    (torch.bfloat16, 64, 8, 2, 128), (torch.float16, 64, 8, 2, 40), (torch.bfloat16, 128, 8, 2, 40),
])
def test_float32_results_of_prompts_are_the_decodes(dtype, d, hq, hkv, buffer):
    """Prompts of shapes that a decode takes as well: the prompt kernel for
    results in the cache's type, the decode, which is nearer to 64 bits, for
    float32 ones."""
    cache = _masked_cache("fp16", 0, dtype, d, hkv, 1, 1400, buffer)
    g = torch.Generator(device="cuda").manual_seed(d + hq)
    q = torch.randn((1, hq, 900, d), generator=g, device="cuda").to(dtype)
    got = S.sunshape_sdpa(q, cache, 0.11, "causal")
    assert "prefill" in cache.codec.last_score_backend
    exact = S.sunshape_sdpa(q, cache, 0.11, "causal", out_dtype=torch.float32)
    assert "fused" in cache.codec.last_score_backend
    assert rel_err(got.float().cpu().numpy(), exact.cpu().numpy()) <= REL_TOL + torch.finfo(dtype).eps


@pytest.mark.parametrize("backend,bits,d,buffer", [("grouped", 2, 128, 20), ("grouped", 4, 64, 20),
                                                   ("turboquant", 2, 128, 20),
                                                   ("sunshape", 8, 128, 20)])
def test_masked_float32_caches_keep_float32_weights(backend, bits, d, buffer):
    cache = _masked_cache(backend, bits, torch.float32, d, 2, 1, 700, buffer)
    q = torch.randn((1, 8, 1, d), device="cuda")
    mask = torch.arange(700, device="cuda") > 9
    assert torch.equal(S.sunshape_sdpa(q, cache, 0.11, mask),
                       attention._two_pass(cache, q, 0.11, mask, torch.float32))


@pytest.mark.parametrize("n_t,offset,d,dtype,pad", [
    (1, 0, 128, torch.float16, 0), (8, 0, 64, torch.float16, 0), (7, 5, 128, torch.float32, 0),
    (30, 3, 128, torch.bfloat16, 0), (17, 8, 64, torch.float16, 1), (9, 7, 33, torch.float16, 0),
])
def test_append_il8_keeps_the_other_tokens(n_t, offset, d, dtype, pad):
    """Blocks at the ends of an append keep the tokens outside it; odd head
    dims, rows at odd addresses, float32 and bf16 values."""
    b, h, cap = 2, 3, 48
    g = torch.Generator(device="cuda").manual_seed(n_t)
    for out_dtype in (torch.float16, torch.bfloat16):
        if out_dtype == torch.bfloat16 and dtype != torch.bfloat16:
            continue
        v = torch.randn((b, h, n_t, d + pad), generator=g, device="cuda").to(dtype)[..., pad:]
        out = torch.randn((b, h, cap // 8, d, 8), generator=g, device="cuda").to(out_dtype)
        want = out.permute(0, 1, 2, 4, 3).reshape(b, h, cap, d).clone()
        want[:, :, offset:offset + n_t] = v.to(out_dtype)
        _hip.append_values_il8(v, out, offset)
        assert torch.equal(out.permute(0, 1, 2, 4, 3).reshape(b, h, cap, d), want)


@pytest.mark.parametrize("nb,bd,n,dtype,use_perm,pad", [
    (16, 8, 1, torch.float16, True, 0),       # one token
    (16, 8, 31, torch.bfloat16, True, 0),     # one short of a workgroup's tokens
    (32, 4, 33, torch.float32, True, 3),      # a workgroup and one, strided index rows
    (8, 8, 100, torch.float16, False, 0),     # head_dim 64, no permutation
    (16, 16, 65, torch.float16, True, 0),     # head_dim 256
    (4, 16, 64, torch.bfloat16, True, 1),
    (12, 8, 40, torch.float32, True, 0),      # 96 dims: the element kernel
])
def test_dequantised_rows_are_the_codebook_rows(nb, bd, n, dtype, use_perm, pad):
    g = torch.Generator(device="cuda").manual_seed(nb * n)
    d = nb * bd
    cents = torch.randn((nb, 200, bd), generator=g, device="cuda")
    store = torch.randint(0, 256, (n, nb + pad), generator=g, device="cuda", dtype=torch.uint8)
    idx = store[:, :nb]
    inv = torch.randperm(d, generator=g, device="cuda").to(torch.int32) if use_perm else None
    got = _hip.dequantize_blockvq(idx, cents, inv, out_dtype=dtype)
    rows = cents[torch.arange(nb, device="cuda"), idx.long().clamp(max=199)].flatten(1)
    want = rows[:, inv.long()] if use_perm else rows
    assert torch.equal(got, want.to(dtype))  # one rounding each


@pytest.mark.parametrize("bits,d,group,n_t,offset,cap,dtype,sz,pad", [
    (2, 128, 64, 1, 5, 32, torch.float16, torch.float16, 0),       # one token inside a word
    (2, 128, 128, 40, 30, 96, torch.bfloat16, torch.float32, 0),   # partial words at both ends
    (4, 128, 64, 33, 8, 64, torch.float16, torch.float16, 1),      # rows at odd addresses
    (4, 64, 32, 100, 29, 160, torch.float32, torch.float16, 0),    # head_dim 64
    (2, 64, 64, 64, 32, 96, torch.float16, torch.float32, 0),      # whole workgroups
])
def test_append_grouped_il_is_quantise_then_interleave(bits, d, group, n_t, offset, cap, dtype, sz, pad):
    """Codes, scales and zeros are the oracle's, and what other tokens hold
    (also in shared words) is left alone."""
    g = torch.Generator(device="cuda").manual_seed(n_t + d)
    v = torch.randn((2, 3, n_t, d + pad), generator=g, device="cuda").to(dtype)[..., pad:]
    il = torch.randint(-2**31, 2**31 - 1, (2, 3, cap * bits // 32, d), generator=g, device="cuda",
                       dtype=torch.int32)
    sc, ze = (torch.full((2, 3, cap, d // group), 7.0, device="cuda", dtype=sz) for _ in range(2))
    old = _hip.grouped_il_to_packed(il, bits, cap)
    _hip.append_values_grouped_il(v, bits, group, il, sc, ze, offset)
    rows = torch.zeros((2, 3, n_t, d * bits // 32), dtype=torch.int32, device="cuda")
    s1, z1 = (torch.zeros((2, 3, n_t, d // group), dtype=sz, device="cuda") for _ in range(2))
    _hip.quantize_values_grouped(v, bits, group, rows, s1, z1)
    packed, osc, oze, _ = O.quantize_values(v.float().cpu().numpy().reshape(-1, d), bits, group)
    assert np.array_equal(rows.cpu().numpy().reshape(packed.shape).view(np.uint32), packed)
    assert np.array_equal(s1.cpu().numpy().reshape(osc.shape), osc.astype(s1.cpu().numpy().dtype))
    assert np.array_equal(z1.cpu().numpy().reshape(oze.shape), oze.astype(z1.cpu().numpy().dtype))
    new = _hip.grouped_il_to_packed(il, bits, cap).view(torch.int32)
    want = old.view(torch.int32).clone()
    want[:, :, offset:offset + n_t] = rows
    assert torch.equal(new, want)
    for got, one in ((sc, s1), (ze, z1)):
        full = torch.full_like(got, 7.0)
        full[:, :, offset:offset + n_t] = one
        assert torch.equal(got, full)


@pytest.mark.parametrize("bits,d,hq,t_kv,t_buf,t_q,splits,spread,qdt", [
    (4, 128, 8, 1, 0, 1, 0, 0, torch.float16),       # one token, the kernel rotates
    (4, 128, 8, 64, 0, 1, 1, 0, torch.float16),      # one unit, one split
    (3, 128, 8, 65, 5, 1, 0, 0, torch.bfloat16),     # a unit and one token, buffered tokens
    (3, 64, 8, 700, 0, 1, 0, 0, torch.float32),      # head_dim 64: words straddled by dims
    (4, 64, 6, 1500, 9, 1, 3, 20, torch.float16),    # norms over 40 powers of two
    (3, 128, 8, 3000, 0, 3, 0, 20, torch.float32),   # ... causal rows
    (4, 128, 14, 5001, 130, 1, 0, 0, torch.float32),  # seven heads a group
])
def test_turboquant_rows_on_the_matrix_cores(bits, d, hq, t_kv, t_buf, t_q, splits, spread, qdt):
    """3/4-bit TurboQuant values read from their packed rows; no less exact
    than the vector-ALU kernel of the same call (1e-6 of the largest output
    for float32 rounding: ~16 roundings of 2^-24 in either)."""
    b, hkv, cap = 2, 2, t_kv + 37
    cents, perm, idx, _, q = decode_case(31 * t_kv + bits, b, hq, hkv, d, t_kv, t_q, cap)
    rng = np.random.default_rng(t_kv)
    codes = rng.integers(0, 1 << bits, (b, hkv, cap, d)).astype(np.uint8)
    packed = O.pack_indices(codes, bits).astype(np.uint32)
    norms = ((rng.random((b, hkv, cap)) + 0.1) *
             np.exp2(rng.integers(-spread, spread + 1, (b, hkv, cap)))).astype(np.float32)
    norms[:, :, t_kv:] = np.nan  # never read as a token
    levels = (O.lloyd_max_gaussian(bits)[0] / np.sqrt(d)).astype(np.float32)
    rot = O.rotation_matrix(d, 43)
    vals = O.turboquant_decode(packed[:, :, :t_kv], norms[:, :, :t_kv], rot, levels, d, bits)
    kb, vb = (rng.standard_normal((b, hkv, max(t_buf, 1), d)).astype(np.float32) for _ in range(2))
    qd = torch.from_numpy(q).to(qdt)
    scale = 1.0 / np.sqrt(d)
    kw = dict(causal=t_q > 1, q_offset=t_kv + t_buf - t_q if t_q > 1 else 0, out_dtype=torch.float32,
              n_splits=splits)
    if t_buf:
        kw.update(buf_keys=t(kb), buf_values=t(vb), buf_len=t_buf)
    cb = _hip.codebook_f16x2(t(cents))
    args = (qd.cuda(), scale, t(perm), t(cents), t(idx), t(packed.view(np.int32)), t(norms), levels,
            t(rot), bits, t_kv)
    outs = [_hip.decode_attn_turboquant(*args, codebook=c, **kw) for c in (cb, None)]
    # the definition in float64
    kc = np.stack([np.stack([O.dequantize_blockvq(idx[i, h, :t_kv], cents) for h in range(hkv)])
                   for i in range(b)]).astype(np.float64)
    qs = (qd * scale).double().numpy()
    inv = np.argsort(perm)
    kx = np.concatenate([kc[..., inv], kb[:, :, :t_buf].astype(np.float64)], 2)
    vx = np.concatenate([vals.astype(np.float64), vb[:, :, :t_buf].astype(np.float64)], 2)
    rep = hq // hkv
    sc = qs @ np.repeat(kx, rep, 1).transpose(0, 1, 3, 2)
    if t_q > 1:
        hide = np.arange(t_kv + t_buf)[None] > kw["q_offset"] + np.arange(t_q)[:, None]
        sc = np.where(hide, -np.inf, sc)
    p = np.exp(sc - sc.max(-1, keepdims=True))
    want = (p / p.sum(-1, keepdims=True)) @ np.repeat(vx, rep, 1)
    err, ref = (rel_err(o.cpu().numpy(), want) for o in outs)
    print("error", err, "vector-ALU kernel", ref)
    assert err <= REL_TOL and err <= ref + 1e-6


def _other_codec_cache(d, block_dim, backend, dtype):
    """A cache whose key codec no fused decode takes."""
    rng = np.random.default_rng(d + block_dim)
    codec = S.SunShapeBlockCodec(d, block_dim=block_dim, device="cuda")
    codec.load_state_dict({"centroids": rng.standard_normal((d // block_dim, 256, block_dim))
                           .astype(np.float32),
                           "permutation": rng.permutation(d).astype(np.int32)})
    cache = S.create_kv_cache(codec, n_kv_heads=2, dtype=dtype, value_backend=backend,
                              value_bits=4 if backend != "fp16" else None, buffer_size=20)
    g = torch.Generator(device="cuda").manual_seed(d)
    k, v = torch.randn((2, 1, 2, 150, d), generator=g, device="cuda").to(dtype)
    cache.update_and_fetch(k, v)
    return cache, torch.randn((1, 8, 1, d), generator=g, device="cuda").to(dtype)


@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("d,block_dim,backend,dtype", [
    (128, 4, "turboquant", torch.float16), (128, 4, "fp16", torch.bfloat16),
    (128, 4, "grouped", torch.bfloat16), (128, 16, "turboquant", torch.bfloat16),
    (64, 4, "fp16", torch.bfloat16),
    (80, 8, "turboquant", torch.float16), (112, 8, "fp16", torch.bfloat16),
    (72, 8, "turboquant", torch.bfloat16),
])
def test_other_codecs_take_the_two_pass_path(d, block_dim, backend, dtype, masked):
    cache, q = _other_codec_cache(d, block_dim, backend, dtype)
    mask = torch.arange(150, device="cuda") > 7 if masked else None
    got = S.sunshape_sdpa(q, cache, 0.1, mask)
    assert torch.equal(got, attention._two_pass(cache, q, 0.1, mask, dtype))


@pytest.mark.parametrize("backend,bits,dtype,d,hq,t_kv,t_q,buffer", [
    ("fp16", 0, torch.float16, 128, 8, 1300, 1, 128),
    ("fp16", 0, torch.float16, 64, 8, 400, 2, 16),
    ("fp16", 0, torch.bfloat16, 128, 8, 700, 1, 40),
    ("grouped", 2, torch.float16, 128, 8, 900, 1, 128),
    ("grouped", 4, torch.float16, 128, 8, 900, 1, 20),
    ("grouped", 3, torch.float16, 128, 8, 900, 1, 140),
    ("turboquant", 2, torch.float16, 128, 8, 900, 1, 140),
    ("turboquant", 4, torch.float16, 128, 8, 900, 1, 30),
    ("turboquant", 4, torch.float16, 64, 2, 900, 1, 30),
    ("sunshape", 8, torch.float16, 128, 8, 2500, 1, 140),
    ("sunshape", 8, torch.float16, 64, 8, 900, 2, 10),
])
def test_masks_of_any_magnitude_equal_the_two_pass_path(backend, bits, dtype, d, hq, t_kv, t_q, buffer):
    """Additive masks that hide by a large finite value: sequence 0 is padded
    on the left by more than a unit of 64 keys (a hidden unit is attended
    before a visible one), sequence 1 is hidden throughout."""
    cache = _masked_cache(backend, bits, dtype, d, 2, 2, t_kv, buffer)
    g = torch.Generator(device="cuda").manual_seed(3)
    q = torch.randn((2, hq, t_q, d), generator=g, device="cuda").to(dtype)
    keep = torch.rand((2, 1, t_q, t_kv), generator=g, device="cuda") > 0.1
    keep[0, ..., :t_kv // 2 + 5] = False
    keep[0, ..., -3:] = True
    keep[1] = False
    for low in (-1e4, -1e9, -1e10, -1e12, -1e30, -3e38):
        for mdt in (torch.float32, torch.bfloat16):
            if mdt == torch.bfloat16 and low not in (-1e9, -1e30):
                continue
            mask = torch.where(keep, 0.25, low).to(mdt)
            ref = attention._two_pass(cache, q, 0.11, mask, torch.float32)
            got = S.sunshape_sdpa(q, cache, 0.11, mask, out_dtype=torch.float32)
            assert torch.isfinite(ref).all() and torch.isfinite(got).all(), (low, mdt)
            err = (got - ref).abs().amax((1, 2, 3)) / ref.abs().amax((1, 2, 3))
            assert float(err.max()) <= REL_TOL, (low, mdt, err)


@pytest.mark.parametrize("backend,bits,dtype,d,buffer,masked,t_q", [
    ("fp16", 0, torch.float16, 128, 128, True, 3),
    ("fp16", 0, torch.bfloat16, 64, 40, True, 2),
    ("sunshape", 8, torch.float16, 128, 30, True, 2),
    ("grouped", 2, torch.bfloat16, 128, 30, False, 3),      # bf16 hybrids of quantised values
    ("turboquant", 4, torch.bfloat16, 64, 30, False, 200),  # ... and their prompts
    ("turboquant", 3, torch.bfloat16, 128, 30, True, 2),
])
def test_query_layouts_and_types_of_the_two_pass_path(backend, bits, dtype, d, buffer, masked, t_q):
    """Calls that the two-pass path takes in any layout and type: queries as
    (B, T, H, D) seen through transpose(1, 2), float64 queries and outputs,
    and gradients through the queries' scores of buffered keys."""
    cache = _masked_cache(backend, bits, dtype, d, 2, 2, 300, buffer)
    g = torch.Generator(device="cuda").manual_seed(t_q)
    q = torch.randn((2, t_q, 8, d), generator=g, device="cuda").to(dtype).transpose(1, 2)
    mask = torch.arange(300, device="cuda") > 9 if masked else "causal"
    ref = attention._two_pass(cache, q, 0.11, mask, torch.float32)
    got = S.sunshape_sdpa(q, cache, 0.11, mask, out_dtype=torch.float32)
    assert rel_err(got.cpu().numpy(), ref.cpu().numpy()) <= REL_TOL
    same = S.sunshape_sdpa(q.contiguous(), cache, 0.11, mask, out_dtype=torch.float32)
    assert torch.equal(got, same)
    for queries, out_dtype in ((q.double(), None), (q, torch.float64)):
        got = S.sunshape_sdpa(queries, cache, 0.11, mask, out_dtype=out_dtype)
        assert torch.equal(got, attention._two_pass(cache, queries, 0.11, mask, torch.float64))
    grads = []
    for fn in (S.sunshape_sdpa, lambda x, c, s, m: attention._two_pass(c, x, s, m, x.dtype)):
        x = q.float().requires_grad_()
        out = fn(x, cache, 0.11, mask)
        if out.requires_grad:  # (no buffered keys: the compressed scores carry none)
            out.square().sum().backward()
        grads.append(x.grad)
    assert grads[0] is grads[1] is None or torch.equal(*grads)


@pytest.mark.parametrize("backend,bits,dtype,d,masked", [
    ("fp16", 0, torch.float16, 128, True), ("grouped", 4, torch.float32, 64, True),
    ("turboquant", 4, torch.float16, 96, True), ("turboquant", 2, torch.bfloat16, 128, False),
    ("grouped", 2, torch.float16, 128, False)])
@pytest.mark.parametrize("hkv", [1, 2])
def test_rotated_hybrids_of_one_head(backend, bits, dtype, d, masked, hkv):
    """Buffered tokens of a rotated codec's cache, of one sequence and one KV
    head (size-1 dims, whose strides contiguous() leaves alone) or two."""
    rng = np.random.default_rng(d)
    codec = S.SunShapeBlockCodec(d, device="cuda", mode="rotated")
    codec.load_state_dict({"centroids": rng.standard_normal((d // 8, 256, 8)).astype(np.float32),
                           "rotation": np.linalg.qr(rng.standard_normal((d, d)))[0].astype(np.float32)})
    cache = S.create_kv_cache(codec, n_kv_heads=hkv, dtype=dtype, value_backend=backend,
                              value_bits=bits or None, buffer_size=50,
                              value_group_size=32)
    g = torch.Generator(device="cuda").manual_seed(d)
    k, v = torch.randn((2, 1, hkv, 130, d), generator=g, device="cuda").to(dtype)
    cache.update_and_fetch(k, v)
    q = torch.randn((1, 4 * hkv, 3, d), generator=g, device="cuda").to(dtype)
    mask = torch.arange(130, device="cuda") != 9 if masked else "causal"
    ref = attention._two_pass(cache, q, 0.1, mask, torch.float32)
    got = S.sunshape_sdpa(q, cache, 0.1, mask)
    assert rel_err(got.float().cpu().numpy(), ref.cpu().numpy()) <= REL_TOL + torch.finfo(dtype).eps


@pytest.mark.parametrize("bdt,t_buf", [(torch.float16, 1), (torch.float32, 127), (torch.bfloat16, 131)])
def test_merge_keeps_an_infinite_value_of_the_last_buffered_token(bdt, t_buf):
    """One dim of the last token is infinite: infinite in the output, the
    other dims as without it."""
    d, t_kv = 128, 200
    cents, perm, idx, vals, q = decode_case(t_buf, 1, 8, 2, d, t_kv, 1, t_kv, v_dtype=np.float32)
    g = torch.Generator(device="cuda").manual_seed(t_buf)
    kb, vb = torch.randn((2, 1, 2, t_buf, d), generator=g, device="cuda").to(bdt)
    outs = []
    for x in (1.0, float("inf")):
        vb[..., -1, 5] = x
        outs.append(_hip.decode_attn_dense(t(q), 0.1, t(perm), t(cents), t(idx), t(vals), t_kv,
                                           buf_keys=kb, buf_values=vb, buf_len=t_buf,
                                           out_dtype=torch.float32))
    assert bool((outs[1][..., 5] == float("inf")).all())
    outs[1][..., 5] = outs[0][..., 5]
    assert torch.equal(*outs)


@pytest.mark.parametrize("dtype,d,t_kv,masked", [
    (torch.bfloat16, 128, 67, False), (torch.bfloat16, 128, 1500, False),
    (torch.bfloat16, 64, 131, True), (torch.float16, 128, 1500, True),
])
def test_decodes_keep_infinite_values(dtype, d, t_kv, masked):
    """Infinite values of a cache: infinite in their dims of the output, and
    the other dims as without them.  (Of a key hidden by the mask: NaN, 0 *
    infinity, as in the two-pass path.)"""
    cache = _masked_cache("fp16", 0, dtype, d, 2, 1, t_kv, 128)
    q = torch.randn((1, 8, 1, d), generator=torch.Generator(device="cuda").manual_seed(1),
                    device="cuda").to(dtype)
    mask = torch.arange(t_kv, device="cuda") != 1 if masked else None
    plain = S.sunshape_sdpa(q, cache, 0.02, mask, out_dtype=torch.float32)
    dims = {7: (t_kv - 1, torch.inf), 20: (t_kv // 2, -torch.inf), 40: (0, torch.inf)}
    if masked:
        dims[41] = (1, torch.inf)
    v = cache._values  # (B, H, cap, D), or (B, H, cap/8, D, 8)
    for dim, (tok, x) in dims.items():
        if v.dim() == 5:
            v[:, :, tok // 8, dim, tok % 8] = x
        else:
            v[:, :, tok, dim] = x
    cache._version += 1
    got = S.sunshape_sdpa(q, cache, 0.02, mask, out_dtype=torch.float32)
    for dim, (_, x) in dims.items():
        col = got[..., dim]
        assert bool((torch.isnan(col) if dim == 41 else col == x).all()), dim
        got[..., dim] = plain[..., dim]
    assert torch.equal(got, plain)


@pytest.mark.parametrize("backend,d,t_q,buffer", [
    ("fp16", 128, 1000, 128), ("fp16", 64, 1100, 128), ("fp16", 128, 2400, 128), ("fp16", 64, 1100, 40),
    ("grouped", 128, 1000, 40)])
def test_bf16_prompts_keep_infinite_values(backend, d, t_q, buffer):
    """Infinite values of tokens that a row sees (of the first alone, with
    probability 1, in row 0): infinite in their dims of the output, the other
    dims as without them.  (Of tokens that it does not see: 0 * infinity, as
    in the two-pass path.)"""
    cache = _masked_cache(backend, 4, torch.bfloat16, d, 2, 1, t_q, buffer)
    g = torch.Generator(device="cuda").manual_seed(1)
    q = torch.randn((1, 8, t_q, d), generator=g, device="cuda").bfloat16()
    before = S.get_kernel_stats()
    plain = S.sunshape_sdpa(q, cache, 0.02, "causal")
    assert any(n > before.get(k, 0) for k, n in S.get_kernel_stats().items() if "prefill" in k)
    dims = {7: (t_q - 1, torch.inf)}  # (buffered, where there is a buffer)
    store, base = (cache._values, 0) if buffer == 128 else \
        (cache._value_buffer, cache.compressed_offset - cache._buf_start)
    if buffer == 128:
        dims.update({20: (t_q // 2, -torch.inf), 40: (0, torch.inf)})
    for dim, (tok, x) in dims.items():
        store[:, :, tok - base, dim] = x
    cache._version += 1
    got = S.sunshape_sdpa(q, cache, 0.02, "causal")
    for dim, (tok, x) in dims.items():
        assert bool((got[:, :, tok:, dim] == x).all()), dim
        got[..., dim] = plain[..., dim]
    assert torch.equal(got, plain)


@pytest.mark.parametrize("backend,bits,dtype,d,t_q,masked", [
    ("grouped", 2, torch.bfloat16, 64, 1, True), ("grouped", 4, torch.float16, 128, 3, True),
    ("fp16", 0, torch.float16, 128, 1, True), ("fp16", 0, torch.float16, 128, 40, False),
    ("grouped", 2, torch.float16, 128, 40, False)])
def test_hybrids_keep_infinite_values(backend, bits, dtype, d, t_q, masked):
    """An infinite value of a buffered token (the buffer's last, and one
    inside) or, as fp16, of a stored one: infinite in its dim for the rows that
    see it, the other dims as without it."""
    t_kv, buffer = 777, 20
    cache = _masked_cache(backend, bits, dtype, d, 2, 1, t_kv, buffer)
    g = torch.Generator(device="cuda").manual_seed(1)
    q = torch.randn((1, 8, t_q, d), generator=g, device="cuda").to(dtype)
    mask = torch.arange(t_kv, device="cuda") != 9 if masked else "causal"
    plain = S.sunshape_sdpa(q, cache, 0.02, mask)
    first = t_kv if masked else t_kv - t_q  # the first key that row 0 does not see, less one
    toks = {7: t_kv - 1, 20: t_kv - 9}
    if backend == "fp16":
        toks[40] = 400
    for dim, tok in toks.items():
        if tok >= cache.compressed_offset:
            cache._value_buffer[:, :, cache._buf_start + tok - cache.compressed_offset, dim] = torch.inf
        else:
            cache._values_il8[:, :, tok // 8, dim, tok % 8] = torch.inf
    cache._version += 1
    got = S.sunshape_sdpa(q, cache, 0.02, mask)
    for dim, tok in toks.items():
        assert bool((got[:, :, max(tok - first, 0):, dim] == torch.inf).all()), dim
        got[..., dim] = plain[..., dim]
    assert torch.equal(got, plain)
