"""GPU parity of kernels a dispatch rule chooses, at the sizes where each can
go wrong: edges of its tiles and chunks, remainders, alignment.

Bar: max |gpu - oracle| <= 1e-3 * max |oracle| (fp32 outputs, float64 oracle),
as for every attention kernel here."""

import numpy as np
import pytest
import torch

from oracle import sunshape_oracle as O
from sunshape_mlx_amd import _hip
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
