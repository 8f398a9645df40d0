"""The work a program has this package do, as cases that can be timed and checked.

Every case goes through the public entry points (``create_kv_cache``,
``update_and_fetch``, ``sunshape_sdpa``, ``trim``, ``codec.quantize`` /
``dequantize``) and stands for one attention layer of a model:

``step``     one decode step: the new tokens' keys and values enter the cache,
             their queries attend over it, and the tokens are trimmed again,
             as a rejected draft or a sampled-and-discarded branch is (so the
             pass can be repeated).  ``n_new`` > 1 is a speculative
             verification (causal rows).  ``mask`` is the padding mask of a
             left-padded batch.
``prefill``  a prompt, or a chunk of one: with ``past`` 0 a new request (a new
             cache, the whole prompt encoded and attended causally); with
             ``past`` > 0 the next chunk of a long prompt.
``codec``    bulk encode of keys to block-VQ indices and their decode.

Sizes are those of the package's own benchmark and tests (32 query / 8 KV
heads of 128 dims; 4096, 32768 and 131072 tokens; batches of 1 to 16) and odd
ones around them.
"""

import math

import numpy as np
import torch

import __graft_entry__

S = __graft_entry__.load_package()

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}
BLOCK = 8          # key dims per codebook block
CENTROIDS = 256
VALUE_BLOCK = 4    # value dims per codebook block of SunShape-coded values
HEAVY = (2, 5, 9, 14)  # heavy blocks of the mixed-precision codec, kept in fp16
VALUE_SEED = 43    # the caches' default rotation seed of TurboQuant values
CHUNK = 1 << 25    # elements of keys generated at a time


def _step(name, backend, dtype, b, hq, hkv, d, t, bits=0, n_new=1, mask="none"):
    c = dict(kind="step", backend=backend, dtype=dtype, bits=bits, b=b, hq=hq, hkv=hkv, d=d, t=t,
             n_new=n_new, mask=mask)
    return dict(c, name=name) if name else c


def _prefill(name, backend, dtype, b, hq, hkv, d, past, t, bits=0):
    c = dict(kind="prefill", backend=backend, dtype=dtype, bits=bits, b=b, hq=hq, hkv=hkv, d=d,
             past=past, t=t)
    return dict(c, name=name) if name else c


def listed():
    return [
        # an interactive chat early in its context: latency and launches
        _step("step_fp16_t509", "fp16", "fp16", 1, 32, 8, 128, 509),
        # the headline workload: one long-context stream, fp16 values
        _step("step_fp16_t32768", "fp16", "fp16", 1, 32, 8, 128, 32768),
        # a small server batch of a bfloat16 model
        _step("step_bf16_b4_t8003", "fp16", "bf16", 4, 32, 8, 128, 8003),
        # a left-padded batch with its padding mask
        _step("step_mask_b8_t4099", "fp16", "fp16", 8, 32, 8, 128, 4099, mask="bool"),
        # hybrid cache with 2-bit grouped values, a server batch
        _step("step_grouped2_b8_t32768", "grouped", "fp16", 8, 32, 8, 128, 32768, bits=2),
        # 4-bit grouped values, a model with 64-dim heads
        _step("step_grouped4_d64_b2_t6001", "grouped", "fp16", 2, 16, 4, 64, 6001, bits=4),
        # TurboQuant values at 4 bits
        _step("step_turbo4_b4_t16001", "turboquant", "fp16", 4, 32, 8, 128, 16001, bits=4),
        # one of the 28 layers of the long-context server: mixed-precision
        # keys, SunShape-coded values
        _step("step_sunshape_b16_t131072", "sunshape", "fp16", 16, 32, 8, 128, 131072, bits=8),
        # a whole prompt of an fp16 model
        _prefill("prefill_fp16_t4096", "fp16", "fp16", 1, 32, 8, 128, 0, 4096),
        # an odd-length prompt of a bfloat16 model
        _prefill("prefill_bf16_t2041", "fp16", "bf16", 1, 32, 8, 128, 0, 2041),
        # a chunk of a long prompt against a 2-bit hybrid cache
        _prefill("prefill_chunk_grouped2_t512", "grouped", "fp16", 2, 32, 8, 128, 8192, 512,
                 bits=2),
        # the encoder's bulk work: 8 heads x 8192 keys
        dict(name="codec_65536", kind="codec", dtype="fp16", d=128, n=65536),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    hq, hkv = rng.choice([(32, 8), (32, 8), (32, 8), (8, 2), (16, 2), (16, 16), (28, 4)])
    d = rng.choice([128, 128, 128, 64])
    backend, bits = rng.choice([("fp16", 0), ("fp16", 0), ("fp16", 0), ("grouped", 2),
                                ("grouped", 3), ("grouped", 4), ("turboquant", 2),
                                ("turboquant", 3), ("turboquant", 4), ("sunshape", 8)])
    dtype = rng.choice(["fp16", "fp16", "bf16"])
    kind = rng.choice(["step"] * 6 + ["prefill"] * 3 + ["codec"])
    if kind == "codec":
        return dict(kind="codec", dtype=dtype, d=d, n=_log_int(rng, 64, 131072))
    if kind == "step":
        b = rng.choice([1, 1, 2, 4, 8, 16])
        # tokens over all sequences at most 2^20, a sequence at most 2^17
        t = _log_int(rng, 200, min(131072, (1 << 20) // b))
        return _step(None, backend, dtype, b, hq, hkv, d, t, bits=bits,
                     n_new=rng.choice([1, 1, 1, 1, 4]),
                     mask=rng.choice(["none"] * 6 + ["bool", "add"]))
    b = rng.choice([1, 1, 2])
    t = _log_int(rng, 64, 4096 // b)
    past = rng.choice([0, 0, _log_int(rng, 200, 8192)])
    return _prefill(None, backend, dtype, b, hq, hkv, d, past, t, bits=bits)


# ------------------------------------------------------------------- inputs


def _gen(seed, salt):
    return torch.Generator(device="cuda").manual_seed((int(seed) * 1000003 + salt) % (1 << 62))


def _codec_arrays(d, seed):
    """Per-dim key scales in [0.5, 4] and, as k-means starts from and stays
    near, centroids that are blocks of calibration keys: the key codebook,
    its permutation, the value codebook and its permutation."""
    g = _gen(seed, 1)
    s = 0.5 + 3.5 * torch.rand((d,), generator=g, device="cuda")
    perm = torch.randperm(d, generator=g, device="cuda")
    cal = (torch.randn((CENTROIDS, d), generator=g, device="cuda") * s)[:, perm]
    cents = cal.reshape(CENTROIDS, d // BLOCK, BLOCK).permute(1, 0, 2).contiguous()
    vperm = torch.randperm(d, generator=g, device="cuda")
    vcal = torch.randn((CENTROIDS, d), generator=g, device="cuda")
    vcents = vcal.reshape(CENTROIDS, d // VALUE_BLOCK, VALUE_BLOCK).permute(1, 0, 2).contiguous()
    return s, perm, cents, vperm, vcents


def _kv(c, seed, salt, n, s):
    """(keys, values) of n tokens a sequence: anisotropic keys, unit values."""
    g = _gen(seed, salt)
    shape = (c["b"], c["hkv"], n, c["d"])
    dt = DTYPES[c["dtype"]]
    k = (torch.randn(shape, generator=g, device="cuda") * s).to(dt)
    v = torch.randn(shape, generator=g, device="cuda").to(dt)
    return k, v


def _chunks(c, seed, total, s):
    per = max(256, CHUNK // (c["b"] * c["hkv"] * c["d"]) // 256 * 256)
    t0, i = 0, 0
    while t0 < total:
        n = min(per, total - t0)
        yield _kv(c, seed, 100 + i, n, s)
        t0, i = t0 + n, i + 1


def _queries(c, seed, n):
    return torch.randn((c["b"], c["hq"], n, c["d"]), generator=_gen(seed, 2),
                       device="cuda").to(DTYPES[c["dtype"]])


def _mask(c, seed):
    """The padding mask of a left-padded batch: up to half of a sequence's
    keys are padding, never the new ones; None without one."""
    if c.get("mask", "none") == "none":
        return None
    t = c["t"] + c["n_new"]
    g = _gen(seed, 3)
    pad = (torch.rand((c["b"],), generator=g, device="cuda") * (c["t"] // 2)).long()
    pos = torch.arange(t, device="cuda")
    keep = pos[None, :] >= pad[:, None]
    if c["n_new"] > 1:
        qpos = torch.arange(c["t"], t, device="cuda")
        keep = keep[:, None, :] & (pos[None, None, :] <= qpos[None, :, None])
    else:
        keep = keep[:, None, :]
    keep = keep[:, None]  # (B, 1, n_new, T)
    if c["mask"] == "bool":
        return keep
    low = torch.finfo(DTYPES[c["dtype"]]).min
    return torch.where(keep, 0.0, low).to(DTYPES[c["dtype"]])


def _heavy(c):
    return c["backend"] == "sunshape" and c["d"] == 128


def _new_cache(c, codec, vcodec):
    kw = {}
    if c["backend"] == "grouped":
        kw = dict(value_bits=c["bits"], value_group_size=min(64, c["d"]),
                  value_scale_dtype=torch.float16)
    elif c["backend"] == "turboquant":
        kw = dict(value_bits=c["bits"], value_seed=VALUE_SEED)
    elif c["backend"] == "sunshape":
        kw = dict(value_bits=c["bits"], value_codec=vcodec)
    total = c.get("past", 0) + c["t"] + c.get("n_new", 0)
    return S.create_kv_cache(codec, n_kv_heads=c["hkv"], dtype=DTYPES[c["dtype"]],
                             value_backend=c["backend"], max_tokens=total + 128, **kw)


def prepare(case, seed):
    c = case
    if c["kind"] == "codec":
        s, perm, cents, _, _ = _codec_arrays(c["d"], seed)
        codec = S.SunShapeBlockCodec(c["d"], device="cuda").load_state_dict(
            {"centroids": cents, "permutation": perm})
        k, _ = _kv(dict(c, b=1, hkv=1), seed, 100, c["n"], s)
        return {"case": c, "codec": codec, "keys": k.reshape(c["n"], c["d"])}
    s, perm, cents, vperm, vcents = _codec_arrays(c["d"], seed)
    if _heavy(c):
        hb = torch.zeros(c["d"] // BLOCK, dtype=torch.bool, device="cuda")
        hb[list(HEAVY)] = True
        codec = S.SunShapeBlockCodec(c["d"], device="cuda", mode="profileperm_mixed_precision",
                                     heavy_fp16=True)
        codec.load_state_dict({"centroids": cents, "permutation": perm,
                               "mixed_high_precision_blocks": hb})
    else:
        codec = S.SunShapeBlockCodec(c["d"], device="cuda").load_state_dict(
            {"centroids": cents, "permutation": perm})
    vcodec = None
    if c["backend"] == "sunshape":
        vcodec = S.SunShapeBlockCodec(c["d"], block_dim=VALUE_BLOCK, device="cuda")
        vcodec.load_state_dict({"centroids": vcents, "permutation": vperm})
    n = c["n_new"] if c["kind"] == "step" else c["t"]
    held = c["t"] if c["kind"] == "step" else c["past"]
    state = {"case": c, "codec": codec, "vcodec": vcodec, "n": n,
             "q": _queries(c, seed, n), "scale": 1.0 / math.sqrt(c["d"]), "cache": None}
    state["k"], state["v"] = _kv(c, seed, 4, n, s)
    mask = _mask(c, seed)
    state["mask"] = mask if mask is not None else ("causal" if n > 1 else None)
    if held:
        cache = _new_cache(c, codec, vcodec)
        if c["kind"] == "step":
            # the tokens of an earlier step are in and out again, as between
            # two passes
            for k, v in _chunks(c, seed, held, s):
                cache.update_and_fetch(k, v)
            cache.update_and_fetch(state["k"], state["v"])
            cache.trim(n)
        else:
            for k, v in _chunks(c, seed, held, s):
                cache.update_and_fetch(k, v)
        state["cache"] = cache
    return state


def run(state):
    if state["case"]["kind"] == "codec":
        codec = state["codec"]
        quantized = codec.quantize(state["keys"])
        return {"indices": quantized.indices, "keys": codec.dequantize(quantized)}
    cache = state["cache"]
    if cache is None:  # a new request
        cache = _new_cache(state["case"], state["codec"], state["vcodec"])
        cache.update_and_fetch(state["k"], state["v"])
        out = S.sunshape_sdpa(state["q"], cache, state["scale"], state["mask"])
        return {"out": out, "indices": cache.key_indices}
    cache.update_and_fetch(state["k"], state["v"])
    out = S.sunshape_sdpa(state["q"], cache, state["scale"], state["mask"])
    cache.trim(state["n"])
    return out


# ------------------------------------------------------------ what it takes


def _token_bytes(c):
    """Stored bytes of one compressed token of one KV head."""
    d, nb = c["d"], c["d"] // BLOCK
    if c["backend"] == "fp16":
        return nb + 2 * d
    if c["backend"] == "grouped":
        return nb + d * c["bits"] // 8 + 4 * (d // min(64, d))
    if c["backend"] == "turboquant":
        return nb + d * c["bits"] // 8 + 4
    heavy = 2 * BLOCK * len(HEAVY) if _heavy(c) else 0
    return nb + heavy + d // VALUE_BLOCK


def work(case):
    c = case
    if c["kind"] == "codec":
        n, d = c["n"], c["d"]
        return {"bytes": n * (2 * d + 2 * (d // BLOCK) + 4 * d),
                "flops": 2 * n * d * CENTROIDS}
    d, rows = c["d"], c["b"] * c["hkv"]
    n = c["n_new"] if c["kind"] == "step" else c["t"]
    past = c["t"] if c["kind"] == "step" else c["past"]
    raw = 0 if c["backend"] == "fp16" else min(past, 128)  # tokens of the hybrid buffer
    read = rows * ((past - raw) * _token_bytes(c) + raw * 4 * d)
    new = rows * n * (4 * d + _token_bytes(c))             # read in, stored
    qo = c["b"] * c["hq"] * n * d * 4
    pairs = c["b"] * c["hq"] * (n * past + n * (n + 1) // 2)
    return {"bytes": read + new + qo, "flops": 4 * pairs * d + 2 * rows * n * d * CENTROIDS}


def tolerance(case):
    c = case
    if c["kind"] == "codec":
        # indices are the exact nearest centroid, keys their float32 centroids
        return "exact"
    # measured against exact(): 2.0e-4 to 3.1e-4 with fp16 outputs, 1.6e-3 to
    # 1.7e-3 with bf16 ones (the output's own rounding); four times that
    return {"rel": 1.3e-3 if c["dtype"] == "fp16" else 7e-3}


# ------------------------------------------------------------ in 64 bits


def _encode64(x, cents):
    """Indices of the nearest centroid of each block of (..., d) rows."""
    nb, nc, bd = cents.shape
    flat = x.reshape(-1, nb, bd)
    out = torch.empty((flat.shape[0], nb), dtype=torch.int64, device=x.device)
    c64 = cents.double()
    c2 = c64.square().sum(-1)
    for i in range(0, flat.shape[0], 1 << 16):
        f = flat[i:i + (1 << 16)].double()
        for b in range(nb):
            out[i:i + (1 << 16), b] = torch.addmm(c2[b], f[:, b], c64[b].t(), alpha=-2.0).argmin(-1)
    return out.reshape(*x.shape[:-1], nb)


def _decode64(idx, cents, perm):
    """(..., nb) indices -> float64 rows in the original basis."""
    nb = cents.shape[0]
    rows = cents.double()[torch.arange(nb, device=idx.device), idx].flatten(-2)
    out = torch.empty_like(rows)
    out[..., perm] = rows
    return out


def _values64(c, v, vperm, vcents):
    """What the cache's value backend makes of values v."""
    if c["backend"] == "fp16":
        return v.double()
    if c["backend"] == "grouped":
        # codes and their float16 scale and zero as the format defines them
        # (float32 steps), then 64 bits
        top = (1 << c["bits"]) - 1
        g = v.float().unflatten(-1, (-1, min(64, c["d"])))
        lo, hi = g.amin(-1, keepdim=True), g.amax(-1, keepdim=True)
        scale = ((hi - lo) / torch.tensor(float(top), device=v.device)).clamp(min=1e-8)
        code = torch.round((g - lo) / scale).clamp(0, top)
        out = (code.double() * scale.half().double() + lo.half().double()).flatten(-2)
    elif c["backend"] == "turboquant":
        gauss = np.random.default_rng(VALUE_SEED).standard_normal((c["d"], c["d"]))
        q, r = np.linalg.qr(gauss)
        rot = (q * np.sign(np.diag(r))[None, :]).astype(np.float32)
        rot = torch.from_numpy(rot).to(v.device).double()
        levels, bounds = S.value_codecs.lloyd_max_gaussian(c["bits"])  # the format's tables
        sc = 1.0 / math.sqrt(c["d"])
        lv = torch.tensor([x * sc for x in levels], dtype=torch.float32, device=v.device).double()
        bd = torch.tensor([x * sc for x in bounds], dtype=torch.float32, device=v.device).double()
        norm = v.double().norm(dim=-1, keepdim=True)
        unit = v.double() / norm.clamp(min=1e-8) @ rot.t()
        code = torch.bucketize(unit, bd)
        out = (lv[code] @ rot) * norm
    else:
        out = _decode64(_encode64(v[..., vperm], vcents), vcents, vperm)
    if c["dtype"] == "bf16":  # a bfloat16 cache holds dequantised values in its own type
        out = out.float().bfloat16().double()
    return out


def exact(case, seed):
    c = case
    if c["kind"] == "codec":
        st = prepare(c, seed)
        _, perm, cents, _, _ = _codec_arrays(c["d"], seed)
        idx = _encode64(st["keys"][:, perm], cents)
        return {"indices": None, "keys": _decode64(idx, cents, perm)}
    s, perm, cents, vperm, vcents = _codec_arrays(c["d"], seed)
    n = c["n_new"] if c["kind"] == "step" else c["t"]
    held = c["t"] if c["kind"] == "step" else c["past"]
    if c["b"] * c["hkv"] * (held + n) > (1 << 23):
        return None
    parts = list(_chunks(c, seed, held, s)) + [_kv(c, seed, 4, n, s)]
    k = torch.cat([p[0] for p in parts], dim=2)
    v = torch.cat([p[1] for p in parts], dim=2)
    total = held + n
    hybrid = c["backend"] != "fp16"
    comp = max(0, total - 128) if hybrid else total  # tokens in compressed form
    kx = torch.empty(k.shape, dtype=torch.float64, device="cuda")
    vx = torch.empty_like(kx)
    idx = torch.zeros((*k.shape[:3], c["d"] // BLOCK), dtype=torch.int64, device="cuda")
    for b in range(c["b"]):
        for h in range(c["hkv"]):
            idx[b, h, :comp] = _encode64(k[b, h, :comp][:, perm], cents)
            kx[b, h, :comp] = _decode64(idx[b, h, :comp], cents, perm)
            if _heavy(c):
                dims = torch.tensor([x * BLOCK + j for x in HEAVY for j in range(BLOCK)],
                                    device="cuda")
                od = perm[dims]
                kx[b, h, :comp, od] = k[b, h, :comp][:, od].to(torch.float16).double()
            kx[b, h, comp:] = k[b, h, comp:].double()
            vx[b, h, :comp] = _values64(c, v[b, h, :comp], vperm, vcents)
            vx[b, h, comp:] = v[b, h, comp:].double()
    q = _queries(c, seed, n)
    qs = (q * (1.0 / math.sqrt(c["d"]))).double()  # scaled in the query's type
    mask = _mask(c, seed)
    pos = torch.arange(total, device="cuda")
    qpos = torch.arange(held, total, device="cuda")
    out = torch.empty(q.shape, dtype=torch.float64, device="cuda")
    rep = c["hq"] // c["hkv"]
    for b in range(c["b"]):
        for h in range(c["hq"]):
            kv = h // rep
            sc = qs[b, h] @ kx[b, kv].t()
            if mask is None:
                sc = sc.masked_fill(pos[None, :] > qpos[:, None], -math.inf)
            elif mask.dtype == torch.bool:
                sc = sc.masked_fill(~mask[b, 0], -math.inf)
            else:
                sc = sc + mask[b, 0].double()
            out[b, h] = torch.softmax(sc, dim=-1) @ vx[b, kv]
    if c["kind"] == "prefill" and c["past"] == 0:
        return {"out": out, "indices": None}
    return out
