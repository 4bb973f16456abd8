"""Performance cases: the calls that a program using this package makes on the GPU, over the sizes it makes them at.

A program that serves a model from the packed cache decodes (one attention call per layer and token, over packed
pages and a recent window), commits (a 128-token codec page encoded every 128 tokens, a whole prompt's pages at
once after prefill) and prefills (the attention of a prompt, or of a prompt chunk over committed pages).  The
recipes differ in the key codec: k2b (the default; on its own page or, off the recipe's geometry, on the general
page), RTN and spectral.

Decode inputs are pages built here from codes of the distributions the codecs produce, in the documented page
formats (include/bmx_k2b.h, bmx_rtn.h, bmx_spectral.h), so that `exact` knows every code.
"""

from __future__ import annotations

import math
from types import SimpleNamespace

import torch

from bmx_amd import k2b, prefill, rtn, spectral
from bmx_amd.cache import PackedStreamingLayer
from bmx_amd.specs import spec_pair

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}
LEVELS = (-1.5194618701934814, -0.46033763885498047, 0.44421979784965515, 1.5017313957214355)  # 2-bit Lloyd levels
PT = 16   # tokens of a page


# ------------------------------------------------------------------ the cases


def listed():
    dec = dict(batch=1, h_kv=8, G=4, head_dim=128, group=64, k_bits=3, table=False, new_row=False, theta=500000.0)
    return [
        # one token's attention of four layers of an 8B model at a long context: the package's headline case
        dict(dec, name="k2b_decode_64k", kind="decode", layers=4, packed=65408, window=128, rank=32, dtype="fp16"),
        # a 36-layer model streaming at about 8k tokens in bf16: the new token's row goes in with the call
        dict(dec, name="k2b_decode_8k_step", kind="decode", layers=36, packed=8576, window=161, rank=16,
             dtype="bf16", new_row=True, theta=1000000.0),
        # the first tokens after a short prompt: one layer's call, all latency
        dict(dec, name="k2b_decode_short", kind="decode", layers=1, packed=256, window=60, rank=16, dtype="fp16"),
        # a serving batch: ragged lengths, pages anywhere in the pool
        dict(dec, name="k2b_decode_batch16", kind="decode", layers=2, batch=16, packed=16384, window=128, rank=32,
             dtype="fp16", table=True),
        # a model with head_dim 64 (the general page), one token's attention of four layers
        dict(dec, name="general_decode_32k", kind="decode", layers=4, packed=32640, window=128, rank=16, head_dim=64,
             group=32, dtype="fp16"),
        # the RTN recipe, 4-bit keys and values, four layers
        dict(name="rtn_decode_32k", kind="rtn_decode", layers=4, h_kv=8, G=4, packed=32640, window=128, k_bits=4,
             v_bits=4, k_group=32, v_group=32, channel=False, dtype="fp16"),
        # the spectral recipe at 2.5 bits, one layer's call
        dict(name="spectral_decode_32k", kind="spectral_decode", h_kv=8, G=4, packed=32640, window=128, budget=2.5,
             v_codec="full", dtype="fp16"),
        # a decoding program's commit: one codec page, every 128 tokens and layer
        dict(name="k2b_commit_page", kind="k2b_append", h_kv=8, tokens=128, rank=32, head_dim=128, group=64, k_bits=3,
             dtype="fp16", first=False),
        # a prompt's pages after its prefill
        dict(name="k2b_commit_prompt_8k", kind="k2b_append", h_kv=8, tokens=8064, rank=16, head_dim=128, group=64,
             k_bits=3, dtype="bf16", first=True),
        # the same for spectral keys, a prompt of 2k tokens
        dict(name="spectral_commit_2k", kind="spectral_append", h_kv=8, tokens=1920, budget=2.5, v_codec="full",
             dtype="fp16"),
        # the second chunk of a prompt: 512 queries over 8192 committed and windowed tokens and their own
        dict(name="cached_prefill_8k", kind="cached_prefill", h_kv=8, G=4, context=8192, queries=512, rank=32,
             window=128, dtype="fp16"),
        # a prompt's own attention
        dict(name="prefill_4k", kind="prefill", h_kv=8, G=4, queries=4096, keys=4096, causal=True, dtype="bf16"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "batch", "general", "rtn_decode", "spectral_decode", "k2b_append",
                       "spectral_append", "cached_prefill", "prefill"])
    h_kv, G, dtype = rng.choice([2, 4, 8, 8]), rng.choice([1, 2, 4, 4, 7, 8]), rng.choice(["fp16", "bf16"])
    window = rng.randint(1, 255)
    if kind in ("decode", "batch", "general"):
        c = dict(kind="decode", h_kv=h_kv, G=G, dtype=dtype, window=window, rank=rng.choice([16, 32]), head_dim=128,
                 group=64, k_bits=3, table=False, batch=1, new_row=rng.random() < 0.5,
                 theta=rng.choice([10000.0, 500000.0, 1000000.0]))
        pages = _log_int(rng, 1, 511)
        if kind == "batch":
            c.update(batch=rng.randint(2, 16), table=True, new_row=False)
            pages = _log_int(rng, 4, 128)
        if kind == "general":
            c.update(head_dim=rng.choice([32, 64, 64, 128]), group=rng.choice([16, 32, 64, 128]),
                     k_bits=rng.choice([2, 3, 4]), rank=rng.choice([16, 32, 64]))
            if c["head_dim"] == 128 and c["group"] == 64 and c["k_bits"] == 3 and c["rank"] < 64:
                c["k_bits"] = 4
            pages = _log_int(rng, 1, 255)
        c["packed"] = 128 * pages
        c["layers"] = max(1, min(rng.randint(1, 8), 262144 // (c["packed"] * c["batch"])))
        return c
    if kind == "rtn_decode":
        packed = 128 * _log_int(rng, 1, 255)
        return dict(kind=kind, layers=max(1, min(rng.randint(1, 8), 131072 // packed)), h_kv=h_kv, G=G, packed=packed,
                    window=window, k_bits=rng.choice([2, 3, 4]), v_bits=rng.choice([2, 4]),
                    k_group=rng.choice([32, 64, 128]), v_group=rng.choice([32, 64, 128]),
                    channel=rng.random() < 0.5, dtype=dtype)
    if kind == "spectral_decode":
        return dict(kind=kind, h_kv=rng.choice([2, 4, 8]), G=G, packed=128 * _log_int(rng, 1, 255), window=window,
                    budget=rng.choice([2.0, 2.5, 3.0]), v_codec=rng.choice(["full", "perhead"]), dtype=dtype)
    if kind == "k2b_append":
        general = rng.random() < 0.3
        return dict(kind=kind, h_kv=h_kv, tokens=128 * _log_int(rng, 1, 63), rank=rng.choice([16, 32]),
                    head_dim=64 if general else 128, group=rng.choice([32, 64]) if general else 64, k_bits=3,
                    dtype=rng.choice(["fp16", "bf16", "fp32"]), first=rng.random() < 0.5)
    if kind == "spectral_append":
        return dict(kind=kind, h_kv=rng.choice([2, 4, 8]), tokens=128 * _log_int(rng, 1, 15),
                    budget=rng.choice([2.0, 2.5, 3.0]), v_codec=rng.choice(["full", "perhead"]), dtype=dtype)
    if kind == "cached_prefill":
        return dict(kind=kind, h_kv=h_kv, G=G, context=_log_int(rng, 200, 8192), queries=_log_int(rng, 2, 512),
                    rank=rng.choice([16, 32]), window=rng.choice([32, 128]), dtype=dtype)
    keys = _log_int(rng, 64, 4096)
    return dict(kind="prefill", h_kv=h_kv, G=rng.choice([1, 2, 4]), queries=rng.choice([keys, rng.randint(1, keys)]),
                keys=keys, causal=rng.random() < 0.8, dtype=dtype)


# ------------------------------------------------------------------ inputs


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(g, *shape, dtype=torch.float32):
    return torch.randn(*shape, generator=g, device="cuda", dtype=dtype)


def _inv_freq(theta, d):
    return 1.0 / (theta ** (torch.arange(0, d, 2, dtype=torch.int64).to(torch.float) / d))


def _signs(n, seed=0):
    """The +-1 signs of the seeded randomized Hadamard."""
    return torch.randint(0, 2, (n,), generator=torch.Generator().manual_seed(seed)) * 2 - 1


def _consts(theta, d):
    words = [0] * 4
    for c, s in enumerate(_signs(d).tolist()):
        words[c // 32] |= (1 << (c % 32)) if s < 0 else 0
    return k2b.CodecConsts(LEVELS, tuple(words), tuple(_inv_freq(theta, d).tolist()))


def _orthonormal(g, n, r):
    """(n, r) orthonormal columns, fp32 on the device."""
    return torch.linalg.qr(_randn(g, n, r).double().cpu())[0].float().cuda().contiguous()


def _spread(r, total):
    """Standard deviations of r directions, falling off as i^-0.35, with squares that sum to `total`."""
    s = torch.arange(1, r + 1, device="cuda", dtype=torch.float32) ** -0.35
    return s * math.sqrt(total / float((s * s).sum()))


def _rope(x, pos, inv_freq, half_tables=False):
    """x (..., n, d) rotated at pos (n,): angle fl32(inv_freq * pos), cos / sin in x's precision (or through fp16)."""
    ang = (pos.to(torch.float32)[:, None] * inv_freq.to(x.device)[None, :]).to(x.dtype)
    ang = torch.cat((ang, ang), -1)
    cos, sin = ang.cos(), ang.sin()
    if half_tables:   # the prefill's tables: fp32 cos / sin, then fp16
        cos, sin = ang.float().cos().half().to(x.dtype), ang.float().sin().half().to(x.dtype)
    d = x.shape[-1]
    return x * cos + torch.cat((-x[..., d // 2:], x[..., : d // 2]), -1) * sin


def _value_codes(g, h, T, d):
    """2-bit codes of Gaussian channels (h, T, d) int32 and fp16 norms (h, T)."""
    mids = torch.tensor([(a + b) / 2 for a, b in zip(LEVELS, LEVELS[1:])], device="cuda")
    idx = torch.bucketize(_randn(g, h, T, d), mids).to(torch.int32)
    norm = (math.sqrt(d) * (0.7 + 0.6 * torch.rand(h, T, generator=g, device="cuda"))).half()
    return idx, norm


def _k2b_fields(g, case, T):
    """Codes of T tokens: low-rank coefficients, residual codes and scales, value codes and norms."""
    h, d, R, grp, b = case["h_kv"], case["head_dim"], case["rank"], case["group"], case["k_bits"]
    qmax = (1 << (b - 1)) - 1
    us = (_randn(g, T, R) * _spread(R, h * d / 2)).half()
    step = 2.4 / max(qmax, 1)
    res = (_randn(g, h, T, d) / step).round().clamp(-qmax - 1, qmax).to(torch.int32)
    scale = (0.3 * step * (0.8 + 0.4 * torch.rand(h, T // grp, d, generator=g, device="cuda"))).half()
    vidx, vnorm = _value_codes(g, h, T, d)
    return dict(us=us, res=res, scale=scale, vidx=vidx, vnorm=vnorm)


def _bytes(t):
    return t.contiguous().view(torch.uint8)


def _value_words(vidx):
    """VCODE of the recipe's page: (P, h, 512) bytes of codes (h, T, 128)."""
    h, T, _ = vidx.shape
    v = vidx.view(h, T // PT, 4, 4, 8, 16).permute(1, 0, 2, 5, 4, 3)                    # P h q m b t
    sh = torch.tensor([0, 2, 4, 6], device="cuda", dtype=torch.int32)
    return (v << sh).sum(-1, dtype=torch.int32).to(torch.uint8).reshape(T // PT, h, 512)


def _k2b_pages(f, case):
    h, d, R, grp, b = case["h_kv"], case["head_dim"], case["rank"], case["group"], case["k_bits"]
    T = f["us"].shape[0]
    P = T // PT
    if d == 128 and grp == 64 and b == 3 and R in (16, 32):
        us = f["us"].view(P, PT, 4, R // 4).permute(0, 2, 1, 3).reshape(P, -1)
        sc = f["scale"].view(h, T // 64, 2, 64).permute(1, 0, 3, 2).reshape(P, -1)
        c = (f["res"] + 4).view(h, P, PT, 2, 4, 4, 4).permute(1, 0, 5, 2, 3, 4, 6).reshape(P, h, 4, PT, 2, 16)
        lo, hi = c[..., 0, :], c[..., 1, :]
        words = []
        for k in range(3):
            w = (((lo[..., 15] >> k) & 1) << 15) | (((hi[..., 15] >> k) & 1) << 31)
            for p in range(5):
                w = w | (lo[..., 5 * k + p] << (3 * p)) | (hi[..., 5 * k + p] << (16 + 3 * p))
            words.append(w)
        kres = torch.stack(words, -1).to(torch.int32).reshape(P, -1)
        parts = [us, f["vnorm"].view(h, P, PT).permute(1, 0, 2).reshape(P, -1), sc, kres,
                 _value_words(f["vidx"]).reshape(P, -1)]
        return torch.cat([_bytes(x) for x in parts], 1).contiguous()
    res = (f["res"] + (1 << (b - 1))).view(h, P, PT, d // 2, 2).permute(1, 0, 2, 3, 4)
    vv = f["vidx"].view(h, P, 4, 4, d).permute(1, 0, 2, 4, 3)
    sh = torch.tensor([0, 2, 4, 6], device="cuda", dtype=torch.int32)
    parts = [f["us"].view(P, -1), f["vnorm"].view(h, P, PT).permute(1, 0, 2).reshape(P, -1),
             f["scale"].permute(1, 0, 2).reshape(P, -1),
             (res[..., 0] | (res[..., 1] << 4)).to(torch.uint8).reshape(P, -1),
             (vv << sh).sum(-1, dtype=torch.int32).to(torch.uint8).reshape(P, -1)]
    parts = [_bytes(x) for x in parts]
    parts = [torch.cat((x, x.new_zeros(P, -x.shape[1] % 16)), 1) if x.shape[1] % 16 else x for x in parts]
    return torch.cat(parts, 1).contiguous()


def _queries(g, case, *shape):
    return (1.5 * _randn(g, *shape)).to(DTYPES[case["dtype"]])


def _window(g, case, *shape):
    return (0.7 * _randn(g, *shape)).to(DTYPES[case["dtype"]]), _randn(g, *shape).to(DTYPES[case["dtype"]])


def _lengths(case, seed):
    """Committed tokens of each sequence: `packed`, or for a batch a quarter of it and up."""
    B, top = case["batch"], case["packed"] // 128
    if B == 1:
        return [case["packed"]]
    r = torch.Generator().manual_seed(seed)
    return [128 * int(x) for x in torch.randint(max(1, top // 4), top + 1, (B,), generator=r)]


def _decode_layers(case, seed):
    """Layer by layer: the sequences' fields, bases, queries and windows."""
    g = _gen(seed)
    B, h, G, d = case["batch"], case["h_kv"], case["G"], case["head_dim"]
    for layer in range(case["layers"]):
        lens = _lengths(case, seed)
        fields = [_k2b_fields(g, case, n) for n in lens]
        basis = torch.stack([_orthonormal(g, h * d, case["rank"]) for _ in range(B)]).half()
        q = _queries(g, case, B, h, G, d)
        k, v = _window(g, case, B, h, case["window"], d)
        yield lens, fields, basis, q, k, v


def _prepare_decode(case, seed):
    calls = []
    consts = _consts(case["theta"], case["head_dim"])
    ws = k2b.DecodeWorkspace()
    T, order = case["window"], torch.Generator().manual_seed(seed + 1)
    for lens, fields, basis, q, k, v in _decode_layers(case, seed):
        rows = torch.cat([_k2b_pages(f, case) for f in fields])
        packed_len = torch.tensor(lens, dtype=torch.int32, device="cuda")
        top, table, pool = max(lens), None, rows
        if case["table"]:
            at = torch.randperm(rows.shape[0], generator=order)
            pool = torch.empty_like(rows)
            pool[at.cuda()] = rows
            table, first = torch.zeros(len(lens), top // PT, dtype=torch.int32), 0
            for i, n in enumerate(lens):
                table[i, : n // PT] = at[first: first + n // PT]
                first += n // PT
            table = table.cuda()
        new = None
        kw = dict(tail_len=torch.full((len(lens),), T, dtype=torch.int32, device="cuda"), tail_cap=T)
        if case["batch"] == 1:   # a cache's window: fixed buffers, the length known to the host
            cap = max(T, 160) + 32
            kb = torch.zeros(1, case["h_kv"], cap, case["head_dim"], dtype=k.dtype, device="cuda")
            vb = torch.zeros_like(kb)
            kb[:, :, :T], vb[:, :, :T] = k, v
            if case["new_row"]:
                new = (k[:, :, T - 1:].contiguous(), v[:, :, T - 1:].contiguous())
                kb[:, :, T - 1], vb[:, :, T - 1] = 0, 0
            k, v, kw = kb, vb, dict(tail_len=T, tail_cap=cap)
        plan = k2b.DecodePlan(q, pool, table, packed_len, top, basis[0] if case["batch"] == 1 else basis, consts,
                              case["head_dim"] ** -0.5, rank=case["rank"], k_tail=k, v_tail=v, workspace=ws,
                              group=case["group"], k_bits=case["k_bits"], **kw)
        calls.append((plan, q, new))
    return dict(kind="decode", calls=calls, window=T, host_len=case["batch"] == 1)


def _rtn_fields(g, case, T):
    h = case["h_kv"]

    def side(bits, sigma, scales):
        qmax = (1 << (bits - 1)) - 1
        codes = (_randn(g, h, T, 128) * max(qmax, 1) / 2.3).round().clamp(-qmax - 1, qmax).to(torch.int32)
        s = sigma * 2.3 / max(qmax, 1) * (0.7 + 0.6 * torch.rand(scales, generator=g, device="cuda"))
        return codes, s
    kshape = (h, T // case["k_group"], 128) if case["channel"] else (h, T, 128 // case["k_group"])
    kq, ks = side(case["k_bits"], 0.7, kshape)
    vq, vs = side(case["v_bits"], 1.0, (h, T, 128 // case["v_group"]))
    if not case["channel"]:
        ks = ks.half()
    return dict(kq=kq, ks=ks, vq=vq, vs=vs.half())


def _rtn_pages(f, case):
    h, T, _ = f["kq"].shape
    P = T // PT
    if case["channel"]:
        hi = f["ks"].half()
        pair = torch.stack((hi, (f["ks"] - hi.float()).half()))                          # 2 h T/gk 128
        order = torch.tensor([0, 4, 1, 5, 2, 6, 3, 7], device="cuda")
        pair = pair.view(2, h, -1, 16, 8)[..., order].reshape(2, h, -1, 128)
        ks = pair.repeat_interleave(case["k_group"] // PT, 2).permute(2, 0, 1, 3).reshape(P, -1)
    else:
        ks = f["ks"].view(h, P, PT, -1).permute(1, 0, 2, 3).reshape(P, -1)
    vs = f["vs"].view(h, P, 4, 4, -1).permute(1, 0, 2, 4, 3).reshape(P, -1)
    nib = 4 * torch.arange(8, device="cuda", dtype=torch.int32)
    kc = (f["kq"] + 8).view(h, P, PT, 4, 4, 8).permute(1, 0, 4, 2, 3, 5)                 # P h q n w j
    kc = (kc << nib).sum(-1, dtype=torch.int64)
    kc = torch.where(kc >= 1 << 31, kc - (1 << 32), kc).to(torch.int32).reshape(P, -1)
    vc = (f["vq"] + 8).view(h, P, 4, 4, 8, 16).permute(1, 0, 2, 5, 4, 3)                 # P h q c b j
    vc = (vc << nib[:4]).sum(-1, dtype=torch.int32)
    vc = torch.stack((vc & 255, vc >> 8), -1).to(torch.uint8).reshape(P, -1)
    return torch.cat([_bytes(x) for x in (ks, vs, kc, vc)], 1).contiguous()


def _rtn_layers(case, seed):
    g = _gen(seed)
    for _ in range(case["layers"]):
        f = _rtn_fields(g, case, case["packed"])
        q = _queries(g, case, 1, case["h_kv"], case["G"], 128)
        yield (f, q) + _window(g, case, 1, case["h_kv"], case["window"], 128)


def _prepare_rtn(case, seed):
    calls, T, P = [], case["window"], case["packed"]
    ws = k2b.DecodeWorkspace()
    codec = dict(k_bits=case["k_bits"], v_bits=case["v_bits"], k_group=case["k_group"], v_group=case["v_group"],
                 k_arm=rtn.CHANNEL if case["channel"] else rtn.TOKEN)
    for f, q, k, v in _rtn_layers(case, seed):
        pool = _rtn_pages(f, case)
        table = torch.arange(P // PT, dtype=torch.int32, device="cuda")[None].contiguous()
        plan = rtn.DecodePlan(q, pool, table, torch.tensor([P], dtype=torch.int32, device="cuda"), P, 128 ** -0.5,
                              k_tail=k, v_tail=v, tail_len=T, tail_cap=T, workspace=ws, **codec)
        calls.append((plan, q, None))
    return dict(kind="decode", calls=calls, window=T, host_len=True)


TIERS = (0, 2, 3, 4, 5, 6, 8)
TIER_STEP = {2: 1.0, 3: 0.59, 4: 0.34, 5: 0.19, 6: 0.104, 8: 0.031}   # quantizer step of a unit Gaussian, by bits
TIER_BITS = {2: 2, 3: 4, 4: 4, 5: 8, 6: 8, 8: 8}                      # bits a code takes in the page


def _pack(case):
    """A fitted pack's content (it comes with the model, whatever the inputs): encoder, decoder, variances, bits."""
    C = 128 * case["h_kv"]
    g = torch.Generator().manual_seed(5)
    E = torch.linalg.qr(torch.randn(C, C, generator=g, dtype=torch.float64))[0]
    w = 0.5 + torch.rand(C, generator=g, dtype=torch.float64)
    lam = torch.arange(1, C + 1, dtype=torch.float64) ** -2.0
    lam *= C / lam.sum()
    grid = torch.tensor(TIERS, dtype=torch.float64)
    lo, hi, bits = math.log(1e-12), math.log(1e6), None
    for _ in range(60):   # the smallest distortion level whose mean rate stays within the budget
        mid = (lo + hi) / 2
        rate = (0.5 * torch.log2(lam / math.exp(mid))).clamp_min(0)
        b = grid[(rate[:, None] - grid[None, :]).abs().argmin(1)]
        if float(b.mean()) <= case["budget"]:
            hi, bits = mid, b
        else:
            lo = mid
    return (w.sqrt()[:, None] * E).float(), (w.rsqrt()[:, None] * E).float(), lam.float(), bits.to(torch.int64)


_PACKS: dict = {}


def _device_pack(case):
    """(pack content, device handle): a program loads a model's packs once."""
    key = (case["h_kv"], case["budget"], case["v_codec"])
    if key not in _PACKS:
        enc, dec, lam, bits = _pack(case)
        pack = spectral.SpectralPack(enc=enc, dec=dec, lam=lam, bits=bits, budget=case["budget"])
        _PACKS.clear()
        _PACKS[key] = ((enc, dec, lam, bits), spectral.DevicePack(pack, case["h_kv"], torch.device("cuda"), "rtn",
                                                                  case["v_codec"]))
    return _PACKS[key]


def _spectral_fields(g, case, content):
    """Page-order columns and their codes: (columns or -1, tier of each slice, codes (T, n), steps (T/64, n))."""
    T = case["packed"]
    lam, bits = content[2], content[3].tolist()
    cols, slices = [], []
    for b in sorted(set(bits) - {0}):
        mine = [j for j, x in enumerate(bits) if x == b]
        mine += [-1] * (-len(mine) % 8)
        cols += mine
        slices += [b] * (len(mine) // 8)
    tier = torch.tensor(slices, device="cuda").repeat_interleave(8)
    unit = torch.tensor([TIER_STEP[b] for b in slices], device="cuda").repeat_interleave(8)
    at = torch.tensor(cols, device="cuda")
    sigma = lam.cuda()[at.clamp_min(0)].sqrt() * (at >= 0)
    half = 2.0 ** (tier - 1)
    codes = (_randn(g, T, len(cols)) / unit).round()
    codes = torch.minimum(torch.maximum(codes, -half), half - 1) * (at >= 0)
    steps = (sigma * unit * (0.8 + 0.4 * torch.rand(T // 64, len(cols), generator=g, device="cuda"))).half()
    h = 1 if case["v_codec"] == "full" else case["h_kv"]
    vidx, vnorm = _value_codes(g, h, T, 128 * case["h_kv"] // h)
    return dict(at=at, slices=slices, tier=tier, codes=codes.to(torch.int64), steps=steps, vidx=vidx, vnorm=vnorm)


def _spectral_pages(f, case):
    T, n = f["codes"].shape
    stored = f["codes"] + (1 << (f["tier"] - 1))
    parts = [_bytes(f["steps"])]
    for s, b in enumerate(f["slices"]):
        w = TIER_BITS[b]
        c = stored[:, 8 * s: 8 * s + 8].reshape(T, w, 8 // w)      # 8 / w codes in a byte
        sh = torch.arange(8 // w, device="cuda") * w
        parts.append((c << sh).sum(-1).to(torch.uint8).reshape(T // 64, 64 * w))
    parts.append(torch.zeros(T // 64, 16, dtype=torch.uint8, device="cuda"))
    v = f["vidx"]                                                   # (1, T, C) or (h, T, 128)
    norm = f["vnorm"].view(-1, T // PT, PT).permute(1, 0, 2).reshape(T // PT, -1)
    v = v.reshape(-1, T, v.shape[2] // 128, 128).permute(0, 2, 1, 3).reshape(-1, T, 128)
    vp = torch.cat((_bytes(norm), _value_words(v.contiguous()).reshape(T // PT, -1)), 1)
    return torch.cat(parts, 1).contiguous(), vp.contiguous()


def _spectral_inputs(case, seed, content):
    g = _gen(seed)
    f = _spectral_fields(g, case, content)
    q = _queries(g, case, case["h_kv"], case["G"], 128)
    return (f, q) + _window(g, case, case["h_kv"], case["window"], 128)


def _prepare_spectral_decode(case, seed):
    content, dp = _device_pack(case)
    f, q, k, v = _spectral_inputs(case, seed, content)
    kp, vp = _spectral_pages(f, case)
    n = case["packed"]
    return dict(kind="spectral_decode", dp=dp, kp=kp, vp=vp, n=n, q=q, k=k, v=v, consts=_consts(500000.0, 128),
                kt=torch.arange(n // 64, dtype=torch.int32, device="cuda"),
                vt=torch.arange(n // PT, dtype=torch.int32, device="cuda"))


def _prepare_k2b_append(case, seed):
    g = _gen(seed)
    h, T, R, d = case["h_kv"], case["tokens"], case["rank"], case["head_dim"]
    basis = _orthonormal(g, h * d, R)
    us = _randn(g, T, R) * _spread(R, h * d / 2)
    keys = us @ basis.T + 0.3 * _randn(g, T, h * d)
    keys = keys.view(T, h, d).transpose(0, 1).half().contiguous()
    v = _randn(g, h, T, d).to(DTYPES[case["dtype"]])
    pb = k2b.page_bytes(h, R, head_dim=d, group=case["group"], k_bits=case["k_bits"])
    return dict(kind="k2b_append", case=case, keys=keys, v=v, basis32=basis, basis16=basis.half(),
                pages=torch.zeros(T // PT, pb, dtype=torch.uint8, device="cuda"),
                ids=torch.arange(T // PT, dtype=torch.int32, device="cuda"), consts=_consts(500000.0, d),
                us_first=us[:128].contiguous() if case["first"] else None)


def _prepare_spectral_append(case, seed):
    (enc, dec, lam, _), dp = _device_pack(case)
    g = _gen(seed)
    h, T = case["h_kv"], case["tokens"]
    keys = (_randn(g, T, 128 * h) * lam.sqrt().cuda()) @ dec.cuda().T
    keys = keys.view(T, h, 128).transpose(0, 1).half().contiguous()
    v = _randn(g, h, T, 128).to(DTYPES[case["dtype"]])
    return dict(kind="spectral_append", dp=dp, keys=keys, v=v, consts=_consts(500000.0, 128),
                kp=torch.zeros(T // 64, dp.k_page_bytes, dtype=torch.uint8, device="cuda"),
                vp=torch.zeros(T // PT, dp.v_page_bytes, dtype=torch.uint8, device="cuda"),
                kids=torch.arange(T // 64, dtype=torch.int32, device="cuda"),
                vids=torch.arange(T // PT, dtype=torch.int32, device="cuda"))


def _cached_prefill_inputs(case, seed):
    """Pre-RoPE keys (T, C), rotated keys and values (h, T, 128) and queries of a prompt, in the model's dtype."""
    g = _gen(seed)
    h, N, dt = case["h_kv"], case["context"] + case["queries"], DTYPES[case["dtype"]]
    basis = _orthonormal(g, h * 128, case["rank"])
    keys = (_randn(g, N, case["rank"]) * _spread(case["rank"], h * 64.0)) @ basis.T + 0.3 * _randn(g, N, h * 128)
    keys = keys.to(dt)
    rot = _rope(keys.view(N, h, 128).transpose(0, 1).float(), torch.arange(N, device="cuda"),
                _inv_freq(500000.0, 128)).to(dt)
    return keys, rot, _randn(g, h, N, 128).to(dt), _queries(g, case, h * case["G"], case["queries"], 128)


def _prepare_cached_prefill(case, seed):
    h, G = case["h_kv"], case["G"]
    keys, rot, v, q = _cached_prefill_inputs(case, seed)
    cfg = SimpleNamespace(hidden_size=128 * h * G, num_attention_heads=h * G, num_key_value_heads=h, head_dim=128,
                          num_hidden_layers=1, max_position_embeddings=131072,
                          rope_parameters={"rope_type": "default", "rope_theta": 500000.0})
    layer = PackedStreamingLayer(*spec_pair("k2b_ph", rank=case["rank"]), cfg, recent_window=case["window"])
    for lo, hi in ((0, case["context"]), (case["context"], keys.shape[0])):
        layer.stash_pre_rope(keys[None, lo:hi])
        layer.update(rot[None, :, lo:hi], v[None, :, lo:hi])
    return dict(kind="cached_prefill", layer=layer, q=q)


def _prefill_inputs(case, seed):
    g, dt = _gen(seed), DTYPES[case["dtype"]]
    q = _queries(g, case, case["h_kv"] * case["G"], case["queries"], 128)
    k = (0.7 * _randn(g, case["h_kv"], case["keys"], 128)).to(dt)
    return q, k, _randn(g, case["h_kv"], case["keys"], 128).to(dt)


def _prepare_prefill(case, seed):
    q, k, v = _prefill_inputs(case, seed)
    return dict(kind="prefill", q=q, k=k, v=v, causal=case["causal"])


PREPARE = dict(decode=_prepare_decode, rtn_decode=_prepare_rtn, spectral_decode=_prepare_spectral_decode,
               k2b_append=_prepare_k2b_append, spectral_append=_prepare_spectral_append,
               cached_prefill=_prepare_cached_prefill, prefill=_prepare_prefill)


def prepare(case, seed):
    return PREPARE[case["kind"]](case, seed)


# ------------------------------------------------------------------ one pass


def run(s):
    kind = s["kind"]
    if kind == "decode":
        if s["host_len"]:
            return [plan.run(q=q, tail_len=s["window"], new_kv=new) for plan, q, new in s["calls"]]
        return [plan.run(q=q) for plan, q, _ in s["calls"]]
    if kind == "spectral_decode":
        return spectral.decode_attention(s["dp"], s["kp"], s["kt"], s["vp"], s["vt"], s["n"], s["consts"], s["q"],
                                         128 ** -0.5, k_win=s["k"], v_win=s["v"])
    if kind == "k2b_append":
        c = s["case"]
        k2b.append(s["keys"], s["v"], s["basis32"], s["basis16"], s["pages"], s["ids"], s["consts"], rank=c["rank"],
                   us_first=s["us_first"], group=c["group"], k_bits=c["k_bits"])
        return s["pages"]
    if kind == "spectral_append":
        spectral.append(s["keys"], s["v"], s["dp"], s["kp"], s["kids"], s["vp"], s["vids"], s["consts"])
        return [s["kp"], s["vp"]]
    if kind == "cached_prefill":
        return s["layer"].attend(s["q"], 128 ** -0.5, is_causal=True)
    return prefill.attention(s["q"], s["k"], s["v"], 128 ** -0.5, causal=s["causal"])


# ------------------------------------------------------------------ what a pass cannot do without


def work(case):
    kind, e = case["kind"], 4 if case["dtype"] == "fp32" else 2
    h = case["h_kv"]
    if kind == "decode":
        d, R, G, W, B = case["head_dim"], case["rank"], case["G"], case["window"], case["batch"]
        C = h * d
        page = 2 * R + 2 * h + C * 2 // case["group"] + C * case["k_bits"] // 8 + C // 4   # bytes a token
        tokens = case["packed"] if B == 1 else int(B * case["packed"] * 0.625)
        fixed = B * (C * R * 2 + 2 * W * C * e + 2 * C * G * e)
        return dict(bytes=case["layers"] * (tokens * page + fixed),
                    flops=case["layers"] * (tokens * (2 * C * R + 4 * G * C) + B * W * 4 * G * C))
    if kind == "rtn_decode":
        C, W, G = 128 * h, case["window"], case["G"]
        page = C * (case["k_bits"] + case["v_bits"]) / 8 + 2 * C / case["k_group"] + 2 * C / case["v_group"]
        return dict(bytes=case["layers"] * (case["packed"] * page + 2 * W * C * e + 2 * C * G * e),
                    flops=case["layers"] * (case["packed"] + W) * 4 * G * C)
    if kind in ("spectral_decode", "spectral_append"):
        C = 128 * h
        T = case["packed"] if kind == "spectral_decode" else case["tokens"]
        page = C * case["budget"] / 8 + 2 * C / 64 + C / 4 + 2 * (1 if case["v_codec"] == "full" else h)
        if kind == "spectral_decode":
            W, G = case["window"], case["G"]
            return dict(bytes=T * page + 2 * C * C + 2 * W * C * e + 2 * C * G * e,
                        flops=T * (2 * C * C + 4 * G * C) + 4 * W * G * C)
        return dict(bytes=T * page + 4 * C * C + T * C * (2 + e), flops=2 * T * C * C)
    if kind == "k2b_append":
        C, T, R = h * case["head_dim"], case["tokens"], case["rank"]
        page = 2 * R + 2 * h + C * 2 // case["group"] + C * case["k_bits"] // 8 + C // 4
        return dict(bytes=T * page + 6 * C * R + T * C * (2 + e), flops=T * (4 * C * R + 10 * C))
    C, nq = 128 * h, case["queries"]
    if kind == "cached_prefill":
        N, R = case["context"] + nq, case["rank"]
        page = 2 * R + 2 * h + C // 32 + C * 5 // 8
        return dict(bytes=N * page + 2 * R * C + 2 * nq * C * case["G"] * e,
                    flops=4 * C * case["G"] * (nq * case["context"] + nq * (nq + 1) / 2) + 2 * N * C * R)
    n = case["keys"]
    seen = nq * (n - nq) + nq * (nq + 1) / 2 if case["causal"] else nq * n
    return dict(bytes=2 * n * C * e + 2 * nq * C * case["G"] * e, flops=4 * C * case["G"] * seen)


def tolerance(case):
    """Encoded pages are whole numbers in a fixed order of operations; attention outputs carry the 16-bit rounding of
    the keys, weights and outputs (against `exact`: 2-norm errors of 0.3e-3 .. 1.0e-3 in fp16, 1.7e-3 .. 2.1e-3 in bf16;
    four times those)."""
    if case["kind"] in ("k2b_append", "spectral_append"):
        return "exact"
    return {"rel": 8e-3, "max": 0.1} if case["dtype"] == "bf16" else {"rel": 4e-3, "max": 0.06}


# ------------------------------------------------------------------ the same in 64 bits


def _hadamard(x):
    """Unnormalized Walsh-Hadamard transform (Sylvester order) of the last dimension."""
    n, shape = 1, x.shape
    while n < shape[-1]:
        y = x.reshape(*shape[:-1], -1, 2, n)
        x = torch.stack((y[..., 0, :] + y[..., 1, :], y[..., 0, :] - y[..., 1, :]), -2).reshape(shape)
        n *= 2
    return x


def _values64(vidx, vnorm, d):
    """(h, T, d) values of 2-bit codes: norm * signs * H levels / d."""
    lv = torch.tensor(LEVELS, dtype=torch.float64, device="cuda")[vidx.long()]
    return _hadamard(lv) * _signs(d).cuda() / d * vnorm.double()[..., None]


def _attend64(q, k, v):
    """q (h, G, d) over keys and values (h, n, d)."""
    s = q.double() @ k.transpose(1, 2) * q.shape[-1] ** -0.5
    return torch.softmax(s, -1) @ v


def _exact_decode(case, seed):
    outs, h, d, R = [], case["h_kv"], case["head_dim"], case["rank"]
    inv = _inv_freq(case["theta"], d)
    for lens, fields, basis, q, kw, vw in _decode_layers(case, seed):
        got = []
        for b, (n, f) in enumerate(zip(lens, fields)):
            k = (f["us"].double() @ basis[b].double().T).view(n, h, d).transpose(0, 1)
            k = k + f["res"].double() * f["scale"].double().repeat_interleave(case["group"], 1)
            k = _rope(k, torch.arange(n, device="cuda"), inv)
            v = _values64(f["vidx"], f["vnorm"], d)
            got.append(_attend64(q[b], torch.cat((k, kw[b].double()), 1), torch.cat((v, vw[b].double()), 1)))
            del k, v
        outs.append(torch.stack(got))
    return outs


def _exact_rtn(case, seed):
    outs = []
    for f, q, kw, vw in _rtn_layers(case, seed):
        ks = f["ks"].double().repeat_interleave(case["k_group"], 1 if case["channel"] else 2)
        k = f["kq"].double() * ks
        v = f["vq"].double() * f["vs"].double().repeat_interleave(case["v_group"], 2)
        outs.append(_attend64(q[0], torch.cat((k, kw[0].double()), 1), torch.cat((v, vw[0].double()), 1))[None])
    return outs


def _exact_spectral(case, seed):
    content = _pack(case)
    f, q, kw, vw = _spectral_inputs(case, seed, content)
    n, h = case["packed"], case["h_kv"]
    dec = content[1].cuda().half().double()[:, f["at"].clamp_min(0)] * (f["at"] >= 0)
    y = f["codes"].double() * f["steps"].double().repeat_interleave(64, 0)
    k = (y @ dec.T).view(n, h, 128).transpose(0, 1)
    k = _rope(k, torch.arange(n, device="cuda"), _inv_freq(500000.0, 128), half_tables=True)
    if case["v_codec"] == "full":
        v = _values64(f["vidx"], f["vnorm"], 128 * h)[0].view(n, h, 128).transpose(0, 1)
    else:
        v = _values64(f["vidx"], f["vnorm"], 128)
    return _attend64(q, torch.cat((k, kw.double()), 1), torch.cat((v, vw.double()), 1))


def _rows64(q, k, v, G, causal):
    """Attention of (h G, n_q, 128) queries, head by head; causal from the bottom right."""
    out = torch.empty(q.shape, dtype=torch.float64, device="cuda")
    nq, n = q.shape[1], k.shape[1]
    hidden = torch.arange(n, device="cuda")[None] > torch.arange(nq, device="cuda")[:, None] + (n - nq)
    for i in range(q.shape[0]):
        s = q[i].double() @ k[i // G].double().T * 128 ** -0.5
        out[i] = torch.softmax(s.masked_fill_(hidden, -math.inf) if causal else s, -1) @ v[i // G].double()
    return out


def _exact_cached_prefill(case, seed):
    h, R = case["h_kv"], case["rank"]
    keys, rot, v, q = _cached_prefill_inputs(case, seed)
    N, W, k, val = keys.shape[0], case["window"], rot.double(), v.double()
    P = (N - W) // 128 * 128 if N > W else 0
    if P:   # the committed tokens through the codec
        m = keys[:P].half().double()
        U, s, Vh = torch.linalg.svd(m[:128].float().cpu(), full_matrices=False)
        us = torch.cat((U[:, :R].double().cuda() * s[:R].double().cuda(), m[128:] @ Vh[:R].double().T.cuda()))
        us, basis = us.half().double(), Vh[:R].half().double().cuda()
        res = (m - us @ basis).view(P // 64, 64, h * 128)
        step = res.abs().amax(1, keepdim=True).clamp_min(1e-12) / 3
        code = (res / step).round().clamp(-4, 3)
        k16 = us @ basis + (code * step.half().double()).view(P, h * 128)
        k16 = _rope(k16.view(P, h, 128).transpose(0, 1), torch.arange(P, device="cuda"), _inv_freq(500000.0, 128),
                    half_tables=True)
        vn = val[:, :P].norm(dim=-1).half()
        r = _hadamard(val[:, :P] / vn.double()[..., None] * _signs(128).cuda())
        mids = torch.tensor([(a + b) / 2 for a, b in zip(LEVELS, LEVELS[1:])], dtype=torch.float64, device="cuda")
        k = torch.cat((k16, k[:, P:]), 1)
        val = torch.cat((_values64(torch.bucketize(r, mids), vn, 128), val[:, P:]), 1)
    return _rows64(q, k, val, case["G"], True)


def exact(case, seed):
    kind = case["kind"]
    if kind == "decode":
        return _exact_decode(case, seed)
    if kind == "rtn_decode":
        return _exact_rtn(case, seed)
    if kind == "spectral_decode":
        return _exact_spectral(case, seed)
    if kind == "cached_prefill":
        return _exact_cached_prefill(case, seed)
    if kind == "prefill":
        q, k, v = _prefill_inputs(case, seed)
        return _rows64(q, k, v, case["G"], case["causal"])
    return None   # encoded pages are whole numbers
