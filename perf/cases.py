"""The calls whose speed this framework is judged by.

Every case goes through the package's public entry points as a program that
serves or bakes with it does; a case is a dict of plain values:

    call      omni_attn, the drop-in call of a per-user loop: everything is
              validated and allocated on each call
    serve     PackedKVAttention.run with a LoRA bank, the serving loop's step
    decode    PackedKVAttention.run over a long cache, one or a few query
              tokens per sequence, head_dim 128 or 32
    paged     one serving step over pages: PagedKVCache.append, then
              PagedKVAttention.run, ragged lengths
    prefill   omni_attn with causal_offset: a chunk of new tokens against the
              cache, head_dim 128 or 32
    encode    PackedKVEncoder.encode of a prompt's K and V (rotation fused)
    bake      rotation, per-head Lloyd-Max calibration and encoding of a raw
              cache, the GPU part of bake_kv_cache
    dequant   dequantize_heads (the unfused path, fidelity checks)
    dense     reference_attn on dense K and V, the block of ReferenceAttention

`listed` holds the sizes of the benchmark configurations and of the
reference's drivers (64 users x 50 tokens, 32 x 8192 cached tokens, 16 x 4096
tokens to encode, 512-token chunks over 16384 tokens, 256 users to bake), one
user alone, and ragged sizes between them; `draw` spreads the same kinds over
their ranges.
"""
from __future__ import annotations

import math
import os
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "omnistack-rs_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from omnistack_rs.attention import reference_attn  # noqa: E402
from omnistack_rs.cache import PagedKVAttention, PagedKVCache  # noqa: E402
from omnistack_rs.kernels.fused_attention import PackedKVAttention, omni_attn  # noqa: E402
from omnistack_rs.kernels.hadamard import _wht_torch  # noqa: E402
from omnistack_rs.kernels.quantize import PackedKVEncoder, dequantize_heads, quantize_heads  # noqa: E402
from omnistack_rs.quantization import calibrate_heads  # noqa: E402

DEV = torch.device("cuda", 0)
UID = 42
DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
# Max's (1960) 16-level quantizer of N(0, 1)
_LEVELS = (0.1284, 0.3881, 0.6568, 0.9424, 1.2562, 1.6181, 2.0690, 2.7326)


# ── the cases ───────────────────────────────────────────────────────────

def listed():
    return [
        # one user of a per-user loop: 50 tokens, f32 query, everything per call
        dict(name="call_1x50", kind="call", B=1, Hq=8, Hkv=8, T=1, S=50, D=128, dtype="f32", qjl=True),
        # the serving loop's step: 64 of 256 cached users, rank-8 adapters
        dict(name="serve_64x50_lora", kind="serve", B=64, pool=256, Hq=32, Hkv=8, S=50, rank=8, hidden=128,
             n_loras=256, dtype="bf16"),
        # long-context decode, one token of each of 32 sequences
        dict(name="decode_32x8192", kind="decode", B=32, Hq=32, Hkv=8, T=1, S=8192, D=128, dtype="bf16", qjl=True),
        # a few draft tokens verified at once over a ragged long cache, wide GQA groups
        dict(name="decode_3x20011_t3", kind="decode", B=3, Hq=64, Hkv=8, T=3, S=20011, D=128, dtype="f16", qjl=True),
        # the manifold-pruned (head_dim 32) cache, one token of each sequence
        dict(name="decode_32x8192_d32", kind="decode", B=32, Hq=32, Hkv=8, T=1, S=8192, D=32, dtype="bf16", qjl=True),
        # one step of a paged server: 48 sequences of 200 to 3000 tokens
        dict(name="paged_48_ragged", kind="paged", B=48, Hq=32, Hkv=8, lo=200, hi=3000, page=16, dtype="bf16"),
        # chunked prefill over a long prompt, both head sizes
        dict(name="prefill_8x512_16k", kind="prefill", B=8, Hq=32, Hkv=8, T=512, S=16384, D=128, dtype="bf16"),
        dict(name="prefill_8x512_16k_d32", kind="prefill", B=8, Hq=32, Hkv=8, T=512, S=16384, D=32, dtype="bf16"),
        # a prompt batch's K and V into the packed cache
        dict(name="encode_16x4096", kind="encode", B=16, H=8, T=4096, D=128, dtype="bf16"),
        # the offline bake of 256 users, float32 as the reference's driver feeds it
        dict(name="bake_256x50", kind="bake", B=256, H=8, T=50, D=128, dtype="f32"),
        # the packed cache back to float32
        dict(name="dequant_8x2049", kind="dequant", B=8, H=8, T=2049, D=128, qjl=True),
        # the dense block on a whole prompt with its causal mask
        dict(name="dense_2x1000", kind="dense", B=2, Hq=32, Hkv=8, T=1000, S=1000, D=128, mask=True, dtype="f32"),
    ]


def _log(rng, lo, hi):
    """A whole number spread over the logarithm of [lo, hi]."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["call", "serve", "decode", "decode", "paged", "prefill", "prefill", "encode", "bake",
                       "dequant", "dense"])
    hkv, g = rng.choice([(8, 4), (8, 1), (8, 8), (4, 4)])
    if kind == "call":
        return dict(kind=kind, B=_log(rng, 1, 64), Hq=hkv * g, Hkv=hkv, T=1, S=_log(rng, 17, 2000), D=128,
                    dtype=rng.choice(["f32", "bf16", "f16"]), qjl=rng.random() < 0.8)
    if kind == "serve":
        B = _log(rng, 1, 256)
        return dict(kind=kind, B=B, pool=rng.choice([0, B + 13, 4 * B]), Hq=32, Hkv=8, S=_log(rng, 17, 600),
                    rank=rng.choice([8, 16]), hidden=rng.choice([128, 256]), n_loras=rng.choice([16, 256]),
                    dtype=rng.choice(["bf16", "f16"]))
    if kind == "decode":
        B = _log(rng, 1, 64)
        S = _log(rng, 150, min(131072, 262144 // B))
        return dict(kind=kind, B=B, Hq=hkv * g, Hkv=hkv, T=rng.choice([1, 1, 2, 4]), S=S, D=rng.choice([128, 128, 32]),
                    dtype=rng.choice(["bf16", "f16", "f32"]), qjl=rng.random() < 0.8)
    if kind == "paged":
        hi = _log(rng, 64, 6000)
        return dict(kind=kind, B=_log(rng, 1, 64), Hq=32, Hkv=8, lo=max(1, hi // rng.choice([1, 3, 20])), hi=hi,
                    page=rng.choice([16, 64, 256]), dtype=rng.choice(["bf16", "f16"]))
    if kind == "prefill":
        B, T = _log(rng, 1, 8), _log(rng, 40, 1000)
        dtype = rng.choice(["bf16", "bf16", "f16", "f32"])
        most = 8 * 512 * 16384 // (2 if dtype == "f32" else 1)
        S = _log(rng, T, max(T, min(16384, most // (B * T))))
        return dict(kind=kind, B=B, Hq=32, Hkv=8, T=T, S=S, D=rng.choice([128, 128, 32]), dtype=dtype)
    if kind == "encode":
        B = _log(rng, 1, 64)
        return dict(kind=kind, B=B, H=8, T=_log(rng, 1, 65536 // B), D=rng.choice([128, 128, 32]),
                    dtype=rng.choice(["bf16", "f16", "f32"]))
    if kind == "bake":
        B = _log(rng, 8, 256)
        return dict(kind=kind, B=B, H=8, T=_log(rng, 10, 50), D=128, dtype=rng.choice(["f32", "bf16"]))
    if kind == "dequant":
        B = _log(rng, 1, 64)
        return dict(kind=kind, B=B, H=8, T=_log(rng, 1, 16384 // B), D=rng.choice([128, 128, 32]),
                    qjl=rng.random() < 0.7)
    T = rng.choice([1, _log(rng, 2, 1000)])
    S = _log(rng, max(T, 33), 1000) if T > 1 else _log(rng, 33, 8000)
    return dict(kind="dense", B=_log(rng, 1, 2 if T > 1 else 16), Hq=32, Hkv=8, T=T, S=S, D=rng.choice([128, 64, 32]),
                mask=T > 1 and rng.random() < 0.7, dtype=rng.choice(["f32", "bf16"]))


# ── inputs ──────────────────────────────────────────────────────────────

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV, dtype=torch.float32)


def _levels():
    c = torch.tensor(_LEVELS, device=DEV)
    return torch.cat([-c.flip(0), c])


def _codebooks(g, H):
    """One N(0, 1) codebook per head, scaled as calibrated heads differ."""
    return _levels() * (0.8 + 0.45 * torch.rand(H, 1, generator=g, device=DEV))


def _nibbles(g, B, H, S, D):
    lv = _levels()
    mid = (lv[1:] + lv[:-1]) / 2
    out = torch.empty(B, H, S, D // 2, dtype=torch.uint8, device=DEV)
    for b in range(B):
        c = torch.bucketize(_randn(g, H, S, D), mid, out_int32=True)
        out[b] = (c[..., 0::2] | (c[..., 1::2] << 4)).to(torch.uint8)
    return out


def _packed(g, B, H, S, D):
    """K nibbles, K signs, K norms, V nibbles as the encoder leaves them for
    N(0, 1) data: residual norms near sqrt(0.0095 D)."""
    kn = _nibbles(g, B, H, S, D)
    vn = _nibbles(g, B, H, S, D)
    kq = torch.randint(0, 256, (B, H, S, D // 16), generator=g, device=DEV, dtype=torch.uint8)
    kr = math.sqrt(0.0095 * D) * (1.0 + 0.09 * _randn(g, B, H, S)).clamp_min(0.1)
    return kn, kq, kr, vn


def _flip(g, D):
    return (torch.randint(0, 2, (D,), generator=g, device=DEV) * 2 - 1).to(torch.int8)


def _raw(g, *shape):
    """Raw activations: N(0, 1), 2 % of the channels eight times larger."""
    x = _randn(g, *shape)
    n = max(1, round(0.02 * shape[-1]))
    x[..., torch.randperm(shape[-1], generator=g, device=DEV)[:n]] *= 8.0
    return x


def _inputs(c, seed):
    """Everything a case's call reads, as tensors (prepare and exact share it)."""
    g = _gen(seed)
    k = c["kind"]
    if k in ("call", "serve", "decode", "prefill"):
        D, T = c.get("D", 128), c.get("T", 1)
        dt = DTYPES[c["dtype"]]
        n = c.get("pool") or c["B"]
        cache = _packed(g, n, c["Hkv"], c["S"], D)
        s = dict(cache=cache, cb=_codebooks(g, c["Hkv"]), q=_randn(g, c["B"], c["Hq"], T, D).to(dt), flip=_flip(g, D))
        if k == "serve":
            s["a"] = (0.02 * _randn(g, c["n_loras"], c["rank"], c["hidden"])).to(dt)
            s["b"] = (0.02 * _randn(g, c["n_loras"], c["Hq"] * D, c["rank"])).to(dt)
            s["x"] = _randn(g, c["B"], 1, c["hidden"]).to(dt)
            s["ids"] = torch.randint(-1, c["n_loras"], (c["B"],), generator=g, device=DEV, dtype=torch.int32)
            if c["pool"]:
                s["index"] = torch.randperm(n, generator=g, device=DEV)[: c["B"]].contiguous()
        return s
    if k == "paged":
        dt = DTYPES[c["dtype"]]
        lens = torch.randint(c["lo"], c["hi"] + 1, (c["B"],), generator=g, device=DEV, dtype=torch.int32)
        return dict(cache=_packed(g, c["B"], c["Hkv"], c["hi"], 128), cb=_codebooks(g, c["Hkv"]), flip=_flip(g, 128),
                    q=_randn(g, c["B"], c["Hq"], 1, 128).to(dt), k=_raw(g, c["B"], c["Hkv"], 1, 128).to(dt),
                    v=_raw(g, c["B"], c["Hkv"], 1, 128).to(dt), lens=lens)
    if k == "encode":
        dt = DTYPES[c["dtype"]]
        return dict(k=_raw(g, c["B"], c["H"], c["T"], c["D"]).to(dt), v=_raw(g, c["B"], c["H"], c["T"], c["D"]).to(dt),
                    cb=_codebooks(g, c["H"]), flip=_flip(g, c["D"]))
    if k == "bake":
        return dict(x=_randn(g, c["B"], c["H"], c["T"], c["D"]).to(DTYPES[c["dtype"]]))
    if k == "dequant":
        kn, kq, kr, _ = _packed(g, c["B"], c["H"], c["T"], c["D"])
        return dict(nib=kn, qjl=kq, nrm=kr, cb=_codebooks(g, c["H"]))
    dt = DTYPES[c["dtype"]]
    s = dict(q=_randn(g, c["B"], c["Hq"], c["T"], c["D"]).to(dt), k=_randn(g, c["B"], c["Hkv"], c["S"], c["D"]).to(dt),
             v=_randn(g, c["B"], c["Hkv"], c["S"], c["D"]).to(dt), mask=None)
    if c["mask"]:
        hide = torch.ones(c["T"], c["S"], dtype=torch.bool, device=DEV).triu(c["S"] - c["T"] + 1)
        s["mask"] = torch.zeros(1, 1, c["T"], c["S"], device=DEV).masked_fill(hide, float("-inf"))
    return s


def prepare(case, seed):
    c, s = case, _inputs(case, seed)
    k = c["kind"]
    s["case"] = c
    if k in ("serve", "decode"):
        kn, kq, kr, vn = s.pop("cache")
        more = {}
        if k == "serve":
            more = dict(lora_a=s.pop("a"), lora_b=s.pop("b"), lora_alpha=1.0)
            if c["pool"]:
                more["batch"] = c["B"]
        s["att"] = PackedKVAttention(kn, kq, kr, vn, s["cb"], n_heads=c["Hq"], q_tokens=c.get("T", 1), user_id=UID,
                                     with_qjl=c.get("qjl", True), q_dtype=DTYPES[c["dtype"]], rotate_q=True,
                                     sign_flip=s["flip"], **more)
    elif k == "paged":
        cache = s.pop("cache")
        order = torch.Generator().manual_seed(seed)
        lens = s["lens"].tolist()
        free = c["B"] * -(-c["hi"] // c["page"]) - sum(-(-n // c["page"]) for n in lens)   # a pool of fixed size
        s["pool"], s["table"], s["lens"] = PagedKVCache.from_contiguous(
            *cache, page_size=c["page"], seq_lens=lens, spare_pages=free, generator=order)
        s["pos"] = s["lens"] - 1
        s["enc"] = PackedKVEncoder(s["cb"], c["Hkv"], user_id=UID, sign_flip=s["flip"], dtype=DTYPES[c["dtype"]])
        s["att"] = PagedKVAttention(s["pool"], s["cb"], n_heads=c["Hq"], batch=c["B"], max_pages=s["table"].shape[1],
                                    user_id=UID, q_dtype=DTYPES[c["dtype"]], rotate_q=True, sign_flip=s["flip"])
    elif k == "encode":
        s["enc"] = PackedKVEncoder(s["cb"], c["H"], user_id=UID, sign_flip=s["flip"], dtype=DTYPES[c["dtype"]],
                                   head_dim=c["D"])
        s["out"] = (s["enc"].empty_outputs(c["B"], c["T"]), s["enc"].empty_outputs(c["B"], c["T"]))
    return s


def run(s):
    c = s["case"]
    k = c["kind"]
    if k == "call":
        kn, kq, kr, vn = s["cache"]
        return omni_attn(s["q"], kn, kq, kr, vn, s["cb"], user_id=UID, with_qjl=c["qjl"])
    if k == "serve":
        return s["att"].run(s["q"], s["x"], s["ids"], cache_index=s.get("index"))
    if k == "decode":
        return s["att"].run(s["q"])
    if k == "paged":
        p = s["pool"]
        p.append(s["enc"], s["k"], s["v"], s["table"], s["pos"], validate=False)
        out = s["att"].run(s["q"], s["table"], s["lens"])
        return out, p.k_nibbles, p.k_qjl, p.k_norms, p.v_nibbles
    if k == "prefill":
        kn, kq, kr, vn = s["cache"]
        return omni_attn(s["q"], kn, kq, kr, vn, s["cb"], user_id=UID, causal_offset=c["S"] - c["T"], rotate_q=True,
                         sign_flip=s["flip"])
    if k == "encode":
        return s["enc"].encode(s["k"], s["v"], out=s["out"])
    if k == "bake":
        rot = _wht_torch(s["x"])
        cb = calibrate_heads(rot)
        return (*quantize_heads(rot, cb, user_id=UID), cb)
    if k == "dequant":
        return dequantize_heads(s["nib"], s["qjl"], s["nrm"], s["cb"], user_id=UID, with_qjl=c["qjl"])
    return reference_attn(s["q"], s["k"], s["v"], mask=s["mask"])


# ── what a pass cannot do without ───────────────────────────────────────

def _token_bytes(D, qjl):
    return D // 2 + D // 2 + (D // 16 + 4 if qjl else 0)


def work(case):
    c, k = case, case["kind"]
    if k in ("call", "serve", "decode", "prefill"):
        D, T = c.get("D", 128), c.get("T", 1)
        qjl = c.get("qjl", True)
        rows = c["B"] * c["Hq"] * T
        keys = c["S"] - (T - 1) / 2 if k == "prefill" else c["S"]
        b = c["B"] * c["Hkv"] * c["S"] * _token_bytes(D, qjl) + rows * D * (DTYPES[c["dtype"]].itemsize + 4)
        f = rows * keys * (4 * D + (D if qjl else 0))
        if k == "serve":
            used = min(c["B"], c["n_loras"])
            b += 2 * used * c["rank"] * (c["hidden"] + c["Hq"] * D) + 2 * c["B"] * c["hidden"]
            f += 2 * c["B"] * c["rank"] * (c["hidden"] + c["Hq"] * D)
        return {"bytes": b, "flops": f}
    if k == "paged":
        toks = c["B"] * (c["lo"] + c["hi"]) / 2
        rows = c["B"] * c["Hq"]
        new = c["B"] * c["Hkv"] * (2 * 256 + 140)
        return {"bytes": toks * c["Hkv"] * 140 + rows * 128 * 6 + new, "flops": toks * c["Hq"] * 5 * 128}
    D = c["D"]
    if k == "encode":
        n = 2 * c["B"] * c["H"] * c["T"]
        return {"bytes": n * (D * DTYPES[c["dtype"]].itemsize + D // 2 + D // 16 + 4), "flops": n * D * D}
    if k == "bake":
        n = c["B"] * c["H"] * c["T"]
        return {"bytes": n * (D * DTYPES[c["dtype"]].itemsize + D // 2 + D // 16 + 4), "flops": n * D * D}
    if k == "dequant":
        n = c["B"] * c["H"] * c["T"]
        return {"bytes": n * (D // 2 + (D // 16 + 4 if c["qjl"] else 0) + 4 * D), "flops": n * D * D if c["qjl"] else 0}
    e = DTYPES[c["dtype"]].itemsize
    b = e * D * (2 * c["B"] * c["Hq"] * c["T"] + 2 * c["B"] * c["Hkv"] * c["S"])
    if c["mask"]:
        b += 4 * c["T"] * c["S"]
    return {"bytes": b, "flops": 4 * c["B"] * c["Hq"] * c["T"] * c["S"] * D}


def tolerance(case):
    k = case["kind"]
    if k == "dequant":
        return "exact"                       # one rounding of an exact integer times a scale
    if k == "encode":
        return {"rel": 1e-6, "max": 1e-6}    # codes and signs are exact, norms within an ulp
    if k == "bake":
        # a codebook's last bits depend on the order of its sums, and move a few codes
        # (this code's codebooks are 6e-7 off 64 bits, and a sign byte then differs about 3e-5 of the time)
        return {"rel": 1e-5, "max": 2e-3, "differ": 1e-4}
    if k == "dense":
        # f32 sums are 4e-7 off 64 bits; 16-bit outputs differ by a last bit where a sum lies near a tie
        return {"rel": 3e-6, "max": 1e-4} if case["dtype"] == "f32" else {"rel": 2e-3, "max": 1e-2}
    # probabilities enter P . V in fp16: 2e-4 off 64 bits, and two runs that hand their tiles to
    # waves in another order differ by 2.6e-4 (largest difference 1.6e-3)
    return {"rel": 1.2e-3, "max": 1e-2}


# ── the same in 64 bits ─────────────────────────────────────────────────

def _g_matrix(h, D):
    gen = torch.Generator().manual_seed((UID % 1024) ^ h)
    return (torch.randint(0, 2, (D // 2, D), generator=gen) * 2 - 1).to(DEV, torch.float64)


def _rotated(x, flip=None):
    """dtype(fp32 WHT): the rotation is defined by its fp32 butterflies."""
    D = x.shape[-1]
    y = x.float() if flip is None else x.float() * flip.float()
    h = 1
    while h < D:
        y = y.reshape(*x.shape[:-1], D // (2 * h), 2, h)
        y = torch.stack([y[..., 0, :] + y[..., 1, :], y[..., 0, :] - y[..., 1, :]], dim=-2).reshape(x.shape)
        h *= 2
    return (y * torch.tensor(1.0 / math.sqrt(D), device=x.device)).to(x.dtype)


def _codes(nib):
    return torch.stack([nib & 15, nib >> 4], dim=-1).reshape(*nib.shape[:-1], 2 * nib.shape[-1]).long()


def _k_hat(nib, qjl, nrm, cb, h):
    """(S, D) in 64 bits of one head's packed rows."""
    D = 2 * nib.shape[-1]
    k = cb.double()[_codes(nib)]
    if qjl is None:
        return k
    bits = (qjl.unsqueeze(-1) >> torch.arange(8, device=DEV, dtype=torch.uint8)) & 1
    b = bits.reshape(*qjl.shape[:-1], D // 2).double() * 2 - 1
    return k + (b @ _g_matrix(h, D)) * (nrm.double() * (math.sqrt(2 / math.pi) / D)).unsqueeze(-1)


def _attend(q, k, v, scale, offset=None):
    """q (rows = (heads, T), D) against k, v (S, D); query t sees keys <= offset + t."""
    s = (q.flatten(0, 1) @ k.t()) * scale
    if offset is not None:
        t = torch.arange(q.shape[1], device=DEV).repeat(q.shape[0])
        s = s.masked_fill(torch.arange(k.shape[0], device=DEV)[None, :] > (offset + t)[:, None], float("-inf"))
    return (torch.softmax(s, dim=-1) @ v).reshape(q.shape)


def _encoded(x, cb, flip, rotate=True):
    """Rotated rows, codes and residuals (fp32, as the encoder defines them)."""
    r = (_rotated(x, flip) if rotate else x).float()
    code = torch.empty(r.shape, dtype=torch.int64, device=DEV)
    for h in range(r.shape[1]):
        for b in range(r.shape[0]):
            code[b, h] = (r[b, h].unsqueeze(-1) - cb[h].float()).abs().argmin(dim=-1)
    c = torch.stack([cb[h].float()[code[:, h]] for h in range(r.shape[1])], dim=1)
    return code, r - c


def exact(case, seed):
    c, k = case, case["kind"]
    s = _inputs(c, seed)
    if k in ("call", "serve", "decode", "prefill"):
        kn, kq, kr, vn = s["cache"]
        q = s["q"]
        D, G = q.shape[-1], c["Hq"] // c["Hkv"]
        if k == "serve":
            a, bw = s["a"].double(), s["b"].double()
            ids = s["ids"].long()
            on = ids.clamp_min(0)
            d = torch.einsum("btr,bor->bto", torch.einsum("bth,brh->btr", s["x"].double(), a[on]), bw[on])
            d = d.reshape(c["B"], 1, c["Hq"], D).transpose(1, 2)
            q = torch.where((ids >= 0)[:, None, None, None], (q.double() + d).to(q.dtype), q)
        if k != "call":
            q = _rotated(q, s["flip"])
        out = torch.empty(q.shape, dtype=torch.float64, device=DEV)
        for b in range(c["B"]):
            j = int(s["index"][b]) if "index" in s else b
            for h in range(c["Hkv"]):
                kh = _k_hat(kn[j, h], kq[j, h] if c.get("qjl", True) else None, kr[j, h], s["cb"][h], h)
                vh = _k_hat(vn[j, h], None, None, s["cb"][h], h)
                out[b, h * G:(h + 1) * G] = _attend(q[b, h * G:(h + 1) * G].double(), kh, vh, 1 / math.sqrt(D),
                                                    c["S"] - c["T"] if k == "prefill" else None)
        return out
    if k == "paged":
        kn, kq, kr, vn = s["cache"]
        G = c["Hq"] // c["Hkv"]
        q = _rotated(s["q"], s["flip"])
        kc, ke = _encoded(s["k"], s["cb"], s["flip"])
        vc, _ = _encoded(s["v"], s["cb"], s["flip"])
        out = torch.empty(q.shape, dtype=torch.float64, device=DEV)
        for b in range(c["B"]):
            n = int(s["lens"][b])
            for h in range(c["Hkv"]):
                kh = _k_hat(kn[b, h, :n], kq[b, h, :n], kr[b, h, :n], s["cb"][h], h)
                vh = _k_hat(vn[b, h, :n], None, None, s["cb"][h], h)
                e = ke[b, h, 0].double()
                sign = (_g_matrix(h, 128) @ e >= 0).double() * 2 - 1
                kh[n - 1] = s["cb"][h].double()[kc[b, h, 0]] + (sign @ _g_matrix(h, 128)) * (
                    e.norm() * math.sqrt(2 / math.pi) / 128)
                vh[n - 1] = s["cb"][h].double()[vc[b, h, 0]]
                out[b, h * G:(h + 1) * G] = _attend(q[b, h * G:(h + 1) * G].double(), kh, vh, 1 / math.sqrt(128))
        return out, None, None, None, None
    if k == "encode":
        return tuple((None, None, _encoded(t, s["cb"], s["flip"])[1].double().norm(dim=-1)) for t in (s["k"], s["v"]))
    if k == "bake":
        rot = _rotated(s["x"])
        cb = torch.stack([_lloyd_max(rot[:, h].reshape(-1).double()) for h in range(c["H"])])
        return None, None, _encoded(rot, cb.float(), None, rotate=False)[1].double().norm(dim=-1), cb
    if k == "dequant":
        return torch.stack([_k_hat(s["nib"][:, h], s["qjl"][:, h] if c["qjl"] else None, s["nrm"][:, h], s["cb"][h], h)
                            for h in range(c["H"])], dim=1)
    G = c["Hq"] // c["Hkv"]
    out = torch.empty(s["q"].shape, dtype=torch.float64, device=DEV)
    for b in range(c["B"]):
        for h in range(c["Hkv"]):
            out[b, h * G:(h + 1) * G] = _attend(s["q"][b, h * G:(h + 1) * G].double(), s["k"][b, h].double(),
                                                s["v"][b, h].double(), 1 / math.sqrt(c["D"]),
                                                c["S"] - c["T"] if c["mask"] else None)
    return out


def _lloyd_max(x, iters=300, tol=1e-6):
    """16 equal-count bins of the sorted samples, then Lloyd steps."""
    x = x.sort().values
    n = x.numel() // 16
    c = x[: 16 * n].reshape(16, n).mean(dim=1)
    total = torch.cat([x.new_zeros(1), x.cumsum(0)])
    for _ in range(iters):
        at = torch.searchsorted(x, (c[1:] + c[:-1]) / 2, right=True)
        at = torch.cat([at.new_zeros(1), at, at.new_full((1,), x.numel())])
        cnt = (at[1:] - at[:-1]).double()
        new = torch.where(cnt > 0, (total[at[1:]] - total[at[:-1]]) / cnt.clamp_min(1), c)
        moved = float((new - c).abs().max())
        c = new
        if moved < tol:
            break
    return c
