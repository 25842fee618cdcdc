"""Dense attention on dequantized tensors (omni_dense_attn) against the
restated reference (oracle.restate.reference_attn, attention/reference.py:
72-177, fp32 torch on the CPU), and the reference's unfused path
(_fused_attn_python, fused_attention.py:435-466: dequantize_heads +
reference_attn) against the restated one.

Bar: fp32 results within 2e-6 absolute + 2e-5 relative (the same sums in a
different order); NaN exactly where the reference's tile loop produces NaN
(a row whose first tile is fully masked, a NaN score), output in q's dtype.
"""
import math

import pytest
import torch

from oracle import restate
from tests import _data
from tests._checks import graph_times

pytestmark = pytest.mark.gpu


def _close(got, want, tag):
    g, w = got.cpu().float(), want.float()
    assert torch.equal(torch.isnan(g), torch.isnan(w)), f"{tag}: NaN pattern differs"
    fin = ~torch.isnan(w)
    d = (g[fin] - w[fin]).abs()
    lim = 2e-6 + 2e-5 * w[fin].abs()
    print(f"[dense] {tag}: max {d.max().item() if d.numel() else 0:.3e}", flush=True)
    assert bool((d <= lim).all()), f"{tag}: max {d.max().item():.3e}"


@pytest.mark.parametrize("B,Hq,Hkv,T,S,D", [
    (2, 8, 2, 5, 300, 128), (1, 4, 4, 1, 33, 128), (2, 32, 8, 3, 100, 64), (1, 6, 3, 70, 40, 32),
    (1, 2, 1, 2, 129, 256), (3, 4, 2, 1, 1, 128), (2, 16, 2, 2, 200, 32), (1, 8, 1, 2, 77, 128),
])
def test_dense_attn_matches_oracle(device, B, Hq, Hkv, T, S, D):
    from omnistack_rs.attention import reference_attn
    g = _data.gen(500 + S + D)
    q = torch.randn(B, Hq, T, D, generator=g)
    k = torch.randn(B, Hkv, S, D, generator=g)
    v = torch.randn(B, Hkv, S, D, generator=g)
    got = reference_attn(q.to(device), k.to(device), v.to(device))
    assert got.dtype == torch.float32 and got.shape == (B, Hq, T, D)
    _close(got, restate.reference_attn(q, k, v), f"B{B} Hq{Hq} Hkv{Hkv} T{T} S{S} D{D}")


def test_dense_attn_masks_scale_and_dtype(device):
    from omnistack_rs.attention import reference_attn
    B, Hq, Hkv, T, S, D = 2, 8, 4, 6, 90, 128
    g = _data.gen(510)
    q = torch.randn(B, Hq, T, D, generator=g).to(torch.bfloat16)
    k = torch.randn(B, Hkv, S, D, generator=g)
    v = torch.randn(B, Hkv, S, D, generator=g)
    causal = torch.full((T, S), float("-inf")).triu(S - T + 1)          # (T, S), broadcast over B, H
    got = reference_attn(q.to(device), k.to(device), v.to(device), mask=causal.to(device), scale=0.3)
    assert got.dtype == torch.bfloat16
    want = restate.reference_attn(q, k, v, mask=causal, scale=0.3)
    # both round an fp32 result to bf16: at most one bf16 ulp apart
    assert bool(((got.cpu().float() - want.float()).abs() <= 2 ** -7 * want.float().abs() + 1e-6).all())
    bias = torch.randn(B, 1, T, S, generator=g)                          # per-batch additive bias
    _close(reference_attn(q.float().to(device), k.to(device), v.to(device), mask=bias.to(device)),
           restate.reference_attn(q.float(), k, v, mask=bias), "bias (B,1,T,S)")


@pytest.mark.parametrize("tile_size,T", [(16, 4), (128, 4), (16, 12), (128, 12)])
def test_dense_attn_nan_rules_follow_the_reference(device, tile_size, T):
    """A row whose first tile of keys is all -inf is NaN in the reference's
    loop (exp(-inf - -inf)); later fully masked tiles are harmless; a NaN
    key poisons its rows.  T=4 (8 rows per kv head) runs the key-split
    launch, T=12 (24 rows) the row-split one."""
    from omnistack_rs.attention import reference_attn
    B, Hq, Hkv, S, D = 1, 4, 2, 200, 64
    g = _data.gen(520)
    q = torch.randn(B, Hq, T, D, generator=g)
    k = torch.randn(B, Hkv, S, D, generator=g)
    v = torch.randn(B, Hkv, S, D, generator=g)
    mask = torch.zeros(T, S)
    mask[0, :20] = float("-inf")       # first 20 keys masked for query 0
    mask[1, 40:] = float("-inf")       # only the first 40 visible for query 1
    mask[2, :] = float("-inf")         # nothing visible for query 2
    got = reference_attn(q.to(device), k.to(device), v.to(device), mask=mask.to(device), tile_size=tile_size)
    want = restate.reference_attn(q, k, v, mask=mask, tile_size=tile_size)
    _close(got, want, f"masks tile {tile_size}")
    k2 = k.clone()
    k2[0, 1, 150, 3] = float("nan")    # kv head 1 -> q heads 2, 3 become NaN
    _close(reference_attn(q.to(device), k2.to(device), v.to(device), tile_size=tile_size),
           restate.reference_attn(q, k2, v, tile_size=tile_size), f"nan key tile {tile_size}")


def test_unfused_python_path_matches_oracle(device):
    """_fused_attn_python (dequantize_heads + reference_attn on the device)
    against its restatement."""
    from omnistack_rs.kernels.fused_attention import _fused_attn_python
    from tests.test_gpu_attn import _cache
    B, Hq, Hkv, T, S, uid = 2, 8, 2, 3, 150, 21
    kn, kq, kr, vn, cb = _cache(B, Hkv, S, seed=530, user_id=uid)
    q = _data.query((B, Hq, T, 128), seed=531)
    got = _fused_attn_python(q.to(device), *(t.to(device) for t in (kn, kq, kr, vn, cb)), uid,
                             1 / math.sqrt(128), True)
    want = restate.fused_attn_python(q, kn, kq, kr, vn, cb, uid, 1 / math.sqrt(128), True)
    assert got.dtype == q.dtype
    # both round an fp32 result to q's dtype: at most one ulp apart
    assert bool(((got.cpu().float() - want.float()).abs() <= 2 ** -7 * want.float().abs() + 1e-6).all())


@pytest.mark.parametrize("D", [32, 64, 128, 256])
@pytest.mark.parametrize("T,S", [(4, 1), (5, 31), (17, 32), (16, 33), (300, 65), (1300, 40)])
def test_dense_attn_row_and_key_edges(device, D, T, S):
    """Rows and keys at the edges of 16-row waves and 32-key tiles, on both
    sides of the rule between the launches that split rows and keys (1300
    queries x 8 kv heads: rows), with a causal mask and its column-major copy
    (same values: same bits)."""
    from omnistack_rs.attention import reference_attn
    B, Hq, Hkv = 1, 16, 8
    g = _data.gen(540 + T + S)
    q = torch.randn(B, Hq, T, D, generator=g)
    k, v = torch.randn(B, Hkv, S, D, generator=g), torch.randn(B, Hkv, S, D, generator=g)
    mask = torch.full((T, S), float("-inf")).triu(1) if T >= S else torch.zeros(T, S)
    mask[:, S // 2:] += 0.25
    dev = [t.to(device) for t in (q, k, v)]
    want = restate.reference_attn(q, k, v, mask=mask)
    got = reference_attn(*dev, mask=mask.to(device))
    _close(got, want, f"T{T} S{S} D{D} mask")
    same = torch.equal(got, reference_attn(*dev, mask=mask.t().contiguous().to(device).t()))
    assert same, "column-major mask"
    _close(reference_attn(*dev), restate.reference_attn(q, k, v), f"T{T} S{S} D{D}")


@pytest.mark.parametrize("where,value", [("k", float("nan")), ("k", float("inf")), ("v", float("nan")), ("v", float("-inf")),
                                         ("k", 3e38), ("q", 3e38), ("v", 3e38)])
def test_dense_attn_hidden_tiles(device, where, value):
    """Whole tiles of hidden keys are skipped only where they change nothing:
    a NaN or infinite key or value there, or scores that overflow, give the
    reference's NaN (0 x inf, inf - inf)."""
    from omnistack_rs.attention import reference_attn
    B, Hq, Hkv, T, S, D = 1, 16, 8, 1100, 160, 32
    g = _data.gen(560)
    t = dict(q=torch.randn(B, Hq, T, D, generator=g), k=torch.randn(B, Hkv, S, D, generator=g),
             v=torch.randn(B, Hkv, S, D, generator=g))
    mask = torch.zeros(T, S)
    mask[:, 64:] = float("-inf")               # keys 64 .. 159 hidden from every query
    if where == "q":
        t["q"][0, 3, 5, 7] = value
        t["k"][0, 1, 100:] *= 1e3
    else:
        t[where][0, 1, 100, 3] = value
    want = restate.reference_attn(t["q"], t["k"], t["v"], mask=mask)
    got = reference_attn(*(x.to(device) for x in (t["q"], t["k"], t["v"])), mask=mask.to(device))
    _close(got, want, f"hidden {where} {value}")


@pytest.mark.parametrize("D", [32, 64, 128, 256])
@pytest.mark.parametrize("S", [33, 40, 63, 97])
def test_dense_attn_tail_stays_inside(device, D, S):
    """Keys past S of a last, partly filled tile are not read (row kernel: 24
    query rows, enough heads for it at every head_dim): K and V are followed
    by NaN, which P = 0 would not hide (0 x NaN), and which must not decide
    whether a hidden tile is skipped."""
    from omnistack_rs.attention import reference_attn
    B, H, T = 50, 8, 24
    g = _data.gen(570 + S + D)
    q = torch.randn(B, H, T, D, generator=g)
    k, v = torch.randn(B, H, S, D, generator=g), torch.randn(B, H, S, D, generator=g)
    mask = torch.full((T, S), float("-inf")).triu(S - T + 1)
    mask[:, 32:] = float("-inf")               # the last tiles hidden from every query

    def before_nan(t):
        wide = torch.full((t.numel() + 64 * D,), float("nan"), device=device)
        wide[: t.numel()] = t.to(device).reshape(-1)
        return wide[: t.numel()].view(t.shape)

    dev = (q.to(device), before_nan(k), before_nan(v))
    _close(reference_attn(*dev), restate.reference_attn(q, k, v), f"tail S{S} D{D}")
    _close(reference_attn(*dev, mask=mask.to(device)), restate.reference_attn(q, k, v, mask=mask), f"tail S{S} D{D} mask")


def test_dense_attn_many_blocks(device):
    """More blocks than one grid dimension of 256-thread blocks holds (2^24; a
    launch of more is cut off without an error): sequences of one key, so
    every query row is that key's value.  79 GB."""
    from omnistack_rs.attention import reference_attn
    torch.cuda.empty_cache()
    B, H, T, D = 4096, 4097, 17, 32
    v = torch.randn(B, H, 1, D, generator=torch.Generator(device=device).manual_seed(580), device=device)
    q = torch.zeros(B, H, T, D, device=device)
    out = reference_attn(q, v, v)
    del q
    for b in range(0, B, 512):
        same = torch.equal(out[b:b + 512], v[b:b + 512].expand(-1, -1, T, -1))
        assert same, f"batch {b}"
    del out, v
    torch.cuda.empty_cache()


@pytest.mark.parametrize("D,rows,more,S", [(128, 1024, 1040, 16), (128, 1024, 1040, 64), (64, 1360, 1552, 16)])
def test_dense_attn_few_keys_take_no_longer_than_more_rows(device, D, rows, more, S):
    """Few keys and many rows: the launch that splits the keys (which leaves
    most of its waves idle there) is not taken, so a call takes no longer than
    one with a few rows more, past its rule (31, 23 and 20 % longer with it)."""
    from omnistack_rs.attention import reference_attn
    ts = [[torch.randn(1, 8, m, D, generator=_data.gen(590)).to(device) for m in (n, S, S)] for n in (rows, more)]
    best = graph_times([lambda t=t: reference_attn(*t) for t in ts], 100)
    print(f"[dense] D{D} S{S}: {rows} rows {best[0]:.2f} us, {more} rows {best[1]:.2f} us", flush=True)
    assert best[0] < 1.1 * best[1]
