"""GPU Lloyd-Max calibration (omni_lloyd_max) and the codec bake.

Pins: the initial codebook (16 equal-count bins of the sorted samples)
equals the bins' correctly rounded means exactly (the radix-select order
statistics and the interval sums); inputs whose answer the mathematics fixes
(16 repeated levels, 16 samples) come out exactly; full runs agree with the
reference's recipe restated on the CPU (oracle.restate.lloyd_max, fp32
torch means) to within the last bits a different summation order allows,
with equal quantization error; the per-head layout, batched groups and
repeated runs agree with each other.
"""
import math

import numpy as np
import pytest
import torch

from oracle import restate
from tests import _data

pytestmark = pytest.mark.gpu


def _bin_means(x: torch.Tensor) -> torch.Tensor:
    xs = np.sort(x.double().numpy())
    bs = xs.size // 16
    return torch.tensor([np.float32(math.fsum(xs[i * bs:(i + 1) * bs]) / bs) for i in range(16)])


def _fit(x, device, **kw):
    from omnistack_rs.quantization import LloydMaxCalibrator
    cal = LloydMaxCalibrator(**kw).fit(x.to(device))
    return cal.codebook.cpu(), int(cal.n_iter.cpu()[0])


@pytest.mark.parametrize("n,dtype", [(20000, torch.float32), (1 << 16 | 7, torch.float32),
                                     (5003, torch.bfloat16), (16 * 50, torch.float16)])
def test_initial_codebook_is_exact_bin_means(device, n, dtype):
    g = _data.gen(400 + n)
    x = torch.randn(n, generator=g) * 2.0
    x[: n // 5] = torch.round(x[: n // 5] * 4) / 4            # many ties, some at bin edges
    x[7] = -0.0
    x = x.to(dtype)
    print(f"[calib] init n={n} {dtype}", flush=True)
    got, iters = _fit(x, device, max_iters=0)
    assert iters == 0
    assert torch.equal(got, _bin_means(x.float()).sort().values)


def test_repeated_levels_are_recovered_exactly(device):
    levels = torch.tensor([-7.5, -3.25, -2.0, -1.5, -1.0, -0.625, -0.25, -0.125,
                           0.0, 0.125, 0.5, 1.0, 1.75, 2.5, 4.0, 9.0])
    x = levels.repeat_interleave(311)[torch.randperm(16 * 311, generator=_data.gen(401))]
    got, iters = _fit(x, device)
    assert torch.equal(got, levels) and iters == 1
    got16, _ = _fit(levels[torch.randperm(16, generator=_data.gen(402))], device)
    assert torch.equal(got16, levels)


@pytest.mark.parametrize("n,scale", [(20000, 1.0), (50000, 0.02), (8192, 30.0)])
def test_full_calibration_matches_reference_recipe(device, n, scale):
    x = torch.randn(n, generator=_data.gen(410 + n)) * scale
    x[: n // 50] *= 8.0                                        # heavy tails, as the outlier channels
    print(f"[calib] full n={n} scale={scale}", flush=True)
    got, iters = _fit(x, device)
    want = restate.lloyd_max(x)
    assert 1 <= iters <= 300
    # the two runs round their means differently and may stop one step
    # apart (each step then moves a centroid by less than tol = 1e-6)
    assert (got - want).abs().max().item() <= 3e-6 + 2e-6 * want.abs().max().item()
    mse = lambda cb: ((x.unsqueeze(1) - cb.unsqueeze(0)).abs().min(dim=1).values ** 2).mean().item()
    assert abs(mse(got) - mse(want)) <= 1e-5 * mse(want)


def test_heads_groups_and_repeats_agree(device):
    from omnistack_rs.quantization import calibrate_heads, calibrate_per_group
    x = torch.randn(3, 4, 50, 128, generator=_data.gen(420))
    x[:, 2] *= 5.0
    xd = x.to(device)
    heads = calibrate_heads(xd).cpu()
    assert heads.shape == (4, 16)
    groups = calibrate_per_group([xd[:, h].reshape(-1) for h in range(4)]).cpu()
    single = torch.stack([_fit(x[:, h].reshape(-1), device)[0] for h in range(4)])
    assert torch.allclose(heads, single, rtol=1e-6, atol=1e-6)
    assert torch.allclose(groups, single, rtol=1e-6, atol=1e-6)
    assert torch.equal(calibrate_heads(xd).cpu(), heads)
    for h in range(4):
        want = restate.lloyd_max(x[:, h].reshape(-1))
        assert (heads[h] - want).abs().max().item() <= 2e-5 * float(x[:, h].abs().max())


def test_calibration_rejects_non_finite(device):
    from omnistack_rs.quantization import calibrate_codebook
    x = torch.randn(100)
    x[3] = float("nan")
    with pytest.raises(ValueError, match="finite"):
        calibrate_codebook(x.to(device))


def test_bake_round_trip_matches_oracle(device, tmp_path):
    from omnistack_rs.bake import BAKE_KEYS, bake_kv_cache, load_bake
    N, H, S, uid = 3, 2, 40, 5
    kv = _data.kv((N, H, S, 128), seed=430, dtype=torch.float32)
    path = tmp_path / "bake.pt"
    nib, qjl, norms, cb, stats = bake_kv_cache(kv, path, seed=uid)
    assert path.exists() and nib.device.type == "cpu"
    assert set(torch.load(path, weights_only=True).keys()) == set(BAKE_KEYS)
    rot = restate.wht(kv)
    for h in range(H):
        want = restate.lloyd_max(rot[:, h].reshape(-1))
        assert (cb[h] - want).abs().max().item() <= 2e-5 * float(rot[:, h].abs().max())
    r_nib, r_qjl, r_norms = restate.quantize_heads(rot, cb, user_id=uid)
    assert torch.equal(nib, r_nib)
    assert (qjl != r_qjl).sum().item() <= 2                   # exact-sign boundary rule
    assert torch.allclose(norms, r_norms, rtol=2.5e-7, atol=0)
    assert stats["compression_ratio"] == round(N * H * S * 128 * 2 / (N * H * S * (64 + 8 + 4)), 3)
    # an existing bake is loaded, not recomputed
    again = bake_kv_cache(None, path)
    assert all(torch.equal(a, b) for a, b in zip(again[:4], (nib, qjl, norms, cb))) and again[4] == stats
    assert load_bake(path)[4] == stats


def test_calibrate_heads_16bit_and_d32_bake(device, tmp_path):
    """bf16 samples calibrate as their fp32 values; a head_dim-32 cache bakes
    and round-trips like the reference's format."""
    from omnistack_rs.bake import bake_kv_cache
    from omnistack_rs.quantization import calibrate_heads
    x = torch.randn(2, 3, 40, 128, generator=_data.gen(440)).to(torch.bfloat16)
    got16 = calibrate_heads(x.to(device)).cpu()
    got32 = calibrate_heads(x.float().to(device)).cpu()
    assert torch.equal(got16, got32)
    kv = torch.randn(2, 2, 30, 32, generator=_data.gen(441))
    nib, qjl, norms, cb, stats = bake_kv_cache(kv, tmp_path / "d32.pt", seed=3)
    assert nib.shape == (2, 2, 30, 16) and qjl.shape == (2, 2, 30, 2) and cb.shape == (2, 16)
    r_nib, _, _ = restate.quantize_heads(restate.wht(kv), cb, user_id=3)
    assert torch.equal(nib, r_nib)
    assert stats["seq_len"] == 30 and stats["n_kv_heads"] == 2


def _step(x: torch.Tensor, c: torch.Tensor) -> torch.Tensor:
    """One Lloyd step by its definition: first-index argmin of the fp32
    distances, correctly rounded means (math.fsum), empty cells kept."""
    out = c.clone()
    code = torch.empty(x.numel(), dtype=torch.int64)
    for s in range(0, x.numel(), 1 << 18):
        code[s:s + (1 << 18)] = (x[s:s + (1 << 18), None] - c[None, :]).abs().argmin(dim=1)
    for k in range(16):
        m = x[code == k].double().numpy()
        if m.size:
            out[k] = float(np.float32(math.fsum(m) / m.size))
    return out


@pytest.mark.parametrize("kind", ["n16", "n17", "one_run", "run_plus_1", "odd_rows", "full_bins", "zeros", "outliers",
                                  "close_levels", "tiny", "bf16_large", "f16", "one_outlier", "cluster", "bf16_close"])
def test_steps_match_their_definition(device, kind):
    """Steps 1, 2 and 3 from the library's own initial centroids, at the edges
    of the binned passes: the smallest groups, a block's run of 32768 samples
    and one more, rows that are no multiple of four, bins with more samples
    than a wave keeps in registers, values so far out or levels so close that
    distances to several centroids round to a tie (steps by bins: one sample
    with a centroid of its own, half the samples within 1e-6 of each other,
    levels an ulp apart), denormals, 16-bit types (one value per bin)."""
    g = _data.gen(450)
    n = {"n16": 16, "n17": 17, "one_run": 32768, "run_plus_1": 32769, "odd_rows": 3 * 4099}.get(kind, 50000)
    x = torch.randn(n, generator=g)
    if kind == "full_bins":
        x[: 3 * n // 4] = 1.0 + torch.rand(3 * n // 4, generator=g) * 2.0 ** -14     # one narrow bump
    elif kind == "zeros":
        x[torch.rand(n, generator=g) < 0.7] = 0.0
        x[5] = -0.0
    elif kind == "outliers":
        x[:4000] *= 1e30
    elif kind == "close_levels":
        x = 1.0 + torch.randint(0, 20, (n,), generator=g) * 2.0 ** -23
    elif kind == "one_outlier":
        x[1234] = 1e8
    elif kind == "cluster":
        x = torch.where(torch.rand(n, generator=g) < 0.9, 1e-6 * torch.rand(n, generator=g), 100 * torch.rand(n, generator=g))
    elif kind == "bf16_close":
        x = (1.0 + torch.randint(0, 24, (n,), generator=g) * 2.0 ** -7).to(torch.bfloat16)
        x[77] = 3e30
    elif kind == "tiny":
        x *= 1e-39
    elif kind == "bf16_large":
        x = torch.randn(200003, generator=g).to(torch.bfloat16)
    elif kind == "f16":
        x = x.to(torch.float16)
    from omnistack_rs.quantization.codebook import _lloyd_max_hip
    if kind == "odd_rows":                         # 3 rows of 4099 in a wider array, 2 groups
        wide = torch.randn(3, 2, 4099 + 2, generator=g)
        wide[:, 1, :4099] = x.reshape(3, 4099)
        args = (wide.to(device), 2, 3, 4099, 2 * 4101, 4101)
    else:
        args = (x.to(device), 1, 1, x.numel(), 0, 0)
    print(f"[calib] steps {kind} n={x.numel()}", flush=True)
    c = _lloyd_max_hip(*args, 0, 1e-6)[0][-1].cpu()
    for it in (1, 2, 3):
        got, done = _lloyd_max_hip(*args, it, 0.0)
        c = _step(x.float(), c)
        assert int(done[-1]) == it
        assert torch.equal(got[-1].cpu(), c.sort().values), f"{kind} step {it}"


@pytest.mark.parametrize("kind,dtype", [("normal", torch.float32), ("ties", torch.float32), ("ties", torch.bfloat16),
                                        ("tiny_n", torch.float16)])
def test_calibration_without_room_for_a_copy(device, kind, dtype, monkeypatch):
    """Where the device cannot hold the stored samples the call runs with the
    least workspace, in place: the same initial centroids and steps (means
    from fp64 sums of another order: one ulp), refused below that size."""
    from omnistack_rs import _lib
    from omnistack_rs.quantization.codebook import _lloyd_max_hip
    L = _lib.lib()
    n = 17 if kind == "tiny_n" else 60001
    x = torch.randn(2, n, generator=_data.gen(480))
    if kind == "ties":
        x = torch.round(x * 4) / 4 + 0.125
    x = x.to(dtype).to(device)
    args = (x, 2, 1, n, 0, n)
    want = [_lloyd_max_hip(*args, it, 0.0) for it in (0, 1, 40)]
    least = L.omni_lloyd_max_workspace_least(2, 1, n)
    assert 0 < least <= L.omni_lloyd_max_workspace_size(2, 1, n) and least < 1 << 18
    monkeypatch.setattr(L, "omni_lloyd_max_workspace_size", lambda *a: 1 << 50)      # more than any device has
    got = [_lloyd_max_hip(*args, it, 0.0) for it in (0, 1, 40)]
    for (c0, i0), (c1, i1), steps in zip(want, got, (0, 1, 40)):
        assert i0.tolist() == i1.tolist() == [steps] * 2
        assert torch.allclose(c0, c1, rtol=2.0 ** -23 if steps < 2 else 1e-6, atol=1e-9 if steps < 2 else 1e-6)
    out = torch.empty(2, 16, device=device)
    ws = torch.empty(least, dtype=torch.uint8, device=device)
    rc = L.omni_lloyd_max(_lib.ptr(x), _lib.dtype_code(dtype), 2, 1, n, 0, n, 1, 0.0, _lib.ptr(out), None, _lib.ptr(ws),
                          least - 1, _lib.stream_of(device))
    assert rc == _lib.OMNI_EWORKSPACE


def test_an_outlier_does_not_slow_the_steps(device):
    """One sample per head so far out that it keeps a centroid to itself puts
    every distance up to it beyond the other centroids' gaps: each step then
    codes bins, not 1.6 M samples one by one (which took thousands of times a
    plain step)."""
    from omnistack_rs.quantization.codebook import _lloyd_max_hip
    n, steps = 1638400, 24
    x = torch.randn(8, n, generator=torch.Generator(device=device).manual_seed(470), device=device)

    def seconds(x):
        times = []
        for _ in range(4):
            e = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
            e[0].record()
            _, done = _lloyd_max_hip(x, 8, 1, n, 0, n, steps, 0.0)
            e[1].record()
            torch.cuda.synchronize()
            assert done.tolist() == [steps] * 8
            times.append(e[0].elapsed_time(e[1]))
        return min(times)

    plain = seconds(x)
    x[:, 5] = 1e8
    far = seconds(x)
    print(f"[calib] {steps} steps: {plain:.3f} ms, with an outlier a head {far:.3f} ms", flush=True)
    assert far < 8 * plain
