"""The normalizer's row sums against the sequential float32 sum, bit for bit:
lengths around the 32 values read at once and the staged chunk, ties, sums
that cross many binades, zeros, subnormals, and rows with negative or
non-finite values."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _rows(kind, rng):
    lengths = [0, 1, 31, 32, 33, 63, 64, 65, 96, 2047, 2048, 2049, 2080, 4095, 4096, 4097, 20011]
    out = []
    for n in lengths:
        if kind == "uniform":
            v = rng.random(n)
        elif kind == "lognormal":
            v = np.exp(8 * rng.standard_normal(n))
        elif kind == "ties":      # small multiples of powers of two: many exact halves
            v = rng.integers(0, 4, n) * 2.0 ** rng.integers(-3, 1, n)
            if n:
                v[0] = 2.0 ** 22
        elif kind == "odd ties":  # an odd sum plus exact halves of its ulp, over and over
            v = np.full(n, 0.5)
            if n:
                v[0] = 2.0 ** 23 + 1
        elif kind == "growing":   # every few values a new binade
            v = 2.0 ** (np.arange(n) % 240 - 120.0) * (1 + rng.random(n))
        elif kind == "doubling":
            v = 2.0 ** np.minimum(np.arange(n) - 140.0, 100)
        elif kind == "zeros":
            v = np.where(rng.random(n) < 0.9, 0.0, rng.random(n))
            v[:n // 2] = 0
            v = np.where(rng.random(n) < 0.5, -0.0, v) if n else v
        elif kind == "subnormal":
            v = rng.random(n) * 1e-41
        elif kind == "huge":
            v = rng.random(n) * 1e37
        else:
            v = rng.random(n)
            if n:
                at = rng.integers(0, n, 3)
                v[at] = {"negative": -0.3, "nan": np.nan, "inf": np.inf, "mixed inf": np.inf}[kind]
                if kind == "mixed inf":
                    v[at[0]] = -np.inf
        out.append(v.astype(np.float32))
    return out


@pytest.mark.parametrize("kind", ["uniform", "lognormal", "ties", "odd ties", "growing", "doubling", "zeros",
                                  "subnormal", "huge", "negative", "nan", "inf", "mixed inf"])
def test_row_sums(kind):
    from flashlog_amd.flashlog_kernel import flashlog_kernel as fk
    rng = np.random.default_rng(len(kind))
    rows = _rows(kind, rng)
    B = len(rows)
    b = np.concatenate([np.full(r.size, i, np.int64) for i, r in enumerate(rows)])
    v = np.concatenate(rows)
    mod = fk.get_module()
    out, denom, start, end = mod.sparse3d_normalize_forward_cuda(
        torch.from_numpy(b).cuda(), torch.zeros(b.size, dtype=torch.int64).cuda(), torch.from_numpy(v).cuda(), B, 1, 1e-7)
    with np.errstate(all="ignore"):
        # numpy's cumsum adds one by one in float32; the fold starts from +0
        want = np.array([np.cumsum(np.concatenate([[np.float32(0)], r]), dtype=np.float32)[-1] for r in rows],
                        np.float32)
        clamp = np.where(want >= np.float32(1e-7), want, np.float32(1e-7))
        scaled = (v / clamp[b]).astype(np.float32)
    got = denom.view(-1).cpu().numpy()
    nan = np.isnan(want)
    np.testing.assert_array_equal(np.isnan(got), nan)
    np.testing.assert_array_equal(got[~nan].view(np.int32), want[~nan].view(np.int32))
    np.testing.assert_array_equal(out.cpu().numpy(), scaled)
    np.testing.assert_array_equal((end - start).cpu().numpy(), [r.size for r in rows])


@pytest.mark.parametrize("B,L", [(4096, 1), (1365, 3), (4097, 1), (1366, 3), (40_000, 5)])
def test_many_rows(B, L):
    """Row counts around the most whose workgroups find their own rows; empty rows at both ends and between."""
    from flashlog_amd.flashlog_kernel import flashlog_kernel as fk
    rng = np.random.default_rng(B)
    sizes = rng.integers(0, 5, B * L)
    sizes[:2] = sizes[-1:] = 0
    row = np.repeat(np.arange(B * L), sizes)
    v = rng.random(row.size).astype(np.float32)
    mod = fk.get_module()
    out, denom, start, end = mod.sparse3d_normalize_forward_cuda(
        *(torch.from_numpy(x).cuda() for x in (row // L, row % L, v)), B, L, 1e-7)
    want = np.zeros(B * L, np.float32)
    first = np.cumsum(sizes) - sizes
    for k in range(4):  # one by one, as the fold adds them
        has = sizes > k
        want[has] += v[first[has] + k]
    np.testing.assert_array_equal(denom.view(-1).cpu().numpy(), want)
    np.testing.assert_array_equal(start.cpu().numpy(), first)
    np.testing.assert_array_equal((end - start).cpu().numpy(), sizes)
    np.testing.assert_array_equal(out.cpu().numpy(), v / np.maximum(want, np.float32(1e-7))[row])


def test_many_rows_find_their_entries_at_once():
    """200,000 rows of four values, two thousand workgroups of which run at a time: found one by one by these, the rows
    took five times as long as the normalizer now takes."""
    from flashlog_amd.flashlog_kernel import flashlog_kernel as fk
    rows = torch.arange(800_000, device="cuda") // 4
    v = torch.rand(800_000, device="cuda")
    mod = fk.get_module()
    times = []
    for _ in range(8):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        mod.sparse3d_normalize_forward_cuda(rows, torch.zeros_like(rows), v, 200_000, 1, 1e-7)
        b.record()
        b.synchronize()
        times.append(a.elapsed_time(b))
    assert min(times) < 0.45  # ms (of its own 0.15)
