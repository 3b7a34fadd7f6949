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
