"""Buckets of the sparse max against the oracle, bit for bit: items around the
512 of a wave and the 2048 above which dense arrays take every bucket,
destinations around the 64 of a wave, buckets of 64 to 8192 entities (dense
arrays serve those of up to 1024 for all sizes), ties, masked edges, and NaN
among the values: first of its destination's items or later."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

ITEMS = [0, 1, 64, 65, 128, 129, 256, 257, 511, 512, 513, 2047, 2048, 2049, 5000]
MAX_BUCKETS, BUCKET_ITEMS = 1022, 16  # buckets a row, items a bucket on average (the hop's rule for their width)


def _shift(E, rows, items):
    s = 6
    while s < 13 and -(-E >> s) > MAX_BUCKETS:
        s += 1
    while s < 13 and -(-E >> s) > 1 and rows * -(-E >> s) * BUCKET_ITEMS > items:
        s += 1
    return s


@pytest.mark.parametrize("E,filler,width", [(60_000, 400_000, 6), (1_046_528, 400_000, 10), (1_046_529, 400_000, 11),
                                            (900_000, 0, 13), (50, 0, 6)])
@pytest.mark.parametrize("dests", [1, 64, 65, 300])
@pytest.mark.parametrize("nan", [False, True])
def test_max_buckets(E, filler, width, dests, nan):
    from flashlog_amd.flashlog_kernel import flashlog_kernel as fk
    from oracle import oracle as O
    rng = np.random.default_rng(dests + width)
    m = max(ITEMS)
    if E == 50:  # fewer entities than one bucket has: every source has many edges
        dests, base, nsrc = min(dests, 49), 0, 49
    else:        # destinations 0 .. dests, then sources of one edge each, then the filler's destinations
        base, nsrc = E // 2, m
    src = base + np.arange(m, dtype=np.int64) % nsrc
    dst = rng.integers(0, dests, m).astype(np.int64)
    dst[rng.random(m) < 0.3] = 0
    fsrc = np.full(filler, base + m, np.int64)   # one entry of the last row fills the row's buckets
    h, t = np.concatenate([src, fsrc]), np.concatenate([dst, np.arange(filler) * 2 % E])
    r = np.concatenate([rng.integers(0, 2, m), np.zeros(filler, np.int64)])
    R, L, B = 2, 1, len(ITEMS) + (1 if filler else 0)
    csr = O.build_csr_structure(h, t, r, E)
    mask = rng.random(h.size) < 0.9
    masks = (mask[csr[3]].astype(np.float32), mask[csr[7]].astype(np.float32))
    ents = [np.unique(src[:n]) for n in ITEMS] + ([fsrc[:1]] if filler else [])
    sb = np.concatenate([np.full(x.size, i, np.int64) for i, x in enumerate(ents)])
    se = np.concatenate(ents)
    sl = np.zeros_like(sb)
    sv = (rng.integers(-4, 5, sb.size) / 4).astype(np.float32)  # many ties, zeros of both signs by the weights
    if nan:
        sv[rng.random(sv.size) < 0.02] = np.nan
        sv[np.unique(sb, return_index=True)[1][::2]] = np.nan   # the first entry of every second row
        sv[-1] = 1.0
    w = (rng.integers(1, 4, (B, L, 2 * R + 1)) / 2).astype(np.float32)
    keys, vals, went, wdir, wpos = O.sparse_max_forward(sb, sl, se, sv, B, L, E, w, csr, masks, R, False, 1 << 60)
    dev = torch.device("cuda:0")
    tcsr = [torch.from_numpy(np.ascontiguousarray(a)).to(dev) for a in csr]
    vt = torch.from_numpy(sv).to(dev).requires_grad_(True)
    wt = torch.from_numpy(w).to(dev).requires_grad_(True)
    fk.plan_log = []
    try:
        out = fk.FlashLogFunctionSparse3DTopKMax.apply(
            *(torch.from_numpy(x).to(dev) for x in (sb, sl, se)), vt, wt, *tcsr, torch.from_numpy(mask).to(dev), None, B,
            L, E, R, False, 1 << 60, False, None, True, False)
        assert _shift(E, B * L, fk.plan_log[0]["items"]) == width
    finally:
        fk.plan_log = None
    idx = out.indices().cpu().numpy()
    np.testing.assert_array_equal((idx[0] * L + idx[1]) * E + idx[2], keys)
    got = out.values().detach().cpu().numpy()
    np.testing.assert_array_equal(np.isnan(got), np.isnan(vals))
    some = ~np.isnan(vals)
    np.testing.assert_array_equal(got[some].view(np.int32), vals[some].view(np.int32))
    assert not nan or (~some).any()
    # every output's gradient goes to its winner: whole numbers times small powers of two, exact in any order
    g = rng.integers(-8, 9, keys.size).astype(np.float32)
    (out.values() * torch.from_numpy(g).to(dev)).sum().backward()
    gv, _ = O.sparse_max_backward(sb, sl, sv, B, L, w, csr, masks, R, g, went, wdir, wpos)
    np.testing.assert_array_equal(vt.grad.cpu().numpy(), gv)
