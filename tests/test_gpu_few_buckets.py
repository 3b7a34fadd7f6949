"""Buckets of few destinations against the oracle, bit for bit: items around
the short buckets' 512, a chunk of the ranking waves (768) and its multiples
and the listed sizes' border (2048), destinations around the 64 that a wave
holds, one hub taking most items, masked edges among them."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

ITEMS = [0, 1, 512, 513, 767, 768, 769, 1023, 1536, 1537, 2048, 2049, 2304, 5000]


@pytest.mark.parametrize("dests", [1, 2, 63, 64, 65])
@pytest.mark.parametrize("hub_share", [0.0, 0.9])
def test_few_destinations(dests, hub_share):
    from flashlog_amd.flashlog_kernel import flashlog_kernel as fk
    from oracle import oracle as O
    rng = np.random.default_rng(dests)
    E, R, K = 200_000, 1, 3          # (wide buckets: the destinations share one)
    B, L = len(ITEMS), 1
    m = max(ITEMS)
    src = np.arange(100_000, 100_000 + m, dtype=np.int64)
    dst = rng.integers(0, dests, m).astype(np.int64)
    dst[rng.random(m) < hub_share] = 0
    rel = np.zeros(m, np.int64)
    csr = O.build_csr_structure(src, dst, rel, E)
    mask = (rng.random(m) < 0.9)
    masks = (mask[csr[3]].astype(np.float32), mask[csr[7]].astype(np.float32))
    sb = np.concatenate([np.full(n, i, np.int64) for i, n in enumerate(ITEMS)])
    se = np.concatenate([src[:n] for n in ITEMS])
    sl = np.zeros_like(sb)
    sv = rng.random(sb.size).astype(np.float32)
    w = rng.random((B, L, 2 * R + 1)).astype(np.float32)
    rk, rv = O.sparse_forward(O.SPARSE_TOPK, sb, sl, se, sv, B, L, E, w, csr, masks, R, True, K, -1)
    dev = torch.device("cuda:0")
    tcsr = [torch.from_numpy(np.ascontiguousarray(a)).to(dev) for a in csr]
    vt = torch.from_numpy(sv).to(dev).requires_grad_(True)
    wt = torch.from_numpy(w).to(dev).requires_grad_(True)
    out = fk.FlashLogFunctionSparse3DTopKSum.apply(
        *(torch.from_numpy(x).to(dev) for x in (sb, sl, se)), vt, wt, *tcsr, torch.from_numpy(mask).to(dev), None, B, L,
        E, R, True, K, False, None, True, False)
    idx = out.indices().cpu().numpy()
    np.testing.assert_array_equal((idx[0] * L + idx[1]) * E + idx[2], rk)
    np.testing.assert_array_equal(out.values().detach().cpu().numpy().view(np.int32),
                                  np.asarray(rv, np.float32).view(np.int32))
    # an entry has one edge: its gradient is one product, its output found by the saved map
    g = rng.standard_normal(rk.size).astype(np.float32)
    (out.values() * torch.from_numpy(g).to(dev)).sum().backward()
    at = np.searchsorted(rk, sb * E + dst[se - 100_000])
    want = np.where(mask[se - 100_000], g[np.minimum(at, rk.size - 1)] * w[sb, 0, 0], 0).astype(np.float32)
    np.testing.assert_array_equal(vt.grad.cpu().numpy(), want)
