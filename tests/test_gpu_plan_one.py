"""Hops around the entries and rows up to which a plan's sums are taken by one
workgroup (4096 of each): forward and gradients against the oracle, in order
of the entries and, from 4096 entries, of their sources."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests.helpers import assert_grad_close, attention, bits, masks_for, small_graph, to_torch_csr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,L,nnz", [(1, 1, 1), (40, 2, 4095), (40, 2, 4096), (40, 2, 4097), (4095, 1, 300), (2048, 2, 4096),
                                     (4097, 1, 300), (4097, 1, 5000)])
@pytest.mark.parametrize("K", [3, 1 << 60])
def test_plan_borders(B, L, nnz, K):
    from flashlog_amd.flashlog_kernel import flashlog_kernel as fk
    rng = np.random.default_rng(nnz + B)
    h, r, t, E, R, csr = small_graph(1, 0.1)
    key = np.sort(rng.choice(B * L * E, nnz, replace=False))
    b, l, e = key // (L * E), key // E % L, key % E
    v = rng.random(nnz).astype(np.float32)
    n = 2 * R + 1
    w = attention(B * L, n, rng).reshape(B, L, n)
    mbool, masks = masks_for(csr, h.shape[0], rng, drop=0.1)
    keys, vals = O.sparse_forward(O.SPARSE_TOPK, b, l, e, v, B, L, E, w, csr, masks, R, False, K, -1)
    dev = torch.device("cuda:0")
    vt = torch.from_numpy(v).to(dev).requires_grad_(True)
    wt = torch.from_numpy(w).to(dev).requires_grad_(True)
    out = fk.FlashLogFunctionSparse3DTopKSum.apply(
        *(torch.from_numpy(x).to(dev) for x in (b, l, e)), vt, wt, *to_torch_csr(csr, dev), torch.from_numpy(mbool).to(dev),
        None, B, L, E, R, False, K, False, None, True, False)
    idx = out.indices().cpu().numpy()
    np.testing.assert_array_equal((idx[0] * L + idx[1]) * E + idx[2], keys)
    np.testing.assert_array_equal(bits(out.values().detach().cpu().numpy()), bits(np.asarray(vals, np.float32)))
    g = rng.standard_normal(keys.size).astype(np.float32)
    (out.values() * torch.from_numpy(g).to(dev)).sum().backward()
    gv, gw = O.sparse_backward(O.SPARSE_TOPK, b, l, e, v, B, L, E, w, csr, masks, R, keys, g, False, K)
    assert_grad_close(vt.grad.cpu().numpy(), gv)
    assert_grad_close(wt.grad.reshape(B * L, n).cpu().numpy(), gw)
