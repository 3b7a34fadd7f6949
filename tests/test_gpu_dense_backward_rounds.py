"""The dense sum's backward at the edges of its rounds, against the oracle:
sources of 1 to 130 edges (items are added 64 at a time, groups cross the
rounds), more groups than a wave has lanes, zero upstream gradients among
them, and rows whose pairs fill one chunk of partials exactly, one less and
one more (8192 floats)."""
import numpy as np
import pytest
import torch

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("R", [1, 3, 20, 70])
@pytest.mark.parametrize("K", [0, 40])
def test_rounds(R, K):
    from flashlog_amd.flashlog_kernel import flashlog_kernel as fk
    rng = np.random.default_rng(10 * R + K)
    n = 2 * R + 1
    per_chunk = 8192 // n
    degs = np.array([1, 3, 4, 5, 15, 16, 17, 63, 64, 65, 127, 128, 130])
    E = max(per_chunk + 2, 400) + 200
    src = np.concatenate([np.full(d, i) for i, d in enumerate(degs)])
    dst = np.concatenate([rng.choice(np.arange(200, E), d, replace=False) for d in degs])
    rel = rng.integers(0, R, src.size)
    csr = O.build_csr_structure(src, dst, rel, E)
    counts = [len(degs), min(per_chunk - 1, E), min(per_chunk, E), min(per_chunk + 1, E)]
    BL = len(counts)
    A = np.zeros((BL, E), np.float32)
    for b, c in enumerate(counts):
        at = np.arange(len(degs)) if b == 0 else np.concatenate(
            [np.arange(len(degs)), rng.choice(np.arange(len(degs), E), max(c - len(degs), 0), replace=False)])
        A[b, at] = 0.1 + rng.random(at.size)
    w = (0.05 + rng.random((BL, n))).astype(np.float32)
    mask = (rng.random(src.size) < 0.9).astype(np.float32)
    masks = (mask[csr[3]], mask[csr[7]])
    g = [rng.standard_normal((BL, E)).astype(np.float32) for _ in range(3)]
    g[1][rng.random((BL, E)) < 0.3] = 0.0
    kk = K if K > 0 else (1 << 60)
    gA_ref, gw_ref = O.dense_backward(*g, A, w, csr, masks, R, wot_i=False, topk_edges=kk)
    dev = torch.device("cuda")
    tcsr = tuple(torch.from_numpy(np.ascontiguousarray(a)).to(dev) for a in csr)
    At = torch.from_numpy(A).to(dev).view(BL, 1, E).requires_grad_(True)
    wt = torch.from_numpy(w).to(dev).view(BL, 1, n).requires_grad_(True)
    mk = tuple(torch.from_numpy(m).to(dev) for m in masks)
    outs = fk.dense_csr_sum_cuda(At, wt, tcsr, None, R, use_topk=K > 0, topk_nodes=E, topk_edges=K, prepared_masks=mk)
    sum((o * torch.from_numpy(x).to(dev).view(BL, 1, E)).sum() for o, x in zip(outs, g)).backward()
    gA = At.grad.reshape(BL, E).cpu().numpy()
    np.testing.assert_array_equal(gA.view(np.int32), gA_ref.view(np.int32))
    # the oracle adds grad_w's terms in another order: at most 8192 terms a
    # column, each sum within terms * 2^-24 of the terms' absolute sum
    _, bound = O.dense_backward(*[np.abs(x) for x in g], A, w, csr, masks, R, wot_i=False, topk_edges=kk)
    got = wt.grad.reshape(BL, n).cpu().numpy()
    assert (np.abs(got - gw_ref) <= 2 * 8192 * 2.0 ** -24 * np.abs(bound) + 1e-30).all()
