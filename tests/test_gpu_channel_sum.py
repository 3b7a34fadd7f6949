"""Channel sum of a coalesced [B, L, E] state (the models' sum_sp_3d,
src/model_DRUM_kernel_sp.py:22-28) through the C-ABI: indices, value bits
and gradients against torch's coalesce of the (b, e) re-index on the GPU
(what the reference runs) and against the oracle."""
import numpy as np
import pytest
import torch

from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _fk():
    from flashlog_amd.flashlog_kernel import flashlog_kernel as fk
    return fk


def _state(seed, B, L, E, n, order_cases=False):
    rng = np.random.default_rng(seed)
    keys = np.unique(rng.choice(B * L * E, size=n, replace=False))
    b, l, e = keys // (L * E), (keys // E) % L, keys % E
    v = rng.random(b.shape[0]).astype(np.float32)
    if order_cases:  # large and small values on one (b, e): rounding depends on the channel order
        big = rng.random(b.shape[0]) < 0.3
        v[big] *= np.float32(1e7)
        v[(~big) & (rng.random(b.shape[0]) < 0.3)] *= np.float32(-1.0)
    return b, l, e, v


def _torch_sum(b, e, v, B, E, dev):
    t = torch.sparse_coo_tensor(torch.stack([b, e]), v, [B, E]).coalesce()
    return t


@pytest.mark.parametrize("B,L,E,n,seed", [
    (4, 3, 60, 300, 0),         # most (b, e) in several channels
    (16, 3, 5000, 20000, 1),
    (8, 1, 1000, 3000, 2),      # one channel: a copy
    (8, 5, 200, 6000, 3),       # dense: nearly every (b, e) in all channels
    (4, 8, 400, 9000, 5),       # many channels: every entry ranked in seven other rows
    (6, 10, 300, 12000, 6),
    (256, 3, 4_600_000, 3_000_000, 4),
])
def test_channel_sum_bitexact(B, L, E, n, seed):
    fk = _fk()
    dev = torch.device("cuda:0")
    b, l, e, v = _state(seed, B, L, E, n, order_cases=True)
    tb, tl, te = (torch.from_numpy(x).to(dev) for x in (b, l, e))
    vt = torch.from_numpy(v).to(dev).requires_grad_(True)
    s = torch.sparse_coo_tensor(torch.stack([tb, tl, te]), vt, [B, L, E], is_coalesced=True)
    got = fk.sum_sp_3d(s)
    vr = vt.detach().clone().requires_grad_(True)
    ref = _torch_sum(tb, te, vr, B, E, dev)
    assert got.is_coalesced() and tuple(got.shape) == (B, E)
    assert torch.equal(got.indices(), ref.indices())
    assert torch.equal(got.values().detach().view(torch.int32), ref.values().detach().view(torch.int32))
    if n <= 20000:
        ob, oe, ov, _ = O.sum_sp_3d(b, l, e, v, B, L, E)
        assert np.array_equal(got.indices().cpu().numpy(), np.stack([ob, oe]))
        assert np.array_equal(got.values().detach().cpu().numpy().view(np.int32), ov.view(np.int32))
    g = torch.randn(ref.values().shape[0], device=dev)
    (got.values() * g).sum().backward()
    (ref.values() * g).sum().backward()
    assert torch.equal(vt.grad, vr.grad)


def test_channel_sum_empty_and_errors():
    fk = _fk()
    dev = torch.device("cuda:0")
    z = torch.zeros((3, 0), dtype=torch.int64, device=dev)
    s = torch.sparse_coo_tensor(z, torch.zeros(0, device=dev), [2, 3, 10], is_coalesced=True)
    got = fk.sum_sp_3d(s)
    assert got.values().numel() == 0 and tuple(got.shape) == (2, 10)
    # marked coalesced, but the entities of row (0, 1) decrease: refused
    idx = torch.tensor([[0, 0, 0], [1, 1, 2], [5, 3, 1]], device=dev)
    bad = torch.sparse_coo_tensor(idx, torch.ones(3, device=dev), [1, 3, 10], is_coalesced=True)
    with pytest.raises(ValueError):
        fk.sum_sp_3d(bad)


def _reference_max_sp_3d(s):
    # the reference's steps (src/model_mmDRUM_kernel_sp.py:17-32) in torch
    s = s.coalesce()
    idx, val = s.indices(), s.values()
    B, _, E = s.shape
    flat_key = idx[0] * E + idx[2]
    order = torch.argsort(flat_key)
    flat_key, val = flat_key[order], val[order]
    uniq, inv = torch.unique_consecutive(flat_key, return_inverse=True)
    out_val = torch.zeros(uniq.shape[0], device=val.device, dtype=val.dtype)
    out_val = out_val.scatter_reduce(0, inv, val, reduce="amax", include_self=False)
    return torch.sparse_coo_tensor(torch.stack([uniq // E, uniq % E]), out_val, [B, E]).coalesce()


@pytest.mark.parametrize("B,L,E,n,seed", [(4, 3, 60, 300, 10), (16, 3, 5000, 20000, 11), (8, 5, 200, 6000, 12),
                                          (256, 3, 4_600_000, 2_000_000, 13)])
def test_channel_max_matches_reference_steps(B, L, E, n, seed):
    fk = _fk()
    dev = torch.device("cuda:0")
    b, l, e, _ = _state(seed, B, L, E, n)
    rng = np.random.default_rng(seed)
    v = (rng.integers(0, 6, b.shape[0]) / 8.0).astype(np.float32)  # ties and exact zeros
    tb, tl, te = (torch.from_numpy(x).to(dev) for x in (b, l, e))
    vt = torch.from_numpy(v).to(dev).requires_grad_(True)
    vr = vt.detach().clone().requires_grad_(True)
    got = fk.max_sp_3d(torch.sparse_coo_tensor(torch.stack([tb, tl, te]), vt, [B, L, E], is_coalesced=True))
    ref = _reference_max_sp_3d(torch.sparse_coo_tensor(torch.stack([tb, tl, te]), vr, [B, L, E]))
    assert torch.equal(got.indices(), ref.indices())
    assert torch.equal(got.values().detach().view(torch.int32), ref.values().detach().view(torch.int32))
    g = torch.randn(ref.values().shape[0], device=dev)
    (got.values() * g).sum().backward()
    (ref.values() * g).sum().backward()
    assert torch.equal(vt.grad.view(torch.int32), vr.grad.view(torch.int32))


@pytest.mark.parametrize("seed", [21, 22])
def test_channel_max_special_values(seed):
    """NaN and +-inf inside (b, e) groups: value bits and the amax gradient
    split as the reference's scatter_reduce steps give them.  (A group
    holding both -0.0 and +0.0 has no fixed reference: torch's atomic amax
    keeps whichever zero it stores first, so such ties are left out.)"""
    fk = _fk()
    dev = torch.device("cuda:0")
    B, L, E, n = 4, 3, 40, 240
    b, l, e, _ = _state(seed, B, L, E, n)
    rng = np.random.default_rng(seed)
    v = (rng.integers(-3, 4, b.shape[0]) / 4.0).astype(np.float32)
    specials = np.array([np.nan, np.inf, -np.inf], dtype=np.float32)
    pick = rng.choice(b.shape[0], size=min(40, b.shape[0]), replace=False)
    v[pick] = specials[rng.integers(0, specials.shape[0], pick.shape[0])]
    tb, tl, te = (torch.from_numpy(x).to(dev) for x in (b, l, e))
    vt = torch.from_numpy(v).to(dev).requires_grad_(True)
    vr = vt.detach().clone().requires_grad_(True)
    got = fk.max_sp_3d(torch.sparse_coo_tensor(torch.stack([tb, tl, te]), vt, [B, L, E], is_coalesced=True))
    ref = _reference_max_sp_3d(torch.sparse_coo_tensor(torch.stack([tb, tl, te]), vr, [B, L, E]))
    assert torch.equal(got.indices(), ref.indices())
    assert torch.equal(got.values().detach().view(torch.int32), ref.values().detach().view(torch.int32))
    g = torch.randn(ref.values().shape[0], device=dev)
    (got.values() * g).sum().backward()
    (ref.values() * g).sum().backward()
    assert torch.equal(vt.grad.view(torch.int32), vr.grad.view(torch.int32))


def _channel_case(seed, ties=False):
    dev = torch.device("cuda:0")
    B, L, E = 4, 3, 60
    b, l, e, v = _state(seed, B, L, E, 300)
    if ties:
        v = (np.random.default_rng(seed).integers(1, 6, b.size) / 8.0).astype(np.float32)
    idx = torch.stack([torch.from_numpy(x).to(dev) for x in (b, l, e)])
    return B, L, E, idx, torch.from_numpy(v).to(dev)


@pytest.mark.parametrize("op", ["sum", "max"])
@pytest.mark.parametrize("how", ["to_dense", "dense", "other pattern", "uncoalesced", "empty", "strided"])
def test_gradients_of_other_forms(op, how):
    """A gradient that is dense, or sparse with other entries than the output, gives what its value at every output
    gives: 0 where it has none."""
    fk = _fk()
    B, L, E, idx, v = _channel_case(31, ties=op == "max")
    reduce = fk.sum_sp_3d if op == "sum" else fk.max_sp_3d
    g = torch.randn(B, E, generator=torch.Generator().manual_seed(5)).cuda()
    if how == "other pattern":   # every third cell, and some that the output does not have
        g = g * (torch.arange(B * E, device="cuda").view(B, E) % 3 == 0)
        up = g.to_sparse()
    elif how == "uncoalesced":   # halves, each cell twice: exact sums
        half = (g * 0.5).to_sparse()
        up = torch.sparse_coo_tensor(half.indices().repeat(1, 2), half.values().repeat(2), (B, E))
    elif how == "empty":
        g = torch.zeros_like(g)
        up = g.to_sparse()
    elif how == "strided":
        full = g.to_sparse()
        up = torch.sparse_coo_tensor(full.indices().t().contiguous().t(), full.values(), (B, E), is_coalesced=True)
    vr = v.clone().requires_grad_(True)
    ref = _torch_sum(idx[0], idx[2], vr, B, E, None) if op == "sum" else \
        _reference_max_sp_3d(torch.sparse_coo_tensor(idx, vr, (B, L, E)))
    want, = torch.autograd.grad(ref.values(), [vr], g[tuple(ref.indices())])
    vt = v.clone().requires_grad_(True)
    out = reduce(torch.sparse_coo_tensor(idx, vt, (B, L, E), is_coalesced=True))
    if how == "to_dense":
        got, = torch.autograd.grad(out.to_dense(), [vt], g)
    elif how == "dense":
        ctx_grad = fk._channel_grad(g, out.indices(), E)
        assert torch.equal(ctx_grad, g[tuple(out.indices())])
        return
    else:
        got, = torch.autograd.grad(out, [vt], up)
    assert torch.equal(got, want)


@pytest.mark.parametrize("op", ["sum", "max"])
@pytest.mark.parametrize("form", ["values", "dense"])
def test_second_derivative(op, form):
    """A gradient with a graph of its own: its derivative by the upstream gradient."""
    fk = _fk()
    B, L, E, idx, v = _channel_case(32, ties=op == "max")
    reduce = fk.Sparse3DChannelSumFunction if op == "sum" else fk.Sparse3DChannelMaxFunction
    vt = v.clone().requires_grad_(True)
    out = reduce.apply(*idx, vt, B, L, E)  # (torch's own backward of a sparse state's values is not differentiable)
    y = out.values() if form == "values" else out.to_dense()
    u = torch.randn_like(y.detach()).requires_grad_(True)
    gv, = torch.autograd.grad(y, [vt], u, create_graph=True)
    p = torch.randn_like(gv)
    got, = torch.autograd.grad(gv, [u], p)
    # gv is linear in u: its transpose, from the same backward on every unit of u in turn
    at = out.indices() if form == "values" else None
    vr = v.clone().requires_grad_(True)
    dense = torch.zeros(B, L, E, dtype=torch.float64, device="cuda").index_put(tuple(idx), vr.double())
    share = torch.autograd.grad(dense.sum(1) if op == "sum" else dense.amax(1), [vr],
                                torch.ones(B, E, dtype=torch.float64, device="cuda"))[0].double()
    want = torch.zeros(B, E, dtype=torch.float64, device="cuda").index_put((idx[0], idx[2]), share * p.double(),
                                                                          accumulate=True)
    want = want[tuple(at)] if at is not None else want
    # at most three float32 products and additions
    torch.testing.assert_close(got.double(), want, rtol=6 * 2.0 ** -24, atol=6 * 2.0 ** -24 * float(p.abs().max()))
