"""Dense filtered ranks from pairs as they come: duplicates, any order, the
targets among them, rows of every alignment, no pairs, and indices out of
range, against the oracle (whole counts: equal)."""
import numpy as np
import pytest
import torch

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,E,n", [(1, 1, 0), (1, 5, 7), (3, 257, 1), (7, 1022, 5000), (64, 3001, 63), (5, 40001, 31)])
@pytest.mark.parametrize("use_eql", [False, True])
@pytest.mark.parametrize("filtered", [False, True])
def test_ranks_from_pairs(B, E, n, use_eql, filtered):
    from flashlog_amd.flashlog_kernel import flashlog_kernel as fk
    rng = np.random.default_rng(B * 1000 + n)
    state = np.round(rng.random((B, E)) * 5).astype(np.float32)
    state[rng.random((B, E)) < 0.3] = 0
    if E > 3:
        state[0, 1], state[B - 1, 2], state[0, 3] = np.nan, np.inf, -np.inf
    targets = rng.integers(0, E, B)
    fb, fe = rng.integers(0, B, n), rng.integers(0, min(E, 50), n)
    got = fk.dense_filtered_ranks_cuda(torch.from_numpy(state).cuda(), torch.from_numpy(targets).cuda(),
                                       (torch.from_numpy(fb).cuda(), torch.from_numpy(fe).int().cuda()) if filtered
                                       else None, use_eql)
    want = O.dense_filtered_ranks(state, targets, fb if filtered else None, fe if filtered else None, use_eql)
    np.testing.assert_array_equal(got.cpu().numpy(), want)


@pytest.mark.parametrize("target,pair,message", [(10, (0, 0), "target"), (-1, (0, 0), "target"),
                                                 (3, (2, 0), "filter"), (3, (0, 10), "filter"), (3, (-1, 4), "filter"),
                                                 (3, (1, -1), "filter"), (10, (9, 9), "target")])
def test_out_of_range(target, pair, message):
    from flashlog_amd.flashlog_kernel import flashlog_kernel as fk
    state = torch.rand(2, 10, device="cuda")
    with pytest.raises(ValueError, match=message + ".* out of range"):
        fk.dense_filtered_ranks_cuda(state, torch.tensor([1, target]).cuda(),
                                     (torch.tensor([pair[0]]).cuda(), torch.tensor([pair[1]]).cuda()))


@pytest.mark.parametrize("B,E,pairs,message", [(0, 10, 1, "filter index out of range"), (2, 0, 0, "target out of range"),
                                               (0, 0, 0, None), (0, 10, 0, None)])
def test_empty_scores(B, E, pairs, message):
    """No query or no entity: every index given is out of range."""
    from flashlog_amd.flashlog_kernel import flashlog_kernel as fk
    z = torch.zeros(pairs, dtype=torch.long, device="cuda")
    args = torch.zeros(B, E, device="cuda"), torch.zeros(B, dtype=torch.long, device="cuda"), (z, z)
    if message is None:
        assert fk.dense_filtered_ranks_cuda(*args).shape == (0,)
    else:
        with pytest.raises(ValueError, match=message):
            fk.dense_filtered_ranks_cuda(*args)


def test_shapes_of_filter_and_targets():
    """A filter needs flat targets and pairs of equal length."""
    from flashlog_amd.flashlog_kernel import flashlog_kernel as fk
    state, t = torch.rand(2, 10, device="cuda"), torch.zeros(2, dtype=torch.long, device="cuda")
    for targets, pair in ((t[:, None], (t, t)), (t, (t, t[:1])), (t, (t[:, None], t[:, None]))):
        with pytest.raises(ValueError, match="1D"):
            fk.dense_filtered_ranks_cuda(state, targets, pair)


@pytest.mark.parametrize("order", ["in runs", "mixed"])
def test_pairs_given_many_times(order):
    """A few pairs, each given thousands of times, are counted once."""
    from flashlog_amd.flashlog_kernel import flashlog_kernel as fk
    B, E = 7, 300
    g = torch.Generator().manual_seed(3)
    scores = torch.randint(0, 5, (B, E), generator=g).float().cuda()
    targets = torch.randint(0, E, (B,), generator=g).cuda()
    fb, fe = torch.randint(0, B, (9,), generator=g), torch.randint(0, E, (9,), generator=g)
    want = fk.dense_filtered_ranks_cuda(scores, targets, (fb.cuda(), fe.cuda()), True)
    pick = torch.randint(0, 9, (20_000,), generator=g)
    if order == "in runs":
        pick = pick.sort().values
    got = fk.dense_filtered_ranks_cuda(scores, targets, (fb[pick].cuda(), fe[pick].cuda()), True)
    assert torch.equal(got, want)


def test_one_pair_given_many_times_is_not_slow():
    """Every one of 20,000 threads put the same pair into the table: 200 us of atomics on one word."""
    from flashlog_amd import _lib
    from flashlog_amd.flashlog_kernel import flashlog_kernel as fk
    B, E = 509, 14500
    scores = torch.rand(B, E, device="cuda")
    targets = torch.zeros(B, dtype=torch.int64, device="cuda")
    pair = torch.zeros(20_000, dtype=torch.int64, device="cuda")
    fk.dense_filtered_ranks_cuda(scores, targets, (pair, pair))
    _lib.prof_enable(True)
    try:
        for _ in range(10):
            fk.dense_filtered_ranks_cuda(scores, targets, (pair, pair))
        ms, launches = _lib.prof_read("k_dr_filter")
    finally:
        _lib.prof_enable(False)
    assert launches == 10 and ms / launches < 0.07


@pytest.mark.parametrize("B,E,n", [(1, 5, 0), (3, 257, 40), (64, 3001, 2000)])
@pytest.mark.parametrize("use_eql", [False, True])
def test_sorted_keys(B, E, n, use_eql):
    """The C entry that takes the filter as sorted unique keys, targets among them."""
    from flashlog_amd import _lib
    from flashlog_amd.flashlog_kernel import flashlog_kernel as fk
    g = torch.Generator().manual_seed(n)
    state = (torch.randint(0, 6, (B, E), generator=g) / 4).float().cuda()
    targets = torch.randint(0, E, (B,), generator=g).cuda()
    fb, fe = torch.randint(0, B, (n,), generator=g).cuda(), torch.randint(0, E, (n,), generator=g).cuda()
    keys = torch.unique(torch.cat([fb * E + fe, torch.arange(B, device="cuda") * E + targets]))
    ranks = torch.empty(B, device="cuda")
    _lib.check(_lib.lib().fl_dense_filtered_ranks(fk._stream(state), _lib.ptr(state), _lib.ptr(targets), _lib.ptr(keys),
                                                  keys.numel(), B, E, 1 if use_eql else 0, _lib.ptr(ranks)), "ranks")
    assert torch.equal(ranks, fk.dense_filtered_ranks_cuda(state, targets, (fb, fe), use_eql))
