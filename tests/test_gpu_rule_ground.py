"""Rule scoring with every chunk grounded by one launch, bit for bit against
the same call grounded operator by operator (a hook object with this
package's own steps), and against the float64 oracle: states at the edge of
the hash table, states that outgrow it, path counts and rows beyond the
kernels' limits, a pool that is too small, and entity counts around the
largest the accumulators hold."""
import types

import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests.helpers import to_torch_csr

pytestmark = pytest.mark.gpu


def _score(ev, *a, **k):
    from flashlog_amd.rules import shared_inference as si
    return si.score(ev, *a, **k)


def _stepwise():
    from flashlog_amd.rules import evaluate as ev
    return types.SimpleNamespace(
        initial_rule_state=ev.initial_rule_state,
        vectorized_operation_sparse3d_fixed_relation=ev.vectorized_operation_sparse3d_fixed_relation,
        advance_single_rule_state_memory_bounded=ev.advance_single_rule_state_memory_bounded)


def _graph(E, fans, pairs=()):
    """Relation i: node i to fans[i] distinct nodes; relation len(fans): node
    j to j + 1; then the edges (h, relation, t) of pairs."""
    rng = np.random.default_rng(5)
    h, r, t = [np.arange(E - 1)], [np.full(E - 1, len(fans))], [np.arange(1, E)]
    for i, n in enumerate(fans):
        h.append(np.full(n, i))
        r.append(np.full(n, i))
        t.append(rng.choice(E, n, replace=False))
    for a, b, c in pairs:
        h.append(np.asarray(a))
        r.append(np.full(len(a), b))
        t.append(np.asarray(c))
    return tuple(np.concatenate(x).astype(np.int64) for x in (h, r, t))


def _both(E, R, trip, sources, bodies, one_launch=True, monkeypatch=None, oracle=True, **kw):
    from flashlog_amd.rules import shared_inference as si
    h, r, t = trip
    tc = to_torch_csr(O.build_csr_structure(h, t, r, E), torch.device("cuda"))
    W = np.random.default_rng(9).random((len(bodies), 2)).astype(np.float32)
    rules = [{"body": b, "rank_weights": [float(x) for x in w]} for b, w in zip(bodies, W)]
    src = torch.tensor(sources).cuda()
    used = []
    real = si._score_in_one_launch
    if monkeypatch is not None:
        monkeypatch.setattr(si, "_score_in_one_launch", lambda *a: used.append(real(*a)) or used[-1])
    got = _score(None, src, rules, tc, R, E, 5, **kw)
    assert not one_launch or used == [] or used[0] is not None
    want = _score(_stepwise(), src, rules, tc, R, E, 5, **kw)
    assert torch.equal(got.indices(), want.indices()) and torch.equal(got.values(), want.values())
    if oracle:
        ref = O.rule_scores(h, r, t, E, R, sources, bodies, W.astype(np.float64), kw.get("reduction", "sum"),
                            kw.get("boolean_paths", False), kw.get("final_max", False))
        # two float32 divisions and at most len(bodies) + 2 additions and products per score
        np.testing.assert_allclose(got.to_dense().cpu().numpy(), ref, rtol=(len(bodies) + 6) * 2.0 ** -24, atol=1e-30)
    return used


@pytest.mark.parametrize("kw", [{}, {"boolean_paths": True}, {"reduction": "max"},
                                {"reduction": "max", "final_max": True}])
@pytest.mark.parametrize("E", [1700, 16384, 16385])
def test_state_sizes(monkeypatch, E, kw):
    """Endpoints just below, at and above the hash table's 1536, and repeated
    paths to one endpoint."""
    fans = [0, 1, 63, 64, 128, 129, 1535, 1536, 1537, 1600]
    R = len(fans) + 3
    back = np.arange(200)
    trip = _graph(E, fans, [(back, R - 2, np.full(200, 3)), (np.full(200, 3), R - 1, back)])
    bodies = [[i] for i in range(len(fans))] + [[i, len(fans)] for i in range(len(fans))]
    bodies += [[2 * R], [], [R - 1, R - 2, R - 1], [R + 3, 4, 2 * R], [R - 1, 2 * R, R - 2], [R + R - 2, R - 2],
               [9, len(fans), R + len(fans)]]
    used = _both(E, R, trip, [0, 1, 2, 3, 6, 7, 8, 9, 9, E - 1], bodies, monkeypatch=monkeypatch, **kw)
    assert (used != []) == (E <= 16384)


@pytest.mark.parametrize("case", ["paths", "edges", "pool"])
def test_beyond_the_limits(monkeypatch, case):
    from flashlog_amd.rules import shared_inference as si
    if case == "pool":
        E, R = 1700, 3
        monkeypatch.setattr(si, "_POOL_ENTRIES", 100)
        trip = _graph(E, [700])
        bodies = [[0], [0, 1]]
    elif case == "paths":
        # 300 parallel edges there, back and there again: 300^3 paths above 2^24
        E, R = 500, 3
        trip = _graph(E, [2], [(np.full(300, 7), 2, np.full(300, 8))])
        bodies = [[2], [2, R + 2], [2, R + 2, 2]]
    else:
        # one row of 2^20 + 1 edges in a step
        E, R = 3000, 3
        n = (1 << 20) + 1
        trip = _graph(E, [2], [(np.full(n, 7), 2, np.arange(n) % E)])
        bodies = [[2], [1, 2]]
    used = _both(E, R, trip, [0, 7, 8], bodies, one_launch=False, monkeypatch=monkeypatch, oracle=case != "edges")
    assert used == [None]


def test_source_outside():
    E, R = 400, 3
    h, r, t = _graph(E, [2])
    tc = to_torch_csr(O.build_csr_structure(h, t, r, E), torch.device("cuda"))
    from flashlog_amd.rules import shared_inference as si
    ops = torch.tensor([[0]]).cuda()
    W = torch.ones(1, 1).cuda()
    with pytest.raises(ValueError, match="out of range"):
        si._score_in_one_launch(torch.tensor([1, E]).cuda(), [(0, 1)], ops, [1], W, tc, R, E, 2, False, False, False,
                                {"chunks": 0, "ground_calls": 0})


@pytest.mark.parametrize("sources,block", [([0], None), ([0, 1, 5, 1], None), ([0, 1, 5, 0], 1), ([0, 5], 1)])
def test_no_scores(sources, block):
    """Bodies that begin at a source and end nowhere: calls, and blocks of a
    call, without one scored entity."""
    E, R = 50, 3
    trip = _graph(E, [2], [([1], 2, [7])])
    kw = {} if block is None else {"dense_budget_bytes": block * 2 * E * 4}
    # (nodes 0 and 5 have no edge of relation 2, and no node has one of it twice)
    _both(E, R, trip, sources, [[1, 2, 2], [0, R, 2, 2], [2]], **kw)
    _both(E, R, trip, [0, 5], [[1, 2, 2], [2, 2]], **kw)


def _hub(E, n):
    """Node 7 with n edges of relation 2; relation 1: node j to j + 1; relation 0: node 0 to two nodes."""
    return _graph(E, [2], [(np.full(n, 7), 2, np.arange(n) % E)])


def _counted_steps(monkeypatch):
    """The calls of the step-by-step form, of this package's own hooks too."""
    from flashlog_amd.flashlog_kernel import flashlog_kernel as fk
    from flashlog_amd.rules import evaluate as ev
    calls = []
    real = fk.vectorized_operation_sparse3d_fixed_relation

    def step(*a, **k):
        calls.append(a[0].shape)
        return real(*a, **k)

    monkeypatch.setattr(fk, "vectorized_operation_sparse3d_fixed_relation", step)
    monkeypatch.setattr(ev, "vectorized_operation_sparse3d_fixed_relation", step)
    return calls


@pytest.mark.parametrize("at", [0, 7, 19])
@pytest.mark.parametrize("block", [None, 2])
def test_what_was_grounded_before_a_limit_is_kept(monkeypatch, at, block):
    """20 rules in chunks of 5, one of them with a row beyond the limits: the chunks (and blocks of sources) before it
    are not grounded again."""
    E, R = 3000, 3
    h, r, t = _hub(E, (1 << 20) + 1)
    tc = to_torch_csr(O.build_csr_structure(h, t, r, E), torch.device("cuda"))
    bodies = [[1, 1]] * 20
    bodies[at] = [2]
    W = np.random.default_rng(9).random((20, 2)).astype(np.float32)
    rules = [{"body": b, "rank_weights": [float(x) for x in w]} for b, w in zip(bodies, W)]
    src = torch.tensor([3, 4, 5, 6, 7, 9]).cuda()  # node 7 in the third block of two
    kw = {} if block is None else {"dense_budget_bytes": block * 2 * E * 4}
    want_stats, stats = {}, {}
    want = _score(_stepwise(), src, rules, tc, R, E, 5, stats=want_stats, **kw)
    calls = _counted_steps(monkeypatch)
    got = _score(None, src, rules, tc, R, E, 5, stats=stats, **kw)
    assert torch.equal(got.indices(), want.indices()) and torch.equal(got.values(), want.values())
    assert stats == want_stats
    assert len(calls) == 2 * (4 - at // 5)  # (every chunk has a body of two steps)


@pytest.mark.parametrize("entries,fits", [(1400, True), (700, True), (175, True), (174, False)])
def test_pool_grows(monkeypatch, entries, fits):
    """Two final states of 700 entities each: the pool is made as large as they ask for, up to eight times."""
    from flashlog_amd.rules import shared_inference as si
    E, R = 1700, 3
    monkeypatch.setattr(si, "_POOL_ENTRIES", entries)
    calls = _counted_steps(monkeypatch)
    h, r, t = _graph(E, [700], [([5], 2, [6])])
    tc = to_torch_csr(O.build_csr_structure(h, t, r, E), torch.device("cuda"))
    rules = [{"body": b, "rank_weights": [0.5, 0.25]} for b in ([2], [2], [2], [2], [2], [0], [0])]
    got = _score(None, torch.tensor([0, 5]).cuda(), rules, tc, R, E, 5)
    assert (calls == []) == fits
    want = _score(_stepwise(), torch.tensor([0, 5]).cuda(), rules, tc, R, E, 5)
    assert torch.equal(got.indices(), want.indices()) and torch.equal(got.values(), want.values())


def test_rows_after_a_limit_are_left():
    """Chunks behind one that outgrew the kernels are not walked."""
    from flashlog_amd import _lib
    E, R = 3000, 4
    n = 1 << 19
    h, r, t = _hub(E, (1 << 20) + 1)
    h, r, t = np.concatenate([h, np.full(n, 7)]), np.concatenate([r, np.full(n, 3)]), np.concatenate([t, np.arange(n) % E])
    tc = to_torch_csr(O.build_csr_structure(h, t, r, E), torch.device("cuda"))

    def walked(bodies):
        rules = [{"body": b, "rank_weights": [0.5]} for b in bodies]
        run = lambda: _score(None, torch.tensor([7]).cuda(), rules, tc, R, E, 1)
        run()
        _lib.prof_enable(True)
        try:
            run()
            return _lib.prof_read("k_rg_rows")[0] + _lib.prof_read("k_rg_dense")[0]
        finally:
            _lib.prof_enable(False)

    assert walked([[2]] + [[3]] * 4) < walked([[3]])


@pytest.mark.parametrize("kw", [{}, {"reduction": "max"}])
@pytest.mark.parametrize("block", [None, 1])
def test_stats_are_those_of_the_steps(kw, block):
    """Steps whose states are all empty are not counted, also where a row dies late, only in the dense form, or where a
    chunk's longest body is not its last to die."""
    E, R = 1700, 5
    h, r, t = _graph(E, [1600, 3], [([0], 3, [7]), ([7], 4, [8])])
    tc = to_torch_csr(O.build_csr_structure(h, t, r, E), torch.device("cuda"))
    kw = dict(kw) if block is None else dict(kw, dense_budget_bytes=block * 2 * E * 4)
    for bodies in ([[3, 3, 3]], [[3, 3, 3], [3]], [[3, 4, 4]], [[3], []], [[0, 0, 2]], [[0, 2, 3, 4]], [[0, 2], [3, 3, 3]],
                   [[3, 2 * R, 3, 3]], [[3, 4]] * 5 + [[3, 3, 2]] * 5 + [[1]], [[3, 2 * R + 3, 0]]):
        rules = [{"body": b, "rank_weights": [0.5, 0.25]} for b in bodies]
        want, got = {}, {}
        a = _score(_stepwise(), torch.tensor([0, 7]).cuda(), rules, tc, R, E, 5, stats=want, **kw)
        b = _score(None, torch.tensor([0, 7]).cuda(), rules, tc, R, E, 5, stats=got, **kw)
        assert torch.equal(a.indices(), b.indices()) and torch.equal(a.values(), b.values())
        assert got == want, bodies


def test_out_of_memory_is_counted(monkeypatch):
    from flashlog_amd.rules import shared_inference as si

    def full(*a):
        raise torch.cuda.OutOfMemoryError("full")

    monkeypatch.setattr(si, "_score_in_one_launch", full)
    E, R = 50, 3
    h, r, t = _graph(E, [2])
    tc = to_torch_csr(O.build_csr_structure(h, t, r, E), torch.device("cuda"))
    stats = {}
    got = _score(None, torch.tensor([0, 1]).cuda(), [{"body": [0], "rank_weights": [0.5]}], tc, R, E, 5, stats=stats)
    assert got._nnz() == 2 and stats["oom_retries"] == 1
