"""The walks that run side by side from lists of every node, against the
oracle, bit for bit: sides at the edge of the small lists (16 and 17 groups),
more positive targets than lanes, heads taken in several calls, and the same
walks where the lists of every node do not fit or do not pay."""
import numpy as np
import pytest
import torch

from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _graph():
    """R = 60: node i < 40 has i groups on each side; node 50 has 300 targets
    of relation 2 and no other node has edges of it; node 60 has none."""
    rng = np.random.default_rng(8)
    E, R = 9000, 60
    h, t, r = [], [], []
    for i in range(1, 40):
        rel = rng.choice(np.delete(np.arange(R), 2), i, replace=False)
        h += [np.full(i, i), rng.integers(0, 50, i)]
        t += [rng.integers(0, 50, i), np.full(i, i)]
        r += [rel, rel]
    h += [np.full(300, 50), rng.integers(0, 50, 300)]
    t += [rng.choice(E, 300, replace=False), np.full(300, 50)]
    r += [np.full(300, 2), rng.choice(np.delete(np.arange(R), 2), 300)]
    back = rng.integers(0, E, 20000)
    h.append(back)
    t.append(rng.integers(0, 60, 20000))
    r.append(rng.choice(np.delete(np.arange(R), 2), 20000))
    h, t, r = (np.concatenate(x).astype(np.int64) for x in (h, t, r))
    keep = (h != 60) & (t != 60)
    h, t, r = h[keep], t[keep], r[keep]
    return E, R, O.build_csr_structure(h, t, r, E)


@pytest.mark.parametrize("room", ["all heads", "one head", "hubs", "none", "few walks"])
@pytest.mark.parametrize("ranks,topk,walks,identity", [(3, 200, 301, 0.01), (1, 7, 65, 1.0), (2, 30, 1, 0.0)])
def test_side_by_side_walks(monkeypatch, room, ranks, topk, walks, identity):
    from flashlog_amd.flashlog_kernel.soft_grounding_kernel import soft_grounding_kernel as sg
    E, R, csr = _graph()
    rng = np.random.default_rng(ranks * 100 + topk)
    heads, seeds = [2, R + 5, 2], [3, 2 ** 50 + 1, 77]
    sources = np.concatenate([np.arange(0, 62), rng.integers(0, E, 20)])
    att = rng.random((3, 3, ranks, 2 * R + 1)).astype(np.float32)
    att[att < 0.2] = 0.0
    att[..., 2 * R] = identity * 5  # how often a step stays
    att[..., 2] = np.maximum(att[..., 2], 0.1)
    dev = torch.device("cuda")
    g, _ = sg._graph(tuple(torch.from_numpy(np.asarray(a)) for a in csr), dev, R)
    one = sg._cache_bytes(g, ranks)
    monkeypatch.setattr(sg, "HUB_CACHE_MAX_BYTES", {"all heads": 3 * one, "one head": one, "few walks": 3 * one,
                                                    "hubs": one - 1, "none": 0}[room])
    monkeypatch.setattr(sg, "LISTS_PER_WALK", 0 if room == "few walks" else 1 << 40)
    n = sources.shape[0]
    th = torch.arange(3, dtype=torch.int32).repeat_interleave(n)
    ts = torch.from_numpy(np.tile(sources, 3))
    ti = torch.arange(n).repeat(3)
    keys, pos = sg._walks(g, torch.from_numpy(att), torch.tensor(heads, device=dev), seeds, th, ts, ti, walks, topk,
                          False, 1.0, dev)
    assert (g.nhub == E) == (room in ("all heads", "one head"))
    keys = keys.cpu().numpy().view(np.uint64).reshape(-1, walks)
    pos = pos.cpu().numpy().reshape(-1, walks)
    for i, head in enumerate(heads):
        rk, rp = O.ground_walks(att[i], R, head, sources, np.arange(n), csr, walks, topk, False, seeds[i], 1.0)
        np.testing.assert_array_equal(keys[i * n:(i + 1) * n], rk)
        np.testing.assert_array_equal(pos[i * n:(i + 1) * n], rp)
