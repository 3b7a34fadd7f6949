"""The first hop of a batch: few one-hot entries, many attention weights."""
import numpy as np
import pytest
import torch

from tests.helpers import to_torch_csr

pytestmark = pytest.mark.gpu


def _hop(B, R, w, E=500):
    from flashlog_amd.flashlog_kernel import flashlog_kernel as fk
    from oracle import oracle as O
    rng = np.random.default_rng(B)
    m = 2000
    h, t, r = rng.integers(0, E, m), rng.integers(0, E, m), rng.integers(0, R, m)
    csr = to_torch_csr(O.build_csr_structure(h, t, r, E), torch.device("cuda"))
    L = w.shape[1]
    b = torch.arange(B, device="cuda").repeat_interleave(L)
    l = torch.arange(L, device="cuda").repeat(B)
    e = torch.randint(0, E, (B * L,), generator=torch.Generator("cuda").manual_seed(1), device="cuda")
    v = torch.ones(B * L, device="cuda")
    mask = torch.ones(m, dtype=torch.bool, device="cuda")
    return lambda: fk.FlashLogFunctionSparse3DTopKSum.apply(b, l, e, v, w, *csr, mask, None, B, L, E, R, False, 20, False,
                                                            None, True, False)


@pytest.mark.parametrize("B,L,R", [(1, 1, 5), (4, 2, 127), (32, 3, 237), (256, 3, 822)])
def test_non_finite_attention_is_found(B, L, R):
    """Wherever it is: at the ends and around the first threads' and workgroups' shares of the weights."""
    n = 2 * R + 1
    w = torch.rand(B, L, n, device="cuda")
    hop = _hop(B, R, w)
    hop()
    flat = w.view(-1)
    total = flat.numel()
    for at in sorted({0, 1, 255, 256, 1023, 1024, total // 2, total - 257, total - 2, total - 1}):
        if not 0 <= at < total:
            continue
        keep = float(flat[at])
        for bad in (float("nan"), float("-inf")):
            flat[at] = bad
            with pytest.raises(RuntimeError, match="non-finite"):
                hop()
        flat[at] = keep
    hop()


def test_checks_of_many_weights_fill_the_chip():
    """256 queries of 822 relations, one entry a row: 1.26 million weights and 768 entries.  One pass over the weights
    takes some microseconds on the whole chip; on the few workgroups that the entries need it took 300."""
    from flashlog_amd import _lib
    hop = _hop(256, 822, torch.rand(256, 3, 1645, device="cuda"))
    for _ in range(3):
        hop()
    torch.cuda.synchronize()
    _lib.prof_enable(True)
    try:
        for _ in range(10):
            hop()
        ms, launches = _lib.prof_read("k_sp_prep")
    finally:
        _lib.prof_enable(False)
    assert launches == 10 and ms / launches < 0.1  # (of its own 9 us)
