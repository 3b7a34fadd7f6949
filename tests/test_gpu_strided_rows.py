"""Index rows of a sparse gradient or state that are not contiguous (indices
made as pairs and transposed) give what contiguous ones give."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _coo(shape, n, strided, seed=3):
    """n distinct sorted entries, the index tensor's rows strided or not."""
    g = torch.Generator().manual_seed(seed)
    total = 1
    for s in shape:
        total *= s
    flat = torch.randperm(total, generator=g)[:n].sort().values
    cols = []
    for s in reversed(shape):
        cols.append(flat % s)
        flat = flat // s
    pairs = torch.stack(cols[::-1], 1).cuda()
    idx = pairs.t() if strided else pairs.t().contiguous()
    return torch.sparse_coo_tensor(idx, torch.rand(n, generator=g).cuda() + 0.5, shape, is_coalesced=True)


@pytest.mark.parametrize("shape", [(5, 97), (4, 3, 97)])
@pytest.mark.parametrize("strided_out", [False, True])
@pytest.mark.parametrize("n", [1, 64, 257])
def test_gradient_lookup(shape, strided_out, n):
    from flashlog_amd.flashlog_kernel import flashlog_kernel as fk
    grad = _coo(shape, n, True)
    assert n == 1 or not grad._indices()[0].is_contiguous()
    out = _coo(shape, 200, strided_out, seed=4)._indices()
    got = fk._grad_at_outputs(grad, out, 1 if len(shape) == 2 else shape[1], shape[-1])
    assert torch.equal(got, grad.to_dense()[tuple(out)])


@pytest.mark.parametrize("is_max", [False, True])
def test_rule_accumulation(is_max):
    from flashlog_amd.rules import evaluate, shared_inference
    nb, C, E = 4, 3, 97
    W = torch.rand(2, C, device="cuda").t()
    want = [torch.zeros(2, nb * E, device="cuda") for _ in range(2)]
    got = [torch.zeros(2, nb * E, device="cuda") for _ in range(2)]
    for dense, strided in ((want, False), (got, True)):
        state = _coo((nb, C, E), 300, strided)
        shared_inference._accumulate_chunk(state, W if strided else W.contiguous(), dense[0], is_max, nb, E)
        evaluate._accumulate(state, W if strided else W.contiguous(), dense[1], is_max, nb, E, False)
    assert bool(want[0].any()) and all(torch.equal(a, b) for a, b in zip(want, got))


def _rows(kind, x):
    """The row as a program may hold it: every second element of a larger one, or 32-bit."""
    if kind == "int32":
        return x.to(torch.int32)
    return torch.stack([x, torch.zeros_like(x)], 1)[:, 0]


@pytest.mark.parametrize("kind", ["strided", "int32"])
@pytest.mark.parametrize("L", [1, 3])
def test_normalize_forward(kind, L):
    from flashlog_amd.flashlog_kernel import flashlog_kernel as fk
    mod = fk.get_module()
    B, E = 5, 97
    state = _coo((B, L, E), 300, False)
    b, l, _ = state._indices()
    want = mod.sparse3d_normalize_forward_cuda(b, l, state._values(), B, L, 1e-7)
    got = mod.sparse3d_normalize_forward_cuda(_rows(kind, b), _rows(kind, l), state._values(), B, L, 1e-7)
    assert all(torch.equal(x, y) for x, y in zip(got, want))
    sums = torch.zeros(B * L, dtype=torch.float64, device="cuda").index_add_(0, b * L + l, state._values().double())
    # at most 300 additions of one rounding each
    torch.testing.assert_close(got[1].view(-1).double(), sums, rtol=300 * 2.0 ** -24, atol=0)


@pytest.mark.parametrize("weight_kind", ["strided", "float64", "contiguous", None])
@pytest.mark.parametrize("mask_kind", ["strided", "contiguous", "strided bool"])
def test_apply_mask(mask_kind, weight_kind):
    from flashlog_amd.flashlog_kernel import flashlog_kernel as fk
    n = 1000
    g = torch.Generator().manual_seed(7)
    mask = torch.rand(n, generator=g).cuda()
    if mask_kind == "strided bool":
        mask = mask < 0.5
    weight = torch.randn(n, generator=g).cuda()
    order = torch.randperm(n, generator=g).to(torch.int32).cuda()
    mod = fk.get_module()
    want = mod.apply_mask_cuda(mask, order, weight if weight_kind else None)
    # the factor sigmoid(weight): expf (2 ulp), a sum, a division and the product, one rounding each
    ref = mask[order.long()].double() * (torch.sigmoid(weight[order.long()].double()) if weight_kind else 1)
    torch.testing.assert_close(want.double(), ref, rtol=8 * 2.0 ** -24, atol=0)
    m = mask if mask_kind == "contiguous" else _rows("strided", mask)
    w = {"strided": _rows("strided", weight), "float64": weight.double(), "contiguous": weight, None: None}[weight_kind]
    assert torch.equal(mod.apply_mask_cuda(m, order, w), want)
