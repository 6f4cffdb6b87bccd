"""Row selection of several arrays under one mask (vx_select_count, vx_select_rows) against
x[mask]: the same bits and the same gradients, over lengths around the tiles of 4096, none, some
and all rows, element types and row widths, strided and unaligned inputs, and the forms that
are indexed instead."""
import pytest
import torch

from voxurf_amd.functional import select_rows

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 16, 257, 4095, 4096, 4097, 100003])
@pytest.mark.parametrize("density", [0.0, 0.01, 0.5, 1.0])
def test_equals_indexing(dev, n, density):
    g = torch.Generator(device=dev).manual_seed(n)
    r = lambda *s, dt=torch.float32: torch.randn(*s, generator=g, device=dev, dtype=dt)
    base = torch.rand(n + 1, generator=g, device=dev) < density
    ids = torch.randint(0, 1 << 40, (n,), generator=g, device=dev)
    arrays = [r(n), r(n, 3), ids, r(n, 3, dt=torch.float64), r(3, n).T, r(n, 2, 5), r(2 * n)[::2],
              ids.int()]
    for mask in (base[:n].clone(), base[1:]):  # the second: not 16-byte aligned
        xs = [a.detach().clone() if i not in (4, 6) else a.detach() for i, a in enumerate(arrays)]
        for a in xs:
            if a.is_floating_point() and a.dtype == torch.float32:
                a.requires_grad_(True)
        got, want = select_rows(mask, *xs), [a[mask] for a in xs]
        for a, b in zip(got, want):
            assert a.dtype == b.dtype and a.requires_grad == b.requires_grad and torch.equal(a, b)
        gs = [torch.randn_like(b) for b in want if b.requires_grad]
        leaves = [a for a in xs if a.requires_grad]
        ga = torch.autograd.grad([a for a in got if a.requires_grad], leaves, gs)
        gb = torch.autograd.grad([b for b in want if b.requires_grad], leaves, gs)
        for a, b in zip(ga, gb):
            assert a.shape == b.shape and torch.equal(a, b)


def test_other_forms_are_indexed(dev):
    mask = torch.tensor([True, False, True], device=dev)
    b = torch.tensor([[True], [False], [True]], device=dev)         # one byte a row
    h = torch.arange(3, device=dev, dtype=torch.float16)            # half a word
    for a in (b, h, torch.zeros((3, 0), device=dev)):
        assert torch.equal(select_rows(mask, a)[0], a[mask])
    assert select_rows(mask[:0], torch.zeros(0, device=dev))[0].numel() == 0
    # an unused output's gradient
    x, y = (torch.ones(3, device=dev, requires_grad=True) for _ in range(2))
    u, _ = select_rows(mask, x, y)
    u.sum().backward()
    assert torch.equal(x.grad, mask.float()) and y.grad is None
    with torch.no_grad():
        assert not select_rows(mask, x)[0].requires_grad


def test_differentiated_twice_and_forward(dev):
    """The gradient's gradient and the forward-mode derivative are indexing's."""
    import torch.autograd.forward_ad as fwd
    g = torch.Generator(device=dev).manual_seed(2)
    mask = torch.rand(5000, generator=g, device=dev) < 0.3
    x, y, t = (torch.randn(5000, 3, generator=g, device=dev, requires_grad=True) for _ in range(3))
    res = []
    for pick in (select_rows, lambda m, *a: tuple(v[m] for v in a)):
        a, b = pick(mask, x, y)
        first = torch.autograd.grad((a.pow(3) * b).sum(), (x, y), create_graph=True)
        second = torch.autograd.grad((first[0] * y + first[1].pow(2)).sum(), (x, y))
        with fwd.dual_level():
            a, b = pick(mask, fwd.make_dual(x.detach(), t.detach()), y.detach())
            a, b = fwd.unpack_dual(a), fwd.unpack_dual(b)
        res.append([*first, *second, a.primal, a.tangent, b.primal])
        assert b.tangent is None
    for u, v in zip(*res):
        assert torch.equal(u, v)


def test_unaligned_and_pending_values(dev):
    """Rows of halves from an odd element, and tensors whose conjugation or sign is still to be
    taken, as sources and as gradients."""
    g = torch.Generator(device=dev).manual_seed(4)
    mask = torch.rand(300, generator=g, device=dev) < 0.5
    h = torch.randn(601, generator=g, device=dev).half()[1:].reshape(300, 2)
    assert h.data_ptr() % 4 == 2
    z = torch.randn(300, 2, generator=g, device=dev, dtype=torch.complex64)
    for a in (h, z.conj(), z.conj().imag):
        got, = select_rows(mask, a)
        assert torch.equal(got, a[mask])
        w = a.detach().clone().requires_grad_(True)
        gout = a[mask]
        if a is h:
            gout = torch.cat([gout.new_zeros(1), gout.reshape(-1)])[1:].reshape(gout.shape)
        ga, = torch.autograd.grad(select_rows(mask, w)[0], w, gout)
        gb, = torch.autograd.grad(w[mask], w, gout)
        assert torch.equal(ga, gb)
