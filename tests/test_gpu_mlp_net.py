"""The whole-network rgbnet forward (vx_mlp_net_fwd), which takes the place of the layer passes
where no gradient follows: the same logits as theirs, bit for bit, over the widths, depths and
row counts in use, scales far from one, rows and weights whose entries lie many powers of ten
apart, zeros, infinities and NaN; and the forms a call can take (row counts around the tiles, a
device row count, values past the input width)."""
import pytest
import torch

from voxurf_amd import mlp_hip
from voxurf_amd._lib import call, ptr, stream_of
from voxurf_amd.mlp import RgbNet

pytestmark = pytest.mark.gpu
PREC = mlp_hip.PREC_F32_SPLIT


def _net(dev, din, depth, seed, scale=1.0):
    torch.manual_seed(seed)
    net = RgbNet(din, 192, depth).to(dev)
    with torch.no_grad():
        for l in net.linears():
            l.bias.uniform_(-0.1, 0.1)
            l.weight.mul_(scale)
    return net, [l.weight.detach().contiguous() for l in net.linears()], \
        [l.bias.detach().contiguous() for l in net.linears()]


def _same(net, x):
    """The logits without a gradient to follow, shown to be those with one."""
    with torch.no_grad():
        a = net(x)
    b = net(x)
    assert b.requires_grad and not a.requires_grad
    assert torch.equal(torch.nan_to_num(a, nan=77.0), torch.nan_to_num(b.detach(), nan=77.0))
    return a


def _rows(dev, M, din, spread, seed):
    """Rows whose columns are scaled by powers of ten between 1 and `spread`."""
    g = torch.Generator().manual_seed(seed)
    x = torch.randn((M, din), generator=g)
    x[:, :din // 2] *= 0.05
    return (x * 10.0 ** (torch.rand(din, generator=g) * torch.log10(torch.tensor(spread)))).to(dev)


@pytest.mark.parametrize("din,depth,M", [(42, 4, 100003), (79, 4, 30011), (54, 4, 5000),
                                         (42, 3, 4097), (96, 5, 3001), (64, 4, 1500), (1, 4, 700)])
@pytest.mark.parametrize("spread", [1.0, 1e4, 1e8, 1e12])
def test_the_layers_logits(dev, din, depth, M, spread):
    net, Ws, _ = _net(dev, din, depth, din + depth)
    with torch.no_grad():
        g = torch.Generator().manual_seed(M)
        w = net.linears()[1].weight
        w *= (10.0 ** (-torch.rand(192, generator=g) * torch.log10(torch.tensor(spread)))).to(dev)
    a = _same(net, _rows(dev, M, din, spread, M))
    assert bool(torch.isfinite(a).all()) and float(a.abs().max()) > 0


@pytest.mark.parametrize("xs,ws", [(1e-6, 1.0), (1e6, 1.0), (1.0, 1e-3), (30.0, 20.0), (1e-30, 1.0)])
def test_scales(dev, xs, ws):
    net, _, _ = _net(dev, 42, 4, 7, ws)
    _same(net, _rows(dev, 3000, 42, 20.0, 7) * xs)


@pytest.mark.parametrize("large", [1e4, 1e8, 1e20])
def test_an_entry_whose_weights_are_zero(dev, large):
    """However large, it adds nothing and takes no bit from the others (the products with zero
    are exact): the logits are those beside an entry of one."""
    net, _, _ = _net(dev, 42, 4, 11)
    with torch.no_grad():
        net.linears()[0].weight[:, 5] = 0.0
    x = _rows(dev, 3000, 42, 1.0, 3)
    x[:, 5] = 1.0
    want = _same(net, x)
    x[:, 5] = large
    assert torch.equal(_same(net, x), want)


@pytest.mark.parametrize("M", [1, 31, 32, 33, 255, 256, 257, 256 * 256 + 1])
def test_row_counts(dev, M):
    """Every row's logits are its own: the same in any batch, with a device row count too, and
    nothing is written past it."""
    _, Ws, bs = _net(dev, 42, 4, 1)
    st = stream_of(Ws[0])
    X = mlp_hip.padded_rows(torch.randn(M + 40, 42, device=dev), 42, PREC)
    packed = mlp_hip.Packed(Ws, PREC, st)
    whole = mlp_hip.net_logits(X, Ws, bs, st)
    assert torch.equal(whole, mlp_hip.forward_rows(X, Ws, bs, PREC, packed, st)[0])
    assert torch.equal(whole[:M], mlp_hip.net_logits(X[:M], Ws, bs, st))
    n = torch.tensor([M], dtype=torch.int64, device=dev)
    b_a = torch.tensor([b.data_ptr() for b in bs[:-1]], dtype=torch.int64)
    lg = torch.full((M + 40, 3), 7.0, device=dev)
    call("vx_mlp_net_fwd", 3, 42, ptr(X), 64, M + 40, ptr(packed.buf), b_a.data_ptr(), ptr(Ws[-1]),
         ptr(bs[-1]), ptr(lg), ptr(n), st)
    assert torch.equal(lg[:M], whole[:M]) and bool((lg[M:] == 7.0).all())


def test_values_past_the_input_width(dev):
    """Finite values in the padding change nothing; an infinity or NaN in a row stays in it, and
    comes out as the layers' passes have it."""
    net, Ws, bs = _net(dev, 42, 4, 2)
    st = stream_of(Ws[0])
    x = torch.randn(700, 42, device=dev)
    x[5] = 0
    X = mlp_hip.padded_rows(x, 42, PREC)
    want = mlp_hip.net_logits(X, Ws, bs, st)
    Y = X.clone()
    Y[:, 42:] = torch.randn(700, 22, device=dev) * 1e20
    Y[3, 7], Y[9, 0] = float("nan"), float("inf")
    got = mlp_hip.net_logits(Y, Ws, bs, st)
    ok = torch.ones(700, dtype=torch.bool, device=dev)
    ok[3] = ok[9] = False
    assert torch.equal(got[ok], want[ok])
    _same(net, Y[:, :42].contiguous())


def test_gradient_free_calls_keep_no_activations(dev):
    net, Ws, _ = _net(dev, 42, 4, 3)
    x = torch.randn(50000, 42, device=dev)
    with torch.no_grad():
        net(x)
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        base = torch.cuda.memory_allocated()
        a = net(x)
        # the padded rows, the logits and the packed weights, no [50000, 192] buffer
        assert torch.cuda.max_memory_allocated() - base < 50000 * 192 * 4
    b = net(x)
    assert b.requires_grad and torch.equal(a, b.detach())
