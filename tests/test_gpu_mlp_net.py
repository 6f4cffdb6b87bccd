"""The whole-network rgbnet forward (two-way FP16 splits, vx_mlp_net_fwd) against float64 beside
the layer passes whose place it takes where no gradient follows (three-way BF16 splits): root
mean square errors no larger, over the widths, depths and row counts in use and over scales
far from one; and the forms a call can take (row counts around the tiles, a device row count,
values past the input width, rows of zeros, infinities and NaN)."""
import pytest
import torch

from voxurf_amd import mlp_hip
from voxurf_amd._lib import call, lib, ptr, stream_of
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


def _rms(a, b):
    return float((a.double() - b).pow(2).mean().sqrt() / b.pow(2).mean().sqrt())


def _both(dev, din, depth, M, seed, xs=1.0, ws=1.0):
    """The layers' logits, the whole network's, and their float64 values."""
    _, Ws, bs = _net(dev, din, depth, seed, ws)
    st = stream_of(Ws[0])
    x = torch.randn(M, din, device=dev) * xs
    x[:, : din // 2] *= 0.05
    X = mlp_hip.padded_rows(x, din, PREC)
    lg, _ = mlp_hip.forward_rows(X, Ws, bs, PREC, mlp_hip.Packed(Ws, PREC, st), st, bits=[])
    ng = mlp_hip.net_logits(X, Ws, bs, st)
    h = x.double()
    for i, (W, b) in enumerate(zip(Ws, bs)):
        h = h @ W.double().T + b.double()
        if i < len(Ws) - 1:
            h = h.relu()
    return _rms(lg, h), _rms(ng, h)


@pytest.mark.parametrize("din,depth,M", [(42, 4, 100003), (79, 4, 30011), (54, 4, 5000),
                                         (42, 3, 4097), (96, 5, 3001), (64, 4, 1500)])
def test_no_less_accurate_than_the_layers(dev, din, depth, M):
    layers, net = _both(dev, din, depth, M, seed=din + depth)
    print(f"{din} {depth} {M}: layers {layers:.3g}, whole network {net:.3g}")
    assert net <= layers


@pytest.mark.parametrize("xs,ws", [(1e-6, 1.0), (1e6, 1.0), (1.0, 1e-3), (30.0, 20.0)])
def test_scales(dev, xs, ws):
    layers, net = _both(dev, 42, 4, 3000, 7, xs, ws)
    assert net <= layers + 1e-9


@pytest.mark.parametrize("M", [1, 31, 32, 33, 255, 256, 257, 256 * 256 + 1])
def test_row_counts(dev, M):
    """Every row's logits are its own: the same in any batch, with a device row count too, and
    nothing is written past it."""
    _, Ws, bs = _net(dev, 42, 4, 1)
    st = stream_of(Ws[0])
    X = mlp_hip.padded_rows(torch.randn(M + 40, 42, device=dev), 42, PREC)
    whole = mlp_hip.net_logits(X, Ws, bs, st)
    assert torch.equal(whole[:M], mlp_hip.net_logits(X[:M], Ws, bs, st))
    n = torch.tensor([M], dtype=torch.int64, device=dev)
    w_a, b_a = mlp_hip._addresses(Ws[:-1]), mlp_hip._addresses(bs[:-1])
    packed = torch.empty(lib().vx_mlp_pack_half_bytes(3, 42), dtype=torch.uint8, device=dev)
    call("vx_mlp_pack_half", 3, w_a.data_ptr(), 42, ptr(packed), st)
    lg = torch.full((M + 40, 3), 7.0, device=dev)
    call("vx_mlp_net_fwd", 3, 42, ptr(X), 64, M + 40, ptr(packed), b_a.data_ptr(), ptr(Ws[-1]),
         ptr(bs[-1]), ptr(lg), ptr(n), st)
    assert torch.equal(lg[:M], whole[:M]) and bool((lg[M:] == 7.0).all())


def test_values_past_the_input_width(dev):
    """Finite values in the padding change nothing; an infinity or NaN in a row stays in it."""
    _, Ws, bs = _net(dev, 42, 4, 2)
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
    assert b.requires_grad
    assert torch.allclose(a, b.detach(), rtol=1e-5, atol=1e-6)
