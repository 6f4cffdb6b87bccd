"""The adjoint of the dense central differences (vx_dense_sdf_gradient_bwd) against a float64
restatement, where its tiles end: rows of whole vectors and not, one to three planes, unaligned
buffers.

The adjoint is six quotients added to the old value: eight roundings of float32 (2^-24) of
terms whose magnitudes are summed for the bound."""
import pytest
import torch

from voxurf_amd._lib import call, dtype_code, ptr, stream_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(1, 1, 1), (2, 3, 4), (3, 2, 5), (17, 5, 64), (5, 33, 31), (40, 64, 132),
                                   (64, 64, 64)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("shift", [0, 1])
def test_dense_gradient_adjoint(dev, shape, dtype, shift):
    X, Y, Z = shape
    n = X * Y * Z
    g = torch.Generator(device=dev).manual_seed(n)
    buf = torch.randn(4 * n + 2 * shift, generator=g, device=dev, dtype=dtype)
    go, gs = buf[shift:shift + 3 * n], buf[3 * n + 2 * shift:]
    before = gs.clone().double().reshape(shape)
    q = torch.zeros(shape, dtype=torch.float64, device=dev, requires_grad=True)
    vs = 0.013
    G = torch.zeros((3, *shape), dtype=torch.float64, device=dev)
    G[0, 1:-1] = (q[2:] - q[:-2]) / 2 / vs if X > 2 else 0
    if Y > 2:
        G[1, :, 1:-1] = (q[:, 2:] - q[:, :-2]) / 2 / vs
    if Z > 2:
        G[2, :, :, 1:-1] = (q[:, :, 2:] - q[:, :, :-2]) / 2 / vs
    w = go.double().reshape(3, *shape)
    want, most = before, before.abs()
    if G.requires_grad:
        want = before + torch.autograd.grad((G * w).sum(), q, retain_graph=True)[0]
        most = most + 6 * float(w.abs().max()) / 2 / vs
    call("vx_dense_sdf_gradient_bwd", dtype_code(gs), ptr(go), X, Y, Z, vs, ptr(gs), stream_of(gs))
    eps = 2.0 ** -24 if dtype == torch.float32 else 2.0 ** -53
    # (vs itself is rounded once more in float32)
    assert bool(((gs.double().reshape(shape) - want).abs() <= 10 * eps * most).all())
