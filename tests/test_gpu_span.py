"""Span-window products (kan_span.hip) of layers with many basis functions:
forward, inference and input gradient against float64, at the fp32 parity bar
(normwise 1e-5), over orders, output widths that fill no block, sample and
feature counts that fill no tile or slice, with and without the base branch;
and what they make of inputs and weights that are not finite."""

import ctypes

import pytest
import torch
import torch.nn.functional as F

from torchsplinekan_amd import _C, _lib
from torchsplinekan_amd.reference_backend import compute_basis
from tests._util import make_grid

pytestmark = pytest.mark.gpu

# (n, I, O, G, k, base) and which of the forward, the inference and the input
# gradient the rule gives to the span kernels there: each of 1, 2 and 4 outputs
# a lane (O up to 64, up to 128, more), with rows staged 16 bytes at a time (O a
# multiple of 4) and value by value, at every order
SHAPES = [((8498, 187, 51, 65, 2, True), (1, 1, 0)), ((3000, 333, 61, 66, 2, True), (0, 1, 0)),
          ((3001, 250, 259, 65, 3, False), (0, 1, 0)), ((13220, 73, 19, 65, 1, True), (0, 1, 0)),
          ((1281, 1068, 461, 65, 1, True), (0, 0, 1)), ((4500, 500, 61, 65, 2, False), (1, 1, 1)),
          ((4729, 948, 61, 65, 3, True), (1, 1, 1)), ((5115, 253, 64, 65, 1, True), (1, 1, 1)),
          ((1798, 853, 64, 65, 2, True), (1, 1, 1)), ((2681, 478, 64, 65, 3, False), (1, 1, 1)),
          ((5565, 251, 96, 65, 1, True), (1, 1, 0)), ((2315, 594, 96, 65, 3, True), (1, 1, 0)),
          ((2191, 544, 100, 65, 1, True), (0, 1, 1)), ((4784, 297, 100, 65, 2, False), (1, 1, 0)),
          ((1193, 993, 100, 65, 3, True), (0, 0, 1)), ((1723, 714, 101, 65, 1, False), (0, 1, 1)),
          ((3154, 460, 101, 65, 2, False), (1, 1, 0)), ((2103, 971, 101, 65, 3, False), (0, 1, 1)),
          ((1949, 696, 101, 65, 3, True), (1, 1, 0)), ((2777, 652, 127, 65, 3, True), (1, 1, 1)),
          ((3144, 472, 128, 65, 1, True), (1, 1, 1)), ((2001, 911, 128, 65, 2, False), (1, 1, 1)),
          ((2416, 593, 128, 65, 3, True), (1, 1, 1)), ((3862, 336, 256, 65, 1, True), (1, 1, 1)),
          ((2168, 582, 256, 65, 2, False), (1, 1, 1)), ((6061, 212, 256, 65, 3, True), (1, 1, 1)),
          ((1418, 668, 384, 65, 2, True), (0, 0, 1))]


def _workspace(fn, *args):
    nbytes = ctypes.c_size_t(0)
    _lib.check(fn(*args, ctypes.byref(nbytes)))
    return nbytes.value


def _routes(n, I, O, G, k, base):
    """Which of (forward, inference, input gradient) run on the span kernels:
    those whose workspace differs from the dense route's."""
    out = []
    for fn, args in ((_lib.LIB.kan_hip_forward_workspace, (0, n, I, O, G, k, int(base))),
                     (_lib.LIB.kan_hip_infer_workspace, (0, n, I, O, G, k, int(base))),
                     (_lib.LIB.kan_hip_backward_workspace, (0, n, I, O, G, k, int(base), 1, 0))):
        auto = _workspace(fn, *args)
        with _lib.route("compact_e", 1):
            out.append(int(auto != _workspace(fn, *args)))
    return tuple(out)


def _layer(n, I, O, G, k, base, seed=0):
    g = torch.Generator().manual_seed(seed)
    knots = torch.arange(-k, G + k + 1) * (2.0 / G) - 1.0
    grid = knots + (torch.rand(I, G + 2 * k + 1, generator=g) - 0.5) * (0.8 / G)
    x = (torch.rand(n, I, generator=g) * 2 - 1) * 1.15
    bw = torch.randn(O, I, generator=g) if base else torch.empty(0)
    sw = torch.randn(O, I, G + k, generator=g) * 0.1
    sc = torch.rand(O, I, generator=g) + 0.5
    return [t.cuda() for t in (x, grid, bw, sw, sc)]


def _norm(u, v):
    u, v = u.detach().double(), v.detach()
    return float((u - v).norm() / v.norm())


@pytest.mark.parametrize("shape,routes", SHAPES)
def test_span_products_match_float64(shape, routes):
    n, I, O, G, k, base = shape
    assert _routes(*shape) == routes
    x, grid, bw, sw, sc = _layer(*shape)
    D = torch.randn(n, O, generator=torch.Generator().manual_seed(1)).cuda()
    xg = x.clone().requires_grad_()
    y = _C.kan_apply(xg, grid, bw, sw, sc, k, True)
    dx, = torch.autograd.grad(y, xg, D)
    waug = _C.pack_weight(bw if base else None, sw, sc, k, True)
    yi = _C.kan_infer(x, grid, waug, k, base)

    xd = x.double().requires_grad_()
    W = (sw * sc.unsqueeze(-1)).double().flatten(1)
    want = torch.cat([compute_basis(xd[i:i + 512], grid.double(), k).flatten(1) @ W.t()
                      for i in range(0, n, 512)])
    if base:
        want = want + F.silu(xd) @ bw.double().t()
    wdx, = torch.autograd.grad(want, xd, D.double())
    assert _norm(y, want.detach()) < 1e-5
    assert _norm(yi, want.detach()) < 1e-5
    assert _norm(dx, wdx) < 1e-5
    assert torch.equal(yi, _C.kan_infer(x, grid, waug, k, base))    # fixed order of sums


@pytest.mark.parametrize("shape", [(5115, 253, 64, 65, 1, True), (2001, 911, 128, 65, 2, True),
                                   (4729, 948, 61, 65, 3, True)])
def test_span_products_of_repeated_knots(shape):
    """Knots of up to full multiplicity, inside and at both ends, and an x on
    every knot, against the dense route."""
    n, I, O, G, k, base = shape
    assert _routes(*shape) == (1, 1, 1)
    x, _, bw, sw, sc = _layer(*shape)
    grid = make_grid(I, G, k, "repeated", seed=1)
    grid[:, 10:11 + k] = grid[:, 10:11]
    grid[:, :k + 1], grid[:, -k - 1:] = grid[:, k:k + 1], grid[:, -k - 1:-k]
    grid = grid.float().cuda()
    x = (x + 1) / 2 * (grid.max() - grid.min()) + grid.min()
    x[:grid.shape[1]] = grid.t()
    D = torch.randn(n, O, generator=torch.Generator().manual_seed(1)).cuda()
    waug = _C.pack_weight(bw, sw, sc, k, True)

    def products():
        xg = x.clone().requires_grad_()
        y = _C.kan_apply(xg, grid, bw, sw, sc, k, True)
        return y, _C.kan_infer(x, grid, waug, k, base), torch.autograd.grad(y, xg, D)[0]

    got = products()
    with _lib.route("compact_e", 1):
        want = products()
    for u, v in zip(got, want):
        assert bool(u.isfinite().all()) and _norm(u, v.detach().double()) < 1e-5


def _same_classes(y, want):
    """NaN and infinities in the same places (sign included), the rest close."""
    assert torch.equal(y.isnan(), want.isnan())
    assert torch.equal(y.isinf(), want.isinf())
    assert torch.equal(y[y.isinf()], want[want.isinf()])
    ok = want.isfinite()
    assert _norm(y[ok], want[ok].double()) < 1e-5


def test_span_inputs_and_weights_that_are_not_finite():
    """As in the dense product: NaN or infinite inputs reach their row through
    silu alone; a weight that is not finite reaches its output's every sample,
    times the sample's basis value or silu, or times zero."""
    shape = (3000, 333, 61, 66, 2, True)
    assert _routes(*shape)[1]
    x, grid, bw, sw, sc = _layer(*shape)
    bw = bw.abs() + 0.1
    x[5, 7], x[6, 8], x[7, 9], x[8, 10], x[9, 50] = float("nan"), float("inf"), 50.0, 0.0, -50.0
    sw[3, 100, 20] = float("nan")
    sw[5, 50, 30], sw[6, 50, 0], sw[7, 332, 67] = float("inf"), -float("inf"), float("inf")
    bw[8, 10], bw[9, 11] = float("inf"), -float("inf")
    waug = _C.pack_weight(bw, sw, sc, 2, True)
    y = _C.kan_infer(x, grid, waug, 2, True)
    with _lib.route("compact_e", 1):     # the dense product
        want = _C.kan_infer(x, grid, waug, 2, True)
    assert bool(y[5].isnan().all()) and bool(y[:, 3].isnan().all())
    for o in (5, 8, 9):                  # infinities among them
        assert bool(want[:, o].isinf().any()) and not bool(want[:, o].isfinite().any())
    _same_classes(y, want)


@pytest.mark.parametrize("shape", [(4500, 500, 61, 65, 2, False), (4729, 948, 61, 65, 3, True),
                                   (4500, 500, 256, 65, 3, True),
                                   (1281, 1068, 461, 65, 1, True)])
def test_span_input_gradient_of_values_that_are_not_finite(shape):
    """As from the dense product's window rows: an x outside the knots meets
    no spline weight and, without a base branch, no dL/dy."""
    n, I, O, G, k, base = shape
    assert _routes(*shape)[2]
    x, grid, bw, sw, sc = _layer(*shape)
    D = torch.randn(n, O, generator=torch.Generator().manual_seed(1)).cuda()
    x[0:3] = 40.0                        # outside every feature's knots
    x[3, 5], x[4, 6], x[5, 7] = float("nan"), float("inf"), -float("inf")
    inf = float("inf")
    D[0, 3], D[10, 4], D[11, 5], D[12, 6], D[12, 9] = inf, inf, -inf, inf, -inf
    D[1, 2], D[13, 7] = float("nan"), float("nan")
    sw[3, 20, 0], sw[4, 21, 1], sw[5, 22, 30] = float("nan"), inf, -inf
    sw[O - 1, I - 1, G + k - 1] = inf
    if base:
        bw[2, 30], bw[3, 31] = inf, float("nan")

    def dx():
        xg = x.clone().requires_grad_()
        return torch.autograd.grad(_C.kan_apply(xg, grid, bw, sw, sc, k, True), xg, D)[0]

    got = dx()
    with _lib.route("compact_e", 1):     # the dense product and its windows
        want = dx()
    if not base:
        assert torch.equal(got[0:3], torch.zeros_like(got[0:3]))
    assert bool(want.isinf().any()) and bool(want.isnan().any())
    _same_classes(got, want)


def test_span_products_in_a_captured_graph():
    n, I, O, G, k, base = shape = (4729, 948, 61, 65, 3, True)
    assert _routes(*shape) == (1, 1, 1)
    x, grid, bw, sw, sc = _layer(*shape)
    D = torch.randn(n, O, device="cuda")
    xg = x.clone().requires_grad_()

    def step():
        y = _C.kan_apply(xg, grid, bw, sw, sc, k, True)
        return y, torch.autograd.grad(y, xg, D)[0]

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            step()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y, dx = step()
    for seed in (3, 4):
        with torch.no_grad():
            xg.copy_(_layer(*shape, seed=seed)[0])
        graph.replay()
        ey, edx = step()
        assert torch.equal(y, ey) and torch.equal(dx, edx)
