"""The autograd binding (replacement of the reference's TF custom-op boundary,
Kernels/cp4_conv_nchw.cc:6-108) against PyTorch's own dense convolution on the
recomposed filter: forward values and all five gradients."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def ops():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    import paralleltnnlayers_amd as p
    p.lib()
    from paralleltnnlayers_amd import torch_ops
    return torch_ops


def recomposed(FK, FC, FH, FW):
    return torch.einsum("tr,cr,yr,xr->tcyx", FK, FC, FH, FW)


@pytest.mark.parametrize("dims", [(2, 16, 12, 14, 24, 3, 8), (1, 64, 20, 20, 64, 5, 16),
                                  (3, 5, 9, 9, 7, 1, 3)],
                         ids=lambda d: "x".join(map(str, d)))
def test_gradients_match_dense_autograd(ops, dims):
    N, C, H, W, T, Y, R = dims
    g = torch.Generator(device="cuda").manual_seed(sum(dims))
    mk = lambda *s: torch.randn(*s, device="cuda", generator=g)
    x = mk(N, C, H, W).requires_grad_()
    fac = [(mk(d, R) / R ** 0.25).requires_grad_() for d in (T, C, Y, Y)]
    dy = mk(N, T, H, W)
    y = ops.cp4_conv2d(x, *fac, Y // 2)
    y.backward(dy)
    got = [x.grad.clone()] + [f.grad.clone() for f in fac]

    # float64 dense reference through PyTorch autograd on the recomposed filter
    xd = x.detach().double().requires_grad_()
    fd = [f.detach().double().requires_grad_() for f in fac]
    yd = torch.nn.functional.conv2d(xd, recomposed(*fd), padding=Y // 2)
    yd.backward(dy.double())
    want = [xd.grad] + [f.grad for f in fd]
    assert (y.detach().double() - yd.detach()).abs().max() <= 1e-4 * yd.detach().abs().max()
    for name, a, b in zip(("dx", "dFK", "dFC", "dFH", "dFW"), got, want):
        tol = 1e-4 if name == "dx" else 1e-3
        assert (a.double() - b).abs().max() <= tol * b.abs().max(), name


def test_only_requested_gradients(ops):
    x = torch.randn(1, 8, 6, 6, device="cuda")
    fac = [torch.randn(d, 4, device="cuda") for d in (8, 8, 3, 3)]
    fac[0].requires_grad_()
    ops.cp4_conv2d(x, *fac, 1).sum().backward()
    assert fac[0].grad is not None and all(f.grad is None for f in fac[1:]) and x.grad is None


def test_padding_other_than_same_gives_the_smaller_output(ops):
    """pad = 0 with a 3x3 filter: the layer's output is (H - 2) x (W - 2), as a dense
    convolution's, and differentiable (the geometry entry points)."""
    x = torch.randn(1, 8, 6, 6, device="cuda", requires_grad=True)
    fac = [torch.randn(d, 4, device="cuda", requires_grad=True) for d in (8, 8, 3, 3)]
    y = ops.cp4_conv2d(x, *fac, 0)
    want = torch.nn.functional.conv2d(x.detach(), recomposed(*[f.detach() for f in fac]))
    assert y.shape == want.shape == (1, 8, 4, 4)
    assert (y.detach() - want).abs().max() <= 1e-4 * want.abs().max()
    y.sum().backward()
    assert x.grad is not None and all(f.grad is not None for f in fac)


def test_layer_trains(ops):
    """A few SGD steps on a CP4Conv2d layer lower a regression loss: forward,
    both backward passes and the optimizer see consistent tensors."""
    torch.manual_seed(0)
    layer = ops.CP4Conv2d(16, 16, 3, rank=8)
    target = ops.CP4Conv2d(16, 16, 3, rank=8)
    x = torch.randn(4, 16, 10, 10, device="cuda")
    with torch.no_grad():
        want = target(x)
    opt = torch.optim.SGD(layer.parameters(), lr=0.05)
    losses = []
    for _ in range(30):
        opt.zero_grad()
        loss = ((layer(x) - want) ** 2).mean()
        loss.backward()
        opt.step()
        losses.append(loss.item())
    assert losses[-1] < 0.7 * losses[0]
    K = layer.dense_filter()
    assert K.shape == (16, 16, 3, 3)
    dense = torch.nn.functional.conv2d(x, K, padding=1)
    assert (layer(x).detach() - dense).abs().max() <= 1e-4 * dense.abs().max()


def test_strided_layer_matches_dense_strided_conv(ops):
    """stride 2 = every second row and column of the stride-1 result, which for
    "same" padding is PyTorch's strided convolution with the recomposed filter;
    the gradients flow through the subsampling."""
    g = torch.Generator(device="cuda").manual_seed(11)
    mk = lambda *s: torch.randn(*s, device="cuda", generator=g)
    N, C, H, W, T, Y, R = 2, 16, 13, 16, 24, 3, 8
    x = mk(N, C, H, W).requires_grad_()
    fac = [(mk(d, R) / R ** 0.25).requires_grad_() for d in (T, C, Y, Y)]
    y = ops.cp4_conv2d(x, *fac, 1, stride=2)
    dy = mk(*y.shape)
    y.backward(dy)
    xd = x.detach().double().requires_grad_()
    fd = [f.detach().double().requires_grad_() for f in fac]
    yd = torch.nn.functional.conv2d(xd, recomposed(*fd), padding=1, stride=2)
    assert yd.shape == y.shape
    yd.backward(dy.double())
    assert (y.detach().double() - yd.detach()).abs().max() <= 1e-4 * yd.detach().abs().max()
    for name, a, b in zip(("dx", "dFK", "dFC", "dFH", "dFW"), [x.grad] + [f.grad for f in fac],
                          [xd.grad] + [f.grad for f in fd]):
        tol = 1e-4 if name == "dx" else 1e-3
        assert (a.double() - b).abs().max() <= tol * b.abs().max(), name


def test_bfloat16_activations_through_autograd(ops):
    """bfloat16 x: forward, input gradient and factor gradients run the library's
    bfloat16-activation entry points; compared with float64 autograd on the same
    (bfloat16-representable) inputs within the bfloat16 rounding of y, dx and dy."""
    g = torch.Generator(device="cuda").manual_seed(21)
    mk = lambda *s: torch.randn(*s, device="cuda", generator=g)
    N, C, H, W, T, Y, R = 2, 32, 12, 16, 48, 3, 8
    x = mk(N, C, H, W).to(torch.bfloat16).requires_grad_()
    fac = [(mk(d, R) / R ** 0.25).requires_grad_() for d in (T, C, Y, Y)]
    y = ops.cp4_conv2d(x, *fac, 1)
    assert y.dtype == torch.bfloat16
    dy = mk(N, T, H, W).to(torch.bfloat16)
    y.backward(dy)
    assert x.grad.dtype == torch.bfloat16 and fac[0].grad.dtype == torch.float32
    xd = x.detach().double().requires_grad_()
    fd = [f.detach().double().requires_grad_() for f in fac]
    yd = torch.nn.functional.conv2d(xd, recomposed(*fd), padding=1)
    yd.backward(dy.double())
    assert (y.detach().double() - yd.detach()).abs().max() <= 2.0 ** -7 * yd.detach().abs().max()
    assert (x.grad.double() - xd.grad).abs().max() <= 2.0 ** -7 * xd.grad.abs().max()
    for name, a, b in zip(("dFK", "dFC", "dFH", "dFW"), [f.grad for f in fac], [f.grad for f in fd]):
        assert (a.double() - b).abs().max() <= 1e-3 * b.abs().max(), name


def _small_layer(ops, **kw):
    layer = ops.CP4Conv2d(8, 12, 3, 4, bias=True, activation="relu", **kw)
    torch.manual_seed(5)
    with torch.no_grad():
        layer.bias.normal_()
    return layer, torch.randn(2, 8, 9, 10, device="cuda")


@pytest.mark.parametrize("kw", [{}, {"stride": 2, "padding": "same"}], ids=["plain", "stride"])
def test_traced_layer_computes_from_its_inputs(ops, kw):
    """A trace holds the layer as an operator: run on another input it gives that input's result."""
    layer, x = _small_layer(ops, **kw)
    traced = torch.jit.trace(layer, x, check_trace=False)
    other = torch.randn_like(x)
    assert torch.equal(traced(other), layer(other))


@pytest.mark.parametrize("kw", [{}, {"stride": 2, "padding": "same"}], ids=["plain", "stride"])
def test_python_autograd_function_matches_the_native_one(ops, kw):
    layer, x = _small_layer(ops, **kw)
    dy = torch.randn_like(layer(x))

    def grads(run):
        xi = x.clone().requires_grad_()
        layer.zero_grad(set_to_none=True)
        y = run(xi)
        y.backward(dy)
        return [y.detach(), xi.grad] + [p.grad for p in layer.parameters()]

    args = lambda xi: (xi, layer.FK, layer.FC, layer.FH, layer.FW, layer.pad, layer.bias,
                       layer.activation, layer.stride, layer.padding)
    for a, b in zip(grads(lambda xi: ops._traced_layer(*args(xi))), grads(layer)):
        assert torch.equal(a, b)


def test_forward_mode_tangents_are_refused(ops):
    import torch.autograd.forward_ad as fwd
    layer, x = _small_layer(ops)
    with torch.no_grad(), fwd.dual_level():
        with pytest.raises((RuntimeError, NotImplementedError)):
            layer(fwd.make_dual(x, torch.ones_like(x)))


def test_bias_gradient_under_create_graph(ops):
    """The bias gradient is linear in dy: its own gradient with respect to dy is the mask."""
    layer, x = _small_layer(ops)
    y = layer(x)
    dy = torch.randn_like(y).requires_grad_()
    (db,) = torch.autograd.grad(y, layer.bias, dy, create_graph=True)
    assert torch.allclose(db, (dy * (y > 0)).sum(dim=(0, 2, 3)), rtol=1e-4, atol=1e-4)
    (gg,) = torch.autograd.grad(db.sum(), dy)
    assert torch.equal(gg, (y > 0).float())


def test_vector_factors_at_rank_one(ops):
    """A tap factor of rank 1 as a vector computes what the one-column matrix does."""
    import paralleltnnlayers_amd as cp4
    x, dy = torch.randn(2, 8, 9, 10, device="cuda"), torch.randn(2, 12, 9, 10, device="cuda")
    cols = [torch.randn(d, 1, device="cuda") for d in (12, 8, 3, 3)]
    vecs = cols[:2] + [f.flatten() for f in cols[2:]]
    assert torch.equal(cp4.conv2d_forward(x, *vecs), cp4.conv2d_forward(x, *cols))
    assert torch.equal(cp4.conv2d_backward_data(dy, *vecs), cp4.conv2d_backward_data(dy, *cols))
    for a, v, c in zip(vecs, cp4.conv2d_backward_filter(x, dy, *vecs),
                       cp4.conv2d_backward_filter(x, dy, *cols)):
        assert v.shape == a.shape and torch.equal(v.flatten(), c.flatten())
    leaves = [[f.clone().requires_grad_() for f in fac] for fac in (vecs, cols)]
    ys = [ops.cp4_conv2d(x, *fac, 1) for fac in leaves]
    assert torch.equal(*ys)
    for y in ys:
        y.backward(dy)
    assert all(torch.equal(a.grad.flatten(), b.grad.flatten()) for a, b in zip(*leaves))


@pytest.mark.parametrize("kw", [{"dtype": torch.float16}, {"stride": 2}], ids=["f16", "stride"])
def test_bias_forms(ops, kw):
    """Half-precision layers and layers with a geometry take a bias of any form."""
    x = torch.randn(2, 16, 9, 10, device="cuda", dtype=kw.get("dtype", torch.float32))
    fac = [torch.randn(d, 4, device="cuda") for d in (16, 16, 3, 3)]
    bias = torch.randn(16, device="cuda")
    run = lambda b: ops.cp4_conv2d(x, *fac, 1, bias=b, stride=kw.get("stride", 1))
    assert torch.equal(run(bias.view(1, 16, 1, 1)), run(bias))
    with pytest.raises(AssertionError):
        run(bias[:15].contiguous())


def test_out_smaller_than_the_result_is_refused(ops):
    import paralleltnnlayers_amd as cp4
    x = torch.randn(2, 8, 9, 10, device="cuda")
    fac = [torch.randn(d, 4, device="cuda") for d in (8, 8, 3, 3)]
    for run in (cp4.conv2d_forward, cp4.conv2d_backward_data):
        with pytest.raises(AssertionError, match="smaller"):
            run(x, *fac, out=torch.empty(2, 8, 9, 9, device="cuda"))
        out = torch.empty(2 * 8 * 9 * 10, device="cuda")
        assert torch.equal(run(x, *fac, out=out).view(2, 8, 9, 10), run(x, *fac))


@pytest.mark.parametrize("kw", [{}, {"stride": 2, "padding": "same"}], ids=["plain", "stride"])
def test_saved_tensor_hooks_see_what_the_layer_saves(ops, kw):
    """Offloading the saved tensors changes nothing; x, the factors and y are what is saved."""
    layer, x = _small_layer(ops, **kw)
    dy = torch.randn_like(layer(x))

    def grads(run):
        xi = x.clone().requires_grad_()
        layer.zero_grad(set_to_none=True)
        run(xi).backward(dy)
        return [xi.grad] + [p.grad for p in layer.parameters()]

    def offloaded(xi):
        with torch.autograd.graph.save_on_cpu():
            return layer(xi)

    want = grads(layer)
    assert all(torch.equal(a, b) for a, b in zip(grads(offloaded), want))
    shapes = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: (shapes.append(tuple(t.shape)), t)[1],
                                                  lambda t: t):
        y = layer(x.clone().requires_grad_())
    assert sorted(shapes) == sorted([tuple(x.shape), tuple(y.shape)] +
                                    [tuple(f.shape) for f in (layer.FK, layer.FC, layer.FH, layer.FW)])


def test_functional_transforms_are_refused(ops):
    """The library sees memory, not batched or wrapped tensors: an error, never a result."""
    import paralleltnnlayers_amd as cp4
    layer, x = _small_layer(ops)
    fac = [f.detach() for f in (layer.FK, layer.FC, layer.FH, layer.FW)]
    dy = torch.randn_like(layer(x)).detach()
    xs = torch.stack([x, x])
    batched = lambda t: torch.stack([t, t])
    with torch.no_grad():
        calls = [lambda: torch.vmap(layer)(xs),
                 lambda: torch.vmap(lambda f: ops.cp4_conv2d(x, f, *fac[1:], 1))(batched(fac[0])),
                 lambda: torch.vmap(lambda b: ops.cp4_conv2d(x, *fac, 1, bias=b))(batched(layer.bias)),
                 lambda: torch.vmap(lambda t: cp4.conv2d_forward(t, *fac))(xs),
                 lambda: torch.vmap(lambda t: cp4.conv2d_backward_data(t, *fac))(batched(dy)),
                 lambda: torch.vmap(lambda t: cp4.conv2d_backward_filter(x, t, *fac)[0])(batched(dy))]
    calls += [lambda: torch.func.grad(lambda t: layer(t).sum())(x),
              lambda: torch.func.jvp(layer, (x,), (x,))]
    xi = x.clone().requires_grad_()
    y = layer(xi)
    calls += [lambda: torch.autograd.grad(y, xi, torch.stack([dy, dy]), is_grads_batched=True)]
    for call in calls:
        with pytest.raises((RuntimeError, NotImplementedError)):
            call()


def test_layer_on_a_side_stream(ops):
    """Forward and backward run on the stream that is current at the forward call."""
    layer, x = _small_layer(ops)
    x = x.repeat(4, 1, 8, 8).requires_grad_()
    dy = torch.randn_like(layer(x))
    layer(x).backward(dy)
    want = [x.grad] + [p.grad for p in layer.parameters()]
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    for _ in range(3):
        x.grad = None
        layer.zero_grad(set_to_none=True)
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            y = layer(x * 1)                      # (work of its own in front of it)
            y.backward(dy)
        torch.cuda.current_stream().wait_stream(side)
        got = [x.grad] + [p.grad for p in layer.parameters()]
        assert all(torch.equal(a, b) for a, b in zip(got, want))
