"""The layer entry points (cp4_layer_forward / cp4_layer_backward): what the activation's
backward and the bias gradient do at the edges of their kernel - planes that are no multiple
of a 16-byte piece, channels of one and of many segments, every element type - against
float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def capi():
    import paralleltnnlayers_amd.capi as c
    c.lib()
    assert torch.cuda.is_available()
    return c


# (N, T, H, W): one pixel / odd plane / a piece and one / several batches per lane / segments
# that end inside a plane / more channels than workgroups per segment
@pytest.mark.parametrize("dims", [(1, 1, 1, 1), (3, 5, 7, 7), (2, 3, 3, 3), (4, 2, 55, 55),
                                  (3, 2, 129, 130), (2, 600, 9, 16)],
                         ids=lambda d: "x".join(map(str, d)))
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16],
                         ids=["f32", "bf16", "f16"])
@pytest.mark.parametrize("relu", [True, False], ids=["relu", "linear"])
def test_bias_and_activation_gradient(capi, dims, dtype, relu):
    N, T, H, W = dims
    C, R = 4, 2
    gen = torch.Generator(device="cuda").manual_seed(sum(dims))
    mk = lambda *s: torch.randn(*s, device="cuda", generator=gen)
    x, dy = mk(N, C, H, W).to(dtype), mk(N, T, H, W).to(dtype)
    fac = [mk(d, R) for d in (T, C, 1, 1)]
    bias = mk(T)
    s = capi.shape_for(x.shape, *fac, 0)
    act = "relu" if relu else None
    y = capi.layer_forward(s, None, x, *fac, bias, act)
    dx, grads, dbias = capi.layer_backward(s, None, x, y, dy, *fac, act)
    masked = torch.where(y > 0, dy, torch.zeros_like(dy)) if relu else dy
    want = masked.double().sum(dim=(0, 2, 3))
    # fp32 sums of N * H * W terms: 2^-24 each step, as a random walk over the terms
    tol = 2.0 ** -22 * (masked.double() ** 2).sum(dim=(0, 2, 3)).sqrt() * (1 + (N * H * W) ** 0.5 / 64)
    assert ((dbias.double() - want).abs() <= tol + 1e-30).all()
    # the gradients are those of the masked dy: 1x1 filter, so the layer is a matrix product
    K = torch.einsum("tr,cr,r->tc", fac[0].double(), fac[1].double(),
                     (fac[2][0] * fac[3][0]).double())
    want_dx = torch.einsum("tc,nthw->nchw", K, masked.double())
    eps = {torch.float32: 1e-5, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    bound = eps * want_dx.abs() * 1.01 + 1e-5 * want_dx.abs().max()
    assert ((dx.double() - want_dx).abs() <= bound).all()
    dK = torch.einsum("nthw,nchw->tc", masked.double(), x.double())
    want_dFK = dK @ (fac[1] * fac[2][0] * fac[3][0]).double()
    assert (grads[0].double() - want_dFK).abs().max() <= 1e-4 * want_dFK.abs().max() + 1e-6


def test_parts_on_their_own(capi):
    """Each gradient alone is the one of the whole call; what is not wanted is not computed."""
    gen = torch.Generator(device="cuda").manual_seed(3)
    mk = lambda *s: torch.randn(*s, device="cuda", generator=gen)
    x, dy = mk(2, 16, 9, 11), mk(2, 24, 9, 11)
    fac = [mk(d, 8) for d in (24, 16, 3, 3)]
    s = capi.shape_for(x.shape, *fac, 1)
    y = capi.layer_forward(s, None, x, *fac, mk(24), "relu")
    dx, grads, db = capi.layer_backward(s, None, x, y, dy, *fac, "relu")
    only_dx = capi.layer_backward(s, None, x, y, dy, *fac, "relu", True, False, False)
    only_f = capi.layer_backward(s, None, x, y, dy, *fac, "relu", False, True, False)
    only_b = capi.layer_backward(s, None, x, y, dy, *fac, "relu", False, False, True)
    # dx alone contracts dy itself, dx beside the factor gradients takes their G1: the same fp32
    # sums (24 channels, 9 taps, 8 ranks) in another order, each rounded to 2^-24 of its terms
    terms = torch.nn.functional.conv_transpose2d(
        torch.where(y > 0, dy, torch.zeros_like(dy)).abs(),
        torch.einsum("tr,cr,yr,xr->tcyx", *[f.abs() for f in fac]), padding=1)
    assert ((only_dx[0] - dx).abs() <= 2 * (24 + 9 + 8) * 2.0 ** -24 * terms + 1e-30).all()
    assert only_dx[2] is None and only_dx[1][0] is None
    # the factor gradients alone may take the mask with them on tiles of their own: the same fp32
    # sums (2 * 9 * 11 pixels, then 24 * 9, 16 * 9 or 24 * 16 * 3 entries of dK) in another order
    dK = torch.nn.grad.conv2d_weight(x.abs(), (24, 16, 3, 3), dy.abs(), padding=1)
    f = [t.abs() for t in fac]
    sums = [torch.einsum("tcyx,cr,yr,xr->tr", dK, f[1], f[2], f[3]),
            torch.einsum("tcyx,tr,yr,xr->cr", dK, f[0], f[2], f[3]),
            torch.einsum("tcyx,tr,cr,xr->yr", dK, f[0], f[1], f[3]),
            torch.einsum("tcyx,tr,cr,yr->xr", dK, f[0], f[1], f[2])]
    for a, b, t, n in zip(only_f[1], grads, sums, (16 * 9, 24 * 9, 24 * 16 * 3, 24 * 16 * 3)):
        assert ((a - b).abs() <= 2 * (198 + n) ** 0.5 * 2.0 ** -24 * t).all()
    assert only_f[0] is None
    assert torch.equal(only_b[2], db)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16],
                         ids=["f32", "bf16", "f16"])
def test_non_finite_gradient_behind_a_clipped_output_is_seen(capi, dtype):
    """The mask is a product, as dy * (y > 0): an infinite dy at a clipped output gives NaN."""
    gen = torch.Generator(device="cuda").manual_seed(8)
    mk = lambda *s: torch.randn(*s, device="cuda", generator=gen)
    x, fac = mk(2, 8, 9, 11).to(dtype), [mk(d, 4) for d in (12, 8, 1, 1)]
    s = capi.shape_for(x.shape, *fac, 0)
    y = capi.layer_forward(s, None, x, *fac, mk(12), "relu")
    n, t, h, w = (int(v) for v in (y == 0).nonzero()[0])
    dy = torch.zeros_like(y)
    dy[n, t, h, w] = float("inf")
    dbias = capi.layer_backward(s, None, x, y, dy, *fac, "relu", False, False, True)[2]
    assert torch.isnan(dbias[t]) and int(torch.isfinite(dbias).sum()) == 11


# The input gradient beside the factor gradients (dx = FC G1): pixels that no piece divides, blocks
# over image boundaries, one channel block and several, every chunk count of ranks, a stride.
BESIDE = [(1, 16, 4, 4, 16, 3, 1, 1), (2, 16, 5, 7, 32, 3, 16, 1), (9, 48, 7, 7, 16, 3, 17, 1),
          (3, 80, 14, 14, 32, 1, 32, 1), (3, 80, 14, 15, 32, 1, 32, 1), (2, 32, 15, 30, 48, 5, 33, 1),
          (3, 272, 20, 20, 16, 3, 64, 1), (3, 272, 21, 21, 16, 3, 64, 1), (2, 64, 18, 19, 16, 3, 64, 1),
          (2, 48, 55, 55, 32, 3, 32, 2), (2, 16, 56, 60, 16, 3, 48, 2)]


@pytest.mark.parametrize("case,dtype", [
    pytest.param(c, t, id="x".join(map(str, c)) + "-" + n) for c in BESIDE
    for t, n in ((torch.float32, "f32"), (torch.bfloat16, "bf16"), (torch.float16, "f16"))
    if c[-1] == 1 or t == torch.float32])             # (layers with a stride take fp32)
def test_input_gradient_beside_the_factors(capi, case, dtype):
    N, C, H, W, T, k, R, stride = case
    gen = torch.Generator(device="cuda").manual_seed(N + C + H + W + R)
    mk = lambda *s: torch.randn(*s, device="cuda", generator=gen)
    x = mk(N, C, H, W).to(dtype)
    fac = [mk(d, R) for d in (T, C, k, k)]
    s = capi.shape_for(x.shape, *fac, k // 2)
    g = capi.geometry(s, stride, "same") if stride > 1 else None
    y = capi.layer_forward(s, g, x, *fac, mk(T), "relu")
    dy = mk(*y.shape).to(dtype)
    dx, _, _ = capi.layer_backward(s, g, x, y, dy, *fac, "relu")
    # (the fp32 factor gradients of some layers run a variant that leaves no G1)
    other = (g is None and dtype == torch.float32 and
             capi.plan_query(s, "backward_filter")["variant"] != "mfma_four_launches")
    assert capi.layer_last_backward_route() == (0 if other else capi.ROUTE_DX_FROM_G1)
    masked = torch.where(y > 0, dy, torch.zeros_like(dy)).double().cpu()
    K = torch.einsum("tr,cr,yr,xr->tcyx", *[f.double().cpu() for f in fac])
    if g is None:
        g = capi.geometry(s, 1, "same")
    pads = (g.pad_left, (g.out_w - 1) * stride + k - W - g.pad_left,
            g.pad_top, (g.out_h - 1) * stride + k - H - g.pad_top)

    def adjoint(d, f):
        z = torch.zeros(N, C, H, W, dtype=torch.float64, requires_grad=True)
        out = torch.nn.functional.conv2d(torch.nn.functional.pad(z, pads), f, stride=stride)
        return torch.autograd.grad(out, z, d)[0]

    want = adjoint(masked, K)
    # three fp32 contractions: 2^-24 a step of the sum of the terms' magnitudes (as a random walk,
    # with a factor of four to spare), and the rounding of the stored result
    terms = adjoint(masked.abs(), torch.einsum("tr,cr,yr,xr->tcyx", *[f.double().cpu().abs() for f in fac]))
    eps = {torch.float32: 0.0, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    bound = 4 * (T + 2 * k + R) ** 0.5 * 2.0 ** -24 * terms + eps * want.abs() + 1e-30
    if dtype == torch.float16:
        bound = bound + 2.0 ** -24          # subnormal results
    assert ((dx.double().cpu() - want).abs() <= bound).all()


# Mask and bias gradient inside the factor gradients' contraction and gradient GEMM: both variants,
# every split of the channels over waves (1, 2, 4), one rank tile and two, planes that no block of 32
# pixels or four divides, strides with planes of either kind, channel groups the last block does
# not fill, every element type.
INSIDE = [(1, 64, 8, 8, 64, 3, 8, 1), (3, 144, 9, 12, 80, 3, 33, 1), (16, 64, 32, 32, 64, 3, 16, 1),
          (2, 32, 16, 20, 272, 5, 64, 1), (2, 32, 7, 9, 48, 3, 16, 1), (5, 256, 15, 15, 144, 1, 64, 1),
          (24, 64, 40, 40, 64, 3, 64, 1), (2, 48, 55, 55, 32, 3, 32, 2), (3, 64, 56, 60, 176, 3, 48, 2),
          (2, 16, 9, 9, 16, 1, 4, 2), (1, 16, 120, 121, 16, 3, 4, 2)]


@pytest.mark.parametrize("relu", [True, False], ids=["relu", "linear"])
@pytest.mark.parametrize("case,dtype", [
    pytest.param(c, t, id="x".join(map(str, c)) + "-" + n) for c in INSIDE
    for t, n in ((torch.float32, "f32"), (torch.bfloat16, "bf16"), (torch.float16, "f16"))
    if c[-1] == 1 or t == torch.float32])
def test_mask_and_bias_gradient_inside_the_passes(capi, case, dtype, relu):
    N, C, H, W, T, k, R, stride = case
    gen = torch.Generator(device="cuda").manual_seed(N + C + H + W + R)
    mk = lambda *s: torch.randn(*s, device="cuda", generator=gen)
    x = mk(N, C, H, W).to(dtype)
    fac = [mk(d, R) for d in (T, C, k, k)]
    s = capi.shape_for(x.shape, *fac, k // 2)
    g = capi.geometry(s, stride, "same") if stride > 1 else None
    act = "relu" if relu else None
    y = capi.layer_forward(s, g, x, *fac, mk(T), act)
    dy = mk(*y.shape).to(dtype)
    dx, grads, dbias = capi.layer_backward(s, g, x, y, dy, *fac, act)
    assert capi.layer_last_backward_mask_inside()
    masked = dy * (y > 0) if relu else dy
    md = masked.double()
    # fp32 sums: 2^-24 a step, as a random walk over the terms (a factor of four to spare)
    n = N * md.shape[2] * md.shape[3]
    tol = 4 * 2.0 ** -24 * ((md ** 2).sum(dim=(0, 2, 3)) * n).sqrt()
    assert ((dbias.double() - md.sum(dim=(0, 2, 3))).abs() <= tol).all()
    # the other gradients are bit for bit the same call's on the masked dy, which it does not mask
    dx2, grads2, _ = capi.layer_backward(s, g, x, None, masked, *fac, None, True, True, False)
    assert not capi.layer_last_backward_mask_inside()
    assert torch.equal(dx, dx2) and all(torch.equal(a, b) for a, b in zip(grads, grads2))
    # ... and right: n roundings of 2^-24 grow as sqrt(n), as sums of n terms with signs at random do; times
    # 4 for the stages one after the other.  dx is rounded to the layer's type.
    bound = 4 * 2.0 ** -24 * (T + C + R + 2 * k + n) ** 0.5
    eps = {torch.float32: 0.0, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    for name, got, w in zip(("x", "FK", "FC", "FH", "FW"), (dx, *grads),
                            layer_reference(x, masked, fac, k, stride, g)):
        err = ((got.double() - w).norm() / w.norm()).item()
        assert err <= bound + (eps if name == "x" else 0), (name, err, bound)


def layer_reference(x, dy, fac, k, stride, geometry):
    """(dx, dFK, dFC, dFH, dFW) of dy by autograd over the four contractions in float64."""
    N, C, H, W = x.shape
    x = x.double().requires_grad_()
    FK, FC, FH, FW = f = [t.double().requires_grad_() for t in fac]
    A = torch.matmul(FC.t(), x.flatten(2)).view(N, -1, H, W)
    sh, top, left = (stride, geometry.pad_top, geometry.pad_left) if geometry else (1, k // 2, k // 2)
    oh, ow = dy.shape[2:]
    A = torch.nn.functional.pad(A, (left, k + sh, top, k + sh))
    rows = lambda t, i, n: t.narrow(2, i, sh * (n - 1) + 1)[:, :, ::sh]
    B = sum(FH[i].view(1, -1, 1, 1) * rows(A, i, oh) for i in range(k))
    Z = sum(FW[j].view(1, -1, 1, 1) * rows(B.transpose(2, 3), j, ow).transpose(2, 3) for j in range(k))
    y = torch.matmul(FK, Z.flatten(2)).view(N, -1, oh, ow)
    return torch.autograd.grad(y, [x] + f, dy.double())


# (N, C, H, W, T, k, R, stride), inside: channels a wave, waves and bytes at either side of where the mask rides
# along, in the three-launch and the four-launch variant; two rank tiles, strides
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("case,inside", [
    ((12, 64, 28, 28, 512, 3, 16, 1), True), ((12, 80, 28, 28, 528, 1, 16, 1), False),
    ((2, 80, 28, 28, 528, 3, 40, 1), True), ((12, 32, 27, 27, 640, 3, 8, 1), True),
    ((12, 32, 27, 27, 656, 3, 8, 1), False),
    ((7, 512, 29, 29, 512, 1, 64, 1), True), ((4, 64, 64, 64, 96, 3, 64, 1), True),
    ((6, 32, 56, 56, 320, 3, 40, 2), True)], ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else v)
def test_mask_inside_wide_layers(capi, case, inside, dtype):
    N, C, H, W, T, k, R, stride = case
    if stride > 1 and dtype != torch.float32:
        pytest.skip("a layer with a stride takes fp32 activations")
    gen = torch.Generator(device="cuda").manual_seed(N + C + H + W + R)
    mk = lambda *s: torch.randn(*s, device="cuda", generator=gen)
    x, fac = mk(N, C, H, W).to(dtype), [mk(d, R) for d in (T, C, k, k)]
    s = capi.shape_for(x.shape, *fac, k // 2)
    g = capi.geometry(s, stride, "same") if stride > 1 else None
    y = capi.layer_forward(s, g, x, *fac, mk(T), "relu")
    dy = mk(*y.shape).to(dtype)
    dx, grads, dbias = capi.layer_backward(s, g, x, y, dy, *fac, "relu")
    assert capi.layer_last_backward_mask_inside() == inside
    masked = dy * (y > 0)
    want = layer_reference(x, masked, fac, k, stride, g)
    # sums of T and C channels, R ranks, the taps and the pixels, signs at random: n roundings of 2^-24
    # grow as sqrt(n), as the sum itself; times 4 for the stages one after the other.  dx is rounded to
    # the layer's type.
    pixels = N * masked.shape[2] * masked.shape[3]
    bound = 4 * 2.0 ** -24 * (T + C + R + 2 * k + pixels) ** 0.5
    for name, got, w in zip(("x", "FK", "FC", "FH", "FW"), (dx, *grads), want):
        err = ((got.double() - w).norm() / w.norm()).item()
        assert err <= bound + (2.0 ** -8 if name == "x" and dtype == torch.bfloat16 else 0), (name, err, bound)
    tol = 4 * 2.0 ** -24 * ((masked.double() ** 2).sum(dim=(0, 2, 3)) * pixels).sqrt()
    assert ((dbias.double() - masked.double().sum(dim=(0, 2, 3))).abs() <= tol).all()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16],
                         ids=["f32", "bf16", "f16"])
def test_non_finite_gradient_is_seen_inside_the_passes(capi, dtype):
    gen = torch.Generator(device="cuda").manual_seed(8)
    mk = lambda *s: torch.randn(*s, device="cuda", generator=gen)
    x, fac = mk(2, 64, 12, 12).to(dtype), [mk(d, 4) for d in (80, 64, 1, 1)]
    s = capi.shape_for(x.shape, *fac, 0)
    y = capi.layer_forward(s, None, x, *fac, mk(80), "relu")
    n, t, h, w = (int(v) for v in (y == 0).nonzero()[-1])
    dy = torch.zeros_like(y)
    dy[n, t, h, w] = float("inf")
    dx, grads, dbias = capi.layer_backward(s, None, x, y, dy, *fac, "relu")
    assert capi.layer_last_backward_mask_inside()
    assert torch.isnan(dbias[t]) and int(torch.isfinite(dbias).sum()) == 79
    assert torch.isnan(grads[0][t]).all() and torch.isnan(dx[n, :, h, w]).all()
    assert int(torch.isnan(dx).sum()) == 64          # (no other pixel)


# A first layer (no input gradient): mask and bias gradient inside the dense-gradient kernel.
# Both counts of row blocks and groups, planes smaller than a tile, widths no piece divides,
# several tiles a workgroup, operands off a 16-byte boundary.
@pytest.mark.parametrize("case", [(1, 3, 1, 1, 1, 1, 1, 0), (2, 3, 7, 9, 16, 3, 4, 0),
                                  (3, 1, 33, 20, 17, 5, 8, 0), (2, 3, 30, 31, 33, 3, 16, 0),
                                  (2, 4, 16, 64, 64, 1, 16, 1), (16, 3, 90, 112, 64, 3, 16, 0),
                                  (4, 3, 112, 112, 40, 3, 16, 1)],
                         ids=lambda c: "x".join(map(str, c)))
@pytest.mark.parametrize("relu", [True, False], ids=["relu", "linear"])
def test_first_layer_without_an_input_gradient(capi, case, relu):
    N, C, H, W, T, k, R, shift = case
    gen = torch.Generator(device="cuda").manual_seed(N * H + W + T)
    mk = lambda *s: torch.randn(*s, device="cuda", generator=gen)

    def placed(t):                      # the same values `shift` floats off the allocation
        flat = torch.empty(t.numel() + shift, device="cuda")[shift:]
        return flat.copy_(t.flatten()).view(t.shape)

    x, dy = placed(mk(N, C, H, W)), placed(mk(N, T, H, W))
    fac = [mk(d, R) for d in (T, C, k, k)]
    s = capi.shape_for(x.shape, *fac, k // 2)
    act = "relu" if relu else None
    y = placed(capi.layer_forward(s, None, x, *fac, mk(T), act))
    _, grads, dbias = capi.layer_backward(s, None, x, y, dy, *fac, act, False, True, True)
    assert capi.layer_last_backward_route() == capi.ROUTE_MASKED_TILES
    alone = capi.layer_backward(s, None, x, y, dy, *fac, act, False, True, False)[1]
    assert all(torch.equal(a, b) for a, b in zip(grads, alone))
    masked = (torch.where(y > 0, dy, torch.zeros_like(dy)) if relu else dy).double().cpu()
    # fp32 sums: 2^-24 a step, as a random walk over the terms (a factor of four to spare)
    n = N * H * W
    want = masked.sum(dim=(0, 2, 3))
    tol = 4 * 2.0 ** -24 * ((masked ** 2).sum(dim=(0, 2, 3)) * n).sqrt()
    assert ((dbias.double().cpu() - want).abs() <= tol + 1e-30).all()
    xd = x.double().cpu()
    K = torch.zeros(T, C, k, k, dtype=torch.float64, requires_grad=True)
    dK, = torch.autograd.grad(torch.nn.functional.conv2d(xd, K, padding=k // 2), K, masked)
    f = [t.double().cpu() for t in fac]
    wants = [torch.einsum("tcyx,cr,yr,xr->tr", dK, f[1], f[2], f[3]),
             torch.einsum("tcyx,tr,yr,xr->cr", dK, f[0], f[2], f[3]),
             torch.einsum("tcyx,tr,cr,xr->yr", dK, f[0], f[1], f[3]),
             torch.einsum("tcyx,tr,cr,yr->xr", dK, f[0], f[1], f[2])]
    # the repository's bar for factor gradients
    for g, w in zip(grads, wants):
        assert (g.double().cpu() - w).abs().max() <= 1e-3 * w.abs().max() + 1e-30


# The one pass over dy of large layers: 2, 3, 4, 5, 7 and 8 waves, planes that no chunk of 64 pixels
# divides, ranks that fill a tile and not, every filter size of the column taps; and layers on the
# other side of the line, where the passes on their own are the quicker.
@pytest.mark.parametrize("case,one_pass", [
    ((33, 32, 46, 54, 96, 5, 32), False), ((24, 16, 64, 64, 128, 3, 16), True),
    ((70, 48, 32, 36, 256, 1, 7), True), ((22, 16, 60, 68, 224, 3, 31), True),
    ((40, 16, 66, 66, 64, 7, 5), True), ((70, 32, 46, 54, 96, 5, 32), True),
    ((48, 32, 40, 44, 160, 3, 32), True), ((96, 64, 56, 60, 64, 3, 16), True),
    ((21, 64, 56, 56, 96, 3, 16), False), ((11, 16, 56, 56, 160, 3, 32), False)],
    ids=lambda c: "x".join(map(str, c)) if isinstance(c, tuple) else ("apart", "one")[c])
def test_large_layer_behind_relu(capi, case, one_pass):
    N, C, H, W, T, k, R = case
    gen = torch.Generator(device="cuda").manual_seed(N * H + W + T)
    mk = lambda *s: torch.randn(*s, device="cuda", generator=gen)
    x, dy = mk(N, C, H, W), mk(N, T, H, W)
    fac = [mk(d, R) for d in (T, C, k, k)]
    s = capi.shape_for(x.shape, *fac, k // 2)
    y = capi.layer_forward(s, None, x, *fac, mk(T), "relu")
    dx, grads, dbias = capi.layer_backward(s, None, x, y, dy, *fac, "relu")
    assert capi.layer_last_backward_route() == (capi.ROUTE_DX_FROM_G1 |
                                                (capi.ROUTE_DY_PASS if one_pass else 0))
    masked = dy * (y > 0)
    # against the passes on their own (each checked against float64 elsewhere): fp32 sums in
    # another order, 2^-24 a step of the sum of the terms' magnitudes as a random walk over the
    # terms (a factor of four to spare)
    md = masked.double()
    tol = 4 * 2.0 ** -24 * ((md ** 2).sum(dim=(0, 2, 3)) * N * H * W).sqrt()
    assert ((dbias.double() - md.sum(dim=(0, 2, 3))).abs() <= tol).all()
    want_dx = capi.conv2d_backward_data(masked, *fac, pad=k // 2)
    terms = capi.conv2d_backward_data(masked.abs(), *[f.abs() for f in fac], pad=k // 2)
    assert ((dx - want_dx).abs() <= 4 * (T + 2 * k + R) ** 0.5 * 2.0 ** -24 * terms).all()
    want = capi.conv2d_backward_filter(x, masked, *fac, pad=k // 2)
    terms = capi.conv2d_backward_filter(x.abs(), masked.abs(), *[f.abs() for f in fac], pad=k // 2)
    for g, w, t in zip(grads, want, terms):
        assert ((g - w).abs() <= 4 * 2.0 ** -24 * (N * H * W) ** 0.5 * t).all()


def _float64_gradients(x, dy, fac, k):
    """(dFK, dFC, dFH, dFW, dx) of the layer without an epilogue, factor by factor in float64."""
    (N, C, H, W), P = x.shape, k // 2
    FK, FC, FH, FW, xd = leaves = [f.double().requires_grad_() for f in (*fac, x)]
    R = FK.shape[1]
    A = torch.matmul(FC.t(), xd.flatten(2)).view(N, R, H, W)
    A = torch.nn.functional.pad(A, (P, P, P, P))
    B = sum(FH[i].view(1, R, 1, 1) * A[:, :, i:i + H] for i in range(k))
    Z = sum(FW[j].view(1, R, 1, 1) * B[..., j:j + W] for j in range(k))
    y = torch.matmul(FK, Z.flatten(2))
    return torch.autograd.grad(y, leaves, dy.double().flatten(2))


# Sums over all pixels that nearly cancel: the matrix cores' accumulation comes out low by a
# little whatever its sign, which the pass over dy cancels by alternating signs (over the waves
# in G3, hence in dFC; over a workgroup's chunks in dFK).  Errors in the 2-norm with the
# alternation and without it: T64 dFK 3.4e-7 and 6.8e-7, dFC 4.3e-7 and 3.0e-6; T256 dFK 3.2e-7
# and 4.3e-7, dFC 2.9e-7 and 4.2e-6.  The bounds lie between.
@pytest.mark.parametrize("case,bounds", [
    ((128, 128, 56, 56, 64, 3, 32), (4.8e-7, 1.2e-6)),
    ((32, 256, 56, 56, 256, 3, 32), (3.7e-7, 1.2e-6)),
], ids=["T64", "T256"])
def test_large_layer_factor_gradients_do_not_drift(capi, case, bounds):
    N, C, H, W, T, k, R = case
    gen = torch.Generator(device="cuda").manual_seed(1)
    mk = lambda *s: torch.randn(*s, device="cuda", generator=gen)
    x = mk(N, C, H, W).clamp_(min=0)
    fac = [mk(d, R) * (2.0 / (C * k * k * R)) ** 0.125 for d in (T, C, k, k)]
    s = capi.shape_for(x.shape, *fac, k // 2)
    y = capi.layer_forward(s, None, x, *fac, 0.1 * mk(T), "relu")
    dy = mk(*y.shape)
    _, grads, _ = capi.layer_backward(s, None, x, y, dy, *fac, "relu")
    assert capi.layer_last_backward_route() == capi.ROUTE_DY_PASS | capi.ROUTE_DX_FROM_G1
    want = _float64_gradients(x, dy * (y > 0), fac, k)
    for g, w, bound in zip(grads, want, bounds):          # dFK, dFC
        assert float((g.double() - w).norm() / w.norm()) <= bound


# The passes on their own, dx from their G1.  Before the products of the high parts had
# accumulators of their own: dx 2.3e-7, dFK 3.3e-7 and dFC 7.4e-7 at T256, 1.8e-7, 3.6e-7 and 1.1e-6 at T64
# (the pass of dx from dy 1.8e-7 and 1.7e-7).  The bounds lie between those and what is measured
# now: dx 1.5e-7 and 1.3e-7, dFK and dFC 1.6e-7 to 1.8e-7.
@pytest.mark.parametrize("case,bounds", [
    ((16, 256, 40, 40, 256, 3, 64), {4: 1.7e-7, 0: 2.4e-7, 1: 2.4e-7}),
    ((16, 64, 80, 80, 64, 3, 64), {4: 1.5e-7, 0: 2.4e-7, 1: 2.4e-7}),
], ids=["T256", "T64"])
def test_gradients_of_the_passes_apart_do_not_drift(capi, case, bounds):
    N, C, H, W, T, k, R = case
    gen = torch.Generator(device="cuda").manual_seed(1)
    mk = lambda *s: torch.randn(*s, device="cuda", generator=gen)
    x = mk(N, C, H, W).clamp_(min=0)
    fac = [mk(d, R) * (2.0 / (C * k * k * R)) ** 0.125 for d in (T, C, k, k)]
    s = capi.shape_for(x.shape, *fac, k // 2)
    y = capi.layer_forward(s, None, x, *fac, 0.1 * mk(T), "relu")
    dy = mk(*y.shape)
    dx, grads, _ = capi.layer_backward(s, None, x, y, dy, *fac, "relu")
    assert capi.layer_last_backward_route() == capi.ROUTE_DX_FROM_G1
    want = _float64_gradients(x, dy * (y > 0), fac, k)
    for i, bound in bounds.items():
        got = (*grads, dx)[i]
        assert float((got.double() - want[i]).norm() / want[i].norm()) <= bound


# A first layer of many input channels: half the accumulators of the plain tile kernel, fewer waves
# that share the pixels.  Without balanced sums dFK is 5.8e-7 and dFH 9.4e-7 of its norm off float64,
# 4.3e-7 and 6.7e-7 in the plain kernel on the masked dy, 2.2e-7 and 2.6e-7 with them.
@pytest.mark.parametrize("case", [(16, 16, 112, 112, 48, 3, 16), (8, 16, 112, 110, 64, 3, 16),
                                  (16, 8, 100, 112, 17, 5, 8)], ids=lambda c: "x".join(map(str, c)))
def test_first_layer_factor_gradients_do_not_drift(capi, case):
    N, C, H, W, T, k, R = case
    gen = torch.Generator(device="cuda").manual_seed(1)
    mk = lambda *s: torch.randn(*s, device="cuda", generator=gen)
    x = mk(N, C, H, W).clamp_(min=0)
    fac = [mk(d, R) * (2.0 / (C * k * k * R)) ** 0.125 for d in (T, C, k, k)]
    s = capi.shape_for(x.shape, *fac, k // 2)
    y = capi.layer_forward(s, None, x, *fac, 0.1 * mk(T), "relu")
    dy = mk(*y.shape)
    grads = capi.layer_backward(s, None, x, y, dy, *fac, "relu", False, True, True)[1]
    assert capi.layer_last_backward_route() == capi.ROUTE_MASKED_TILES
    masked = dy * (y > 0)
    want = _float64_gradients(x, masked, fac, k)
    plain = capi.conv2d_backward_filter(x, masked, *fac, pad=k // 2)
    error = lambda g, w: float((g.double() - w).norm() / w.norm())
    for g, p, w in zip(grads, plain, want):
        assert error(g, w) <= 1.1 * error(p, w)
        assert error(g, w) <= 4e-7


# The same layers and one of three channels: in no gradient further from float64 than the plain kernel.
@pytest.mark.parametrize("case", [(16, 16, 112, 112, 48, 3, 16), (8, 16, 112, 110, 64, 3, 16),
                                  (16, 3, 112, 112, 32, 5, 16)], ids=lambda c: "x".join(map(str, c)))
def test_first_layer_factor_gradients_no_further_off_than_the_plain_kernels(capi, case):
    N, C, H, W, T, k, R = case
    gen = torch.Generator(device="cuda").manual_seed(1)
    mk = lambda *s: torch.randn(*s, device="cuda", generator=gen)
    x = mk(N, C, H, W).clamp_(min=0)
    fac = [mk(d, R) * (2.0 / (C * k * k * R)) ** 0.125 for d in (T, C, k, k)]
    s = capi.shape_for(x.shape, *fac, k // 2)
    y = capi.layer_forward(s, None, x, *fac, 0.1 * mk(T), "relu")
    dy = mk(*y.shape)
    grads = capi.layer_backward(s, None, x, y, dy, *fac, "relu", False, True, True)[1]
    assert capi.layer_last_backward_route() == capi.ROUTE_MASKED_TILES
    masked = dy * (y > 0)
    want = _float64_gradients(x, masked, fac, k)
    plain = capi.conv2d_backward_filter(x, masked, *fac, pad=k // 2)
    for g, p, w in zip(grads, plain, want):
        assert float((g.double() - w).norm()) <= float((p.double() - w).norm())


def test_first_layer_bias_gradient_adds_up_in_short_chains(capi):
    """Its error against float64 is that of a tree of sums (1.5e-7 over these seeds; 2.7e-7 with
    a slot's, then a channel's entries added one after the other)."""
    N, C, H, W, T, k, R = 64, 3, 128, 128, 16, 3, 16
    errors = []
    for seed in range(4):
        gen = torch.Generator(device="cuda").manual_seed(seed)
        mk = lambda *s: torch.randn(*s, device="cuda", generator=gen)
        x, fac = mk(N, C, H, W), [mk(d, R) * (2.0 / (C * k * k * R)) ** 0.125 for d in (T, C, k, k)]
        s = capi.shape_for(x.shape, *fac, k // 2)
        y = capi.layer_forward(s, None, x, *fac, 0.1 * mk(T), "relu")
        dy = mk(*y.shape)
        dbias = capi.layer_backward(s, None, x, y, dy, *fac, "relu", False, True, True)[2]
        assert capi.layer_last_backward_route() == capi.ROUTE_MASKED_TILES
        want = (dy * (y > 0)).double().sum(dim=(0, 2, 3))
        errors.append(float((dbias.double() - want).norm() / want.norm()))
    assert (sum(e * e for e in errors) / 4) ** 0.5 <= 2e-7
