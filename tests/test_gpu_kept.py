"""What a training step's forward call leaves for its backward call (cp4_layer_forward_keeping,
cp4_layer_backward_kept): the signs of y, against the backward call that reads y itself and against
float64.  Keeping them changes no bit of y nor of any gradient."""
import ctypes

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu

MASK = 1                                  # CP4_KEEP_*
KEPT_MASK = 8                             # CP4_ROUTE_*


@pytest.fixture(scope="module")
def capi():
    import paralleltnnlayers_amd.capi as c
    c.lib()
    assert torch.cuda.is_available()
    return c


def _shift(z, i, j, k):
    p, H, W = k // 2, *z.shape[2:]
    return F.pad(z, (p, p, p, p))[:, :, i:i + H, j:j + W]


def _exact(x, dy, FK, FC, FH, FW, k):
    """dx, (dFK, dFC, dFH, dFW), dbias in float64, factor by factor."""
    N, C, H, W = x.shape
    R, T = FK.shape[1], dy.shape[1]
    x, dy, FK, FC, FH, FW = (t.double() for t in (x, dy, FK, FC, FH, FW))
    row = lambda f, i: f[i].view(1, R, 1, 1)
    A = torch.matmul(FC.t().contiguous(), x.view(N, C, -1)).view(N, R, H, W)
    B = sum(row(FH, i) * _shift(A, i, k // 2, k) for i in range(k))
    Cc = sum(row(FW, j) * _shift(B, k // 2, j, k) for j in range(k))
    G3 = torch.matmul(FK.t().contiguous(), dy.view(N, T, -1)).view(N, R, H, W)
    G2 = sum(row(FW, j) * _shift(G3, k // 2, k - 1 - j, k) for j in range(k))
    G1 = sum(row(FH, i) * _shift(G2, k - 1 - i, k // 2, k) for i in range(k))
    mm = lambda a, b: sum(a[n].view(a.shape[1], -1) @ b[n].view(R, -1).t() for n in range(N))
    dFW = torch.stack([(G3 * _shift(B, k // 2, j, k)).sum((0, 2, 3)) for j in range(k)])
    dFH = torch.stack([(G2 * _shift(A, i, k // 2, k)).sum((0, 2, 3)) for i in range(k)])
    dx = torch.matmul(FC, G1.view(N, R, -1)).view(N, C, H, W)
    return dx, (mm(dy, Cc), mm(x, G1), dFH, dFW), dy.sum((0, 2, 3))


def _inputs(N, C, H, W, T, k, R):
    gen = torch.Generator(device="cuda").manual_seed(N + C + H + W + T + R)
    mk = lambda *s: torch.randn(*s, device="cuda", generator=gen)
    return mk(N, C, H, W).clamp_(min=0), mk(N, T, H, W), [mk(d, R) for d in (T, C, k, k)], mk(T)


def _forward(capi, s, x, fac, bias, wanted):
    L, p = capi.lib(), lambda t: ctypes.c_void_p(t.data_ptr())
    L.cp4_layer_kept_bytes.restype = ctypes.c_size_t
    room = L.cp4_layer_kept_bytes(ctypes.byref(s), None, 0, 1, wanted)
    y = torch.empty(s.N, s.T, s.H, s.W, device="cuda")
    kept = torch.full((max(room, 1),), 0x55, device="cuda", dtype=torch.uint8)
    parts = ctypes.c_int(-1)
    capi.check(L.cp4_layer_forward_keeping(
        ctypes.byref(s), None, 0, p(x), *map(p, fac), p(bias), 1, wanted, p(y), p(kept),
        ctypes.c_size_t(room), ctypes.byref(parts), None, ctypes.c_size_t(0), None))
    return y, kept, parts.value


def _backward(capi, s, x, y, dy, fac, wanted, kept, parts):
    L, p = capi.lib(), lambda t: ctypes.c_void_p(t.data_ptr()) if t is not None else None
    need = L.cp4_layer_backward_workspace_bytes(ctypes.byref(s), None, 0, 1, wanted)
    ws = torch.empty(max(need, 1), device="cuda", dtype=torch.uint8)
    dx = torch.empty_like(x) if wanted & 1 else None
    grads, dbias = [torch.empty_like(f) for f in fac], torch.empty(s.T, device="cuda")
    capi.check(L.cp4_layer_backward_kept(
        ctypes.byref(s), None, 0, p(x), p(y), p(dy), *map(p, fac), 1, p(dx), *map(p, grads), p(dbias),
        p(kept), ctypes.c_size_t(kept.numel()), parts, p(ws), ctypes.c_size_t(need), None))
    return dx, grads, dbias, L.cp4_layer_last_backward_route()


# First layers, behind which the direct filter gradient reads the signs: whole and ragged blocks of channels,
# every filter; rows of an odd number of fours, whose last signs are half a load, down to the image's
# last row; one to four blocks of 16 channels, one to five of columns.
TILES = [(5, 3, 352, 360, 33, 3, 4), (6, 3, 227, 228, 64, 3, 16), (24, 4, 214, 220, 16, 3, 8), (13, 4, 203, 212, 32, 3, 8),
         (28, 6, 213, 220, 13, 1, 4), (8, 1, 225, 236, 64, 5, 5), (11, 2, 229, 236, 31, 5, 6), (17, 8, 180, 184, 32, 1, 8),
         (8, 3, 224, 228, 48, 5, 16)]
# ... and the tile kernel, which reads y: rows off the multiples of four, more than 15 blocks
LEFT_OUT = [(4, 3, 351, 353, 34, 3, 16), (17, 8, 180, 182, 32, 1, 8), (6, 3, 224, 228, 64, 5, 16)]
# The pass over dy: producers that split the channels (whole and ragged quarters, one rank quad past a
# half, 2 to 8 blocks of output channels) and, with few channels, whole blocks.
PASSES = [(12, 256, 56, 56, 256, 3, 32), (48, 80, 52, 60, 96, 3, 17), (40, 128, 40, 44, 256, 1, 20),
          (24, 64, 80, 80, 256, 1, 32), (40, 16, 60, 64, 128, 3, 8)]


@pytest.mark.parametrize("dims", TILES + PASSES, ids=lambda d: "x".join(map(str, d)))
def test_backward_from_what_the_forward_left(capi, dims):
    N, C, H, W, T, k, R = dims
    x, dy, fac, bias = _inputs(*dims)
    s = capi.shape_for(x.shape, *fac, k // 2)
    wanted = 6 if dims in TILES else 7            # factors and bias; dx too
    y, kept, left = _forward(capi, s, x, fac, bias, wanted)
    assert left == MASK
    # the signs: 16 bits a pixel and half, bit 4 a + b of half h is channel 8 a + 4 h + b
    nkb = (T + 31) // 32
    bits = kept[:N * nkb * H * W * 4].view(torch.int16).view(N, nkb, 2, H * W)
    for c in {0, 3, 4, 8, T // 2, T - 1}:
        word = bits[:, c // 32, c // 4 % 2].int()
        assert torch.equal(word >> (4 * (c % 32 // 8) + c % 4) & 1, (y[:, c].view(N, -1) > 0).int())
    # y is what the call that keeps nothing gives
    assert torch.equal(y, capi.layer_forward(s, None, x, *fac, bias, "relu"))
    got = _backward(capi, s, x, y, dy, fac, wanted, kept, left)
    want = _backward(capi, s, x, y, dy, fac, wanted, kept, 0)
    assert got[3] == want[3] | KEPT_MASK
    # nothing but where the mask comes from differs
    assert torch.equal(got[2], want[2])
    assert got[0] is None or torch.equal(got[0], want[0])
    assert all(torch.equal(a, b) for a, b in zip(got[1], want[1]))
    if dims in TILES or T // 32 % 2:              # (an odd number of blocks of output channels leaves one
        return                                    # block's share of the matrix cores' drift in G3: 1.3e-6)
    exact = _exact(x, dy * (y > 0), *fac, k)
    # exact products; each sum rounds by 2^-24 a term, which over the C + T + R channels and ranks and 2 k taps
    # of an entry add up as a random walk
    tol = 2.0 ** -24 * (C + T + R + 2 * k) ** 0.5
    for a, b in zip([got[0]] + got[1], (exact[0],) + exact[1]):
        assert (a.double() - b).norm() <= tol * b.norm()


@pytest.mark.parametrize("dims", LEFT_OUT, ids=lambda d: "x".join(map(str, d)))
def test_nothing_is_kept_for_the_tile_kernel(capi, dims):
    x, _, fac, bias = _inputs(*dims)
    s = capi.shape_for(x.shape, *fac, dims[5] // 2)
    y, kept, left = _forward(capi, s, x, fac, bias, 6)
    assert left == 0 and kept.numel() == 1
    assert torch.equal(y, capi.layer_forward(s, None, x, *fac, bias, "relu"))


def test_signs_are_left_alone_where_operands_are_off_their_boundaries(capi):
    """The direct filter gradient wants 16-byte boundaries; without them the tile kernel reads y."""
    N, C, H, W, T, k, R = dims = TILES[1]
    x, dy, fac, bias = _inputs(*dims)
    s = capi.shape_for(x.shape, *fac, k // 2)
    y, kept, left = _forward(capi, s, x, fac, bias, 6)
    assert left == MASK
    off = torch.empty(dy.numel() + 1, device="cuda")[1:].view_as(dy).copy_(dy)
    got = _backward(capi, s, x, y, off, fac, 6, kept, left)
    want = _backward(capi, s, x, y, off, fac, 6, kept, 0)
    assert got[3] == want[3] and not got[3] & KEPT_MASK
    assert all(torch.equal(a, b) for a, b in zip([got[2]] + got[1], [want[2]] + want[1]))


@pytest.mark.parametrize("dims", TILES + LEFT_OUT + PASSES, ids=lambda d: "x".join(map(str, d)))
def test_a_training_steps_output_is_that_of_inference(capi, dims):
    from paralleltnnlayers_amd import torch_ops
    N, C, H, W, T, k, R = dims
    x, _, fac, bias = _inputs(*dims)
    layer = torch_ops.CP4Conv2d(C, T, k, R, bias=True, activation="relu")
    with torch.no_grad():
        for p, f in zip((layer.FK, layer.FC, layer.FH, layer.FW, layer.bias), fac + [bias]):
            p.copy_(f)
        want = layer(x)
    assert torch.equal(layer(x.clone().requires_grad_(dims in PASSES)).detach(), want)


def test_layer_under_hooks_on_saved_tensors(capi):
    """What hooks give back - moved and returned, or as another type - changes no gradient."""
    from paralleltnnlayers_amd import torch_ops
    N, C, H, W, T, k, R = 12, 256, 56, 56, 256, 3, 32
    x, dy, fac, bias = _inputs(N, C, H, W, T, k, R)
    layer = torch_ops.CP4Conv2d(C, T, k, R, bias=True, activation="relu")
    with torch.no_grad():
        for p, f in zip((layer.FK, layer.FC, layer.FH, layer.FW, layer.bias), fac + [bias]):
            p.copy_(f)

    def grads():
        xi = x.clone().requires_grad_()
        layer.zero_grad(set_to_none=True)
        layer(xi).backward(dy)
        return [xi.grad] + [p.grad for p in layer.parameters()]

    want = grads()
    with torch.autograd.graph.save_on_cpu():
        assert all(torch.equal(a, b) for a, b in zip(grads(), want))
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t.float(), lambda t: t):
        got = grads()                             # (the bytes as floats: not taken up)
    assert all(torch.equal(a, b) for a, b in zip(got, want))
