"""Results that go through the L2, past the memory-side cache or by plain stores, by their size and
where their planes start (csrc/store_policy.h): every kernel that chooses, at either side of its
lines, against float64 on the first and the last image."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def cp4():
    import paralleltnnlayers_amd as m
    m.lib()
    assert torch.cuda.is_available()
    return m


def reference(x, fac, k, b=None):
    """y and the sum of its terms' magnitudes, factor by factor in float64."""
    out = []
    for d, f in ((x.double(), [t.double() for t in fac]), (x.double().abs(), [t.double().abs() for t in fac])):
        (N, C, H, W), (FK, FC, FH, FW), P = d.shape, f, k // 2
        A = torch.matmul(FC.t(), d.flatten(2)).view(N, -1, H, W)
        A = torch.nn.functional.pad(A, (P, P, P, P))
        B = sum(FH[i].view(1, -1, 1, 1) * A[:, :, i:i + H] for i in range(k))
        Z = sum(FW[j].view(1, -1, 1, 1) * B[..., j:j + W] for j in range(k))
        y = torch.matmul(FK, Z.flatten(2)).view(N, -1, H, W)
        if b is not None:
            y = y + (b.double() if not out else b.double().abs()).view(1, -1, 1, 1)
        out.append(y)
    return out


# streamed (from 96 MB, behind an epilogue from 128 MB), through, off the lines small and large: whole
# rows, tiles of wide planes, the few-channel kernel
@pytest.mark.parametrize("bias", [False, True], ids=["plain", "bias"])
@pytest.mark.parametrize("dims", [(44, 64, 56, 56, 256, 1, 16), (44, 64, 56, 56, 256, 3, 32),
                                  (44, 320, 56, 56, 256, 5, 16), (11, 64, 224, 224, 64, 3, 16),
                                  (8, 16, 512, 512, 16, 3, 16), (4, 16, 512, 512, 16, 3, 16),
                                  (16, 64, 66, 66, 64, 3, 16), (2, 64, 66, 66, 64, 3, 16),
                                  (40, 16, 102, 90, 16, 3, 8), (2, 16, 102, 90, 16, 3, 8)],
                         ids=lambda d: "x".join(map(str, d)))
def test_forward(cp4, dims, bias):
    N, C, H, W, T, k, R = dims
    gen = torch.Generator(device="cuda").manual_seed(sum(dims))
    mk = lambda *s: torch.randn(*s, device="cuda", generator=gen)
    x, fac = mk(N, C, H, W), [mk(d, R) for d in (T, C, k, k)]
    b = mk(T) if bias else None
    y = (cp4.conv2d_forward_bias_act(x, *fac, b, None, pad=k // 2) if bias
         else cp4.conv2d_forward(x, *fac, pad=k // 2))
    ends = [0, N - 1]
    want, terms = reference(x[ends], fac, k, b)
    # fp32 contractions and taps: 2^-24 a step of the terms' magnitudes as a random walk (a factor of
    # four to spare)
    assert ((y[ends].double() - want).abs() <= 4 * (C + 2 * k + R) ** 0.5 * 2.0 ** -24 * terms).all()


def factor_gradients(x, dy, fac, k):
    """dFK, dFC, dFH, dFW of the layer without an epilogue by autograd in float64."""
    (N, C, H, W), P = x.shape, k // 2
    FK, FC, FH, FW = f = [t.double().requires_grad_() for t in fac]
    A = torch.nn.functional.pad(torch.matmul(FC.t(), x.double().flatten(2)).view(N, -1, H, W), (P, P, P, P))
    B = sum(FH[i].view(1, -1, 1, 1) * A[:, :, i:i + H] for i in range(k))
    Z = sum(FW[j].view(1, -1, 1, 1) * B[..., j:j + W] for j in range(k))
    return torch.autograd.grad(torch.matmul(FK, Z.flatten(2)), f, dy.double().flatten(2))


# the input gradient beside the factors': dx streamed, through and off the lines
@pytest.mark.parametrize("dims", [(36, 256, 56, 56, 64, 3, 16), (8, 64, 56, 56, 64, 3, 64),
                                  (40, 64, 58, 58, 64, 3, 64), (2, 64, 36, 36, 64, 3, 64)],
                         ids=lambda d: "x".join(map(str, d)))
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
def test_layer_backward(cp4, dims, dtype):
    N, C, H, W, T, k, R = dims
    capi = cp4.capi
    gen = torch.Generator(device="cuda").manual_seed(sum(dims))
    mk = lambda *s: torch.randn(*s, device="cuda", generator=gen)
    x, fac = mk(N, C, H, W).to(dtype), [mk(d, R) for d in (T, C, k, k)]
    s = capi.shape_for(x.shape, *fac, k // 2)
    y = capi.layer_forward(s, None, x, *fac, mk(T), "relu")
    dy = mk(*y.shape).to(dtype)
    dx, grads, dbias = capi.layer_backward(s, None, x, y, dy, *fac, "relu")
    masked = dy * (y > 0)
    ends = [0, N - 1]
    flipped = [fac[1], fac[0], fac[2].flip(0), fac[3].flip(0)]
    want, terms = reference(masked[ends], flipped, k)
    eps = 2.0 ** -8 if dtype == torch.bfloat16 else 0.0
    bound = 4 * (T + 2 * k + R) ** 0.5 * 2.0 ** -24 * terms + eps * want.abs()
    assert ((dx[ends].double() - want).abs() <= bound).all()
    # the factor gradients in float64: n roundings of 2^-24 grow as sqrt(n), as sums of n terms with signs at
    # random do; times 4 for the stages one after the other
    near = 4 * 2.0 ** -24 * (T + C + R + 2 * k + N * H * W) ** 0.5
    for g, w in zip(grads, factor_gradients(x, masked, fac, k)):
        assert (g.double() - w).norm() <= near * w.norm()
    # and their intermediates: the same call without dx and bias computes them again
    alone = capi.layer_backward(s, None, x, None, masked, *fac, None, False, True, False)[1]
    mags = capi.layer_backward(s, None, x.abs(), None, masked.abs(), *[f.abs() for f in fac], None, False,
                               True, False)[1]
    for g, w, t in zip(grads, alone, mags):
        assert ((g - w).abs() <= 4 * 2.0 ** -24 * (N * H * W) ** 0.5 * t).all()


# results that the next launch reads again - another pass, the bias kernel -, at either side of the lines;
# strips of three, five and eight rows, small, large and too large to go through
@pytest.mark.parametrize("bias", [False, True], ids=["plain", "bias"])
@pytest.mark.parametrize("dims", [(36, 64, 56, 56, 256, 1, 128), (44, 64, 56, 56, 256, 1, 96),
                                  (33, 64, 56, 56, 256, 1, 64), (44, 64, 56, 56, 256, 3, 48),
                                  (12, 64, 56, 56, 256, 3, 32), (20, 64, 56, 56, 256, 3, 32),
                                  (26, 64, 56, 56, 256, 3, 32)], ids=lambda d: "x".join(map(str, d)))
def test_forward_read_again(cp4, dims, bias):
    test_forward(cp4, dims, bias)
