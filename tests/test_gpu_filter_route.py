"""Factor gradients on either side of the pixel lines between the three-launch and the four-launch
variant (csrc/bwd_filter_fused.hip), against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def cp4():
    import paralleltnnlayers_amd as m
    m.lib()
    assert torch.cuda.is_available()
    return m


def reference(x, dy, fac, k):
    """(dFK, dFC, dFH, dFW) by autograd over the four contractions in float64 on the CPU."""
    x, dy = x.double().cpu(), dy.double().cpu()
    FK, FC, FH, FW = f = [t.double().cpu().requires_grad_() for t in fac]
    (N, C, H, W), P = x.shape, k // 2
    A = torch.nn.functional.pad((x.flatten(2).transpose(1, 2) @ FC).transpose(1, 2).reshape(N, -1, H, W),
                                (P, P, P, P))
    B = sum(FH[i].view(1, -1, 1, 1) * A[:, :, i:i + H] for i in range(k))
    Z = sum(FW[j].view(1, -1, 1, 1) * B[..., j:j + W] for j in range(k))
    y = (Z.flatten(2).transpose(1, 2) @ FK.t()).transpose(1, 2).reshape(N, -1, H, W)
    return torch.autograd.grad(y, f, dy)


@pytest.mark.parametrize("dims,route", [
    ((16, 32, 28, 28, 32, 5, 8), "mfma_fused_taps"),          # 12,544 pixels: the line itself
    ((17, 32, 28, 28, 32, 5, 8), "mfma_four_launches"),
    ((66, 48, 14, 14, 32, 5, 20), "mfma_four_launches"),      # few pixels a plane, ragged rank
    ((4, 32, 56, 60, 48, 5, 40), "mfma_four_launches"),       # unequal sides, two rank tiles
    ((49, 32, 28, 28, 48, 3, 16), "mfma_fused_taps"),         # 38,416 pixels
    ((50, 32, 28, 28, 48, 3, 16), "mfma_four_launches"),      # 39,200
    ((50, 32, 28, 28, 48, 3, 17), "mfma_fused_taps"),         # a rank above 16 keeps the wider line
], ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else v)
def test_either_side_of_the_line(cp4, dims, route):
    N, C, H, W, T, k, R = dims
    gen = torch.Generator(device="cuda").manual_seed(sum(dims))
    mk = lambda *s: torch.randn(*s, device="cuda", generator=gen)
    x, dy, fac = mk(N, C, H, W), mk(N, T, H, W), [mk(d, R) for d in (T, C, k, k)]
    s = cp4.capi.shape_for(x.shape, *fac, k // 2)
    assert cp4.capi.plan_query(s, "backward_filter")["variant"] == route
    grads = cp4.conv2d_backward_filter(x, dy, *fac, pad=k // 2)
    # each gradient is a sum of n = N H W products per element, signs at random: its size grows as
    # sqrt(n), and m roundings of partial sums in fp32 (2^-24 each) as 2^-24 sqrt(m) of that size.  A
    # matrix instruction adds 16 pixels at a time: m = n / 16, and the channels and taps before them;
    # times 4 for the contraction, the taps, the sums and the tap gradients' sum over the ranks' planes
    bound = 4 * 2.0 ** -24 * (N * H * W / 16 + C + T + 2 * k) ** 0.5
    for name, g, want in zip(("FK", "FC", "FH", "FW"), grads, reference(x, dy, fac, k)):
        err = ((g.double().cpu() - want).norm() / want.norm()).item()
        assert err <= bound, (name, err, bound)
