"""The matrix-core factor gradients on planes whose rows do not move as aligned 16-byte pieces:
sizes around a piece and around a chunk of 32 pixels, one and two rank tiles, every activation
type, against the general kernel."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("plane", [(1, 1), (1, 3), (1, 5), (3, 11), (5, 7), (3, 21), (9, 11), (2, 17)],
                         ids=lambda p: "x".join(map(str, p)))
@pytest.mark.parametrize("rank", [7, 40])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16],
                         ids=["f32", "bf16", "f16"])
def test_odd_planes(plane, rank, dtype):
    import paralleltnnlayers_amd.capi as capi
    H, W = plane
    N, C, T, k = 3, 48, 160, 3
    gen = torch.Generator(device="cuda").manual_seed(H * W + rank)
    mk = lambda *s: torch.randn(*s, device="cuda", generator=gen)
    x, dy = mk(N, C, H, W).to(dtype), mk(N, T, H, W).to(dtype)
    fac = [mk(d, rank) for d in (T, C, k, k)]
    if dtype == torch.float32:
        got = capi.conv2d_backward_filter(x, dy, *fac, pad=1, variant=1)
    else:
        run = (capi.conv2d_backward_filter_bf16 if dtype == torch.bfloat16
               else capi.conv2d_backward_filter_f16)
        got = run(x, dy, *fac, pad=1)
    want = capi.conv2d_backward_filter(x.float(), dy.float(), *fac, pad=1, variant=0)
    terms = capi.conv2d_backward_filter(x.float().abs(), dy.float().abs(), *[f.abs() for f in fac],
                                        pad=1, variant=0)
    # the same fp32 sums (channels, taps, ranks, pixels) in another order on either side: 2^-24 a
    # step as a random walk over the terms, a factor of four to spare
    steps = (T + C + 4 * k + rank + N * H * W) ** 0.5
    for g, w, t in zip(got, want, terms):
        assert ((g - w).abs() <= 4 * 2.0 ** -24 * steps * t + 1e-30).all()


# waves of the gradient GEMM without a row of their own (32 channels a wave, four waves a workgroup), one to
# five chunks of 32 pixels
@pytest.mark.parametrize("channels", [(2, 34), (30, 98), (16, 144), (128, 48)], ids=lambda c: "x".join(map(str, c)))
@pytest.mark.parametrize("plane", [(4, 8), (4, 10), (8, 12), (8, 16), (9, 16)], ids=lambda p: "x".join(map(str, p)))
@pytest.mark.parametrize("rank", [5, 64])
def test_waves_without_a_row(channels, plane, rank):
    import paralleltnnlayers_amd.capi as capi
    (C, T), (H, W), N, k = channels, plane, 3, 3
    gen = torch.Generator(device="cuda").manual_seed(C + T + H * W + rank)
    mk = lambda *s: torch.randn(*s, device="cuda", generator=gen)
    fac = [mk(d, rank) for d in (T, C, k, k)]
    steps = (T + C + 4 * k + rank + N * H * W) ** 0.5
    for dtype in [torch.float32] + [torch.bfloat16, torch.float16] * (C % 16 == T % 16 == 0):
        x, dy = mk(N, C, H, W).to(dtype), mk(N, T, H, W).to(dtype)
        if dtype == torch.float32:
            got = capi.conv2d_backward_filter(x, dy, *fac, pad=1, variant=1)
        else:
            run = (capi.conv2d_backward_filter_bf16 if dtype == torch.bfloat16
                   else capi.conv2d_backward_filter_f16)
            got = run(x, dy, *fac, pad=1)
        want = capi.conv2d_backward_filter(x.float(), dy.float(), *fac, pad=1, variant=0)
        terms = capi.conv2d_backward_filter(x.float().abs(), dy.float().abs(), *[f.abs() for f in fac],
                                            pad=1, variant=0)
        for g, w, t in zip(got, want, terms):       # (as above)
            assert ((g - w).abs() <= 4 * 2.0 ** -24 * steps * t + 1e-30).all()
