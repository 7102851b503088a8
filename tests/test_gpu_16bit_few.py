"""16-bit layers of few channels: the few-channel and the recomposed-filter kernel on bfloat16 and
half-precision activations, where the producer / consumer kernel ran before.

The kernels widen exactly, sum in fp32 and round once: against float64 (of the 16-bit inputs) the
bound is half a unit in the last place of the result's type, at most 2^-8 or 2^-11 of the value, and 1e-5 of
the result's largest value for the sums in fp32."""
import numpy as np
import pytest
import torch

import paralleltnnlayers_amd as cp4
from paralleltnnlayers_amd import capi

pytestmark = pytest.mark.gpu

TYPES = {"bf16": (torch.bfloat16, 2.0 ** -8, capi.conv2d_forward_bf16, capi.conv2d_backward_data_bf16),
         "f16": (torch.float16, 2.0 ** -11, capi.conv2d_forward_f16, capi.conv2d_backward_data_f16)}

FEW, DENSE, PIPE = "mfma_bf16x3_few", "dense_small_valu", "mfma_bf16x3_pipe"

# (shape, the kernel of the forward pass, that of the input gradient)
SHAPES = [
    # few-channel kernel: one, two rows of tiles; odd and even rows; one chunk of channels and two
    ((9, 5, 14, 97, 83, 3, 6), FEW, FEW), ((8, 16, 16, 96, 128, 3, 16), FEW, FEW),
    ((2, 32, 33, 200, 161, 3, 16), FEW, PIPE), ((5, 17, 31, 120, 130, 5, 3), FEW, FEW),
    ((61, 3, 64, 33, 32, 3, 16), FEW, PIPE), ((70, 12, 5, 47, 47, 1, 9), FEW, FEW),
    ((3, 31, 64, 151, 138, 1, 16), FEW, PIPE), ((20, 4, 64, 57, 56, 5, 8), FEW, PIPE),
    # recomposed filter: whole tiles of 64 columns and ragged ones, groups of eight channels, ranks past 16
    ((1, 1, 1, 260, 260, 5, 1), DENSE, DENSE), ((2, 2, 7, 240, 240, 3, 20), DENSE, PIPE),
    ((3, 1, 9, 88, 107, 3, 21), DENSE, PIPE), ((9, 3, 2, 128, 64, 7, 20), DENSE, DENSE),
    ((9, 2, 11, 41, 128, 1, 30), DENSE, DENSE), ((2, 1, 9, 136, 181, 1, 27), DENSE, DENSE),
    ((8, 9, 1, 146, 128, 3, 27), DENSE, DENSE), ((5, 9, 1, 195, 170, 5, 30), DENSE, DENSE),
    ((7, 1, 2, 30, 76, 5, 20), DENSE, DENSE),
    # on the other side of the rules
    ((4, 4, 3, 130, 70, 5, 30), PIPE, PIPE), ((2, 12, 1, 300, 101, 1, 27), PIPE, DENSE),
    ((1, 16, 4, 500, 128, 3, 24), PIPE, PIPE),
    # rows that leave much of a tile of 32 columns empty: strips of whole rows with up to four ranks, by the
    # number of pixels and of output channels; tiles with more ranks
    ((39, 3, 24, 66, 66, 3, 4), PIPE, PIPE), ((39, 3, 24, 66, 66, 3, 5), FEW, PIPE),
    ((57, 4, 64, 40, 40, 3, 2), PIPE, PIPE), ((40, 4, 64, 40, 40, 3, 2), FEW, PIPE),
    ((57, 4, 32, 40, 40, 3, 2), FEW, FEW),
]


def _inputs(N, C, T, H, W, k, R, seed):
    gen = torch.Generator().manual_seed(seed)
    f = [torch.randn(d, R, generator=gen) * (2.0 / (C * k * k * R)) ** 0.125 for d in (T, C, k, k)]
    return gen, f, torch.einsum("tr,cr,hr,wr->tchw", *[v.double() for v in f])


@pytest.mark.parametrize("kind", ["bf16", "f16"])
@pytest.mark.parametrize("shape,forward_kernel,backward_kernel", SHAPES,
                         ids=["x".join(map(str, s[0])) for s in SHAPES])
@pytest.mark.parametrize("bias", [False, True])
def test_passes_over_activations(shape, forward_kernel, backward_kernel, kind, bias):
    N, C, T, H, W, k, R = shape
    dtype, ulp, forward, backward_data = TYPES[kind]
    s = capi.Shape(N=N, H=H, W=W, pad=k // 2, T=T, C=C, Y=k, X=k, Rank=R)
    assert capi.plan_query(s, "forward", dtype)["variant"] == forward_kernel
    assert capi.plan_query(s, "backward_data", dtype)["variant"] == backward_kernel
    gen, f, K = _inputs(*shape, seed=7)
    fd = [v.cuda() for v in f]
    x = torch.randn(N, C, H, W, generator=gen).to(dtype)
    b = 0.1 * torch.randn(T, generator=gen)
    want = torch.nn.functional.conv2d(x.double(), K, b.double() if bias else None, padding=k // 2)
    if bias:
        want = want.clamp(min=0)
        got = forward(x.cuda(), *fd, bias=b.cuda(), activation="relu", pad=k // 2)
    else:
        got = forward(x.cuda(), *fd, pad=k // 2)
    err = (got.cpu().double() - want).abs()
    assert (err <= ulp * want.abs() + 1e-5 * want.abs().max()).all()
    if bias:
        return
    dy = torch.randn(N, T, H, W, generator=gen).to(dtype)
    want = torch.nn.functional.conv_transpose2d(dy.double(), K, padding=k // 2)
    err = (backward_data(dy.cuda(), *fd, pad=k // 2).cpu().double() - want).abs()
    assert (err <= ulp * want.abs() + 1e-5 * want.abs().max()).all()


@pytest.mark.parametrize("shape", [(9, 5, 14, 97, 84, 3, 6), (2, 2, 7, 128, 128, 3, 20)])
def test_operands_off_their_boundaries(shape):
    """Activations that start on a 2-byte boundary only: narrower loads and stores, the same values."""
    N, C, T, H, W, k, R = shape
    gen, f, _ = _inputs(*shape, seed=3)
    fd = [v.cuda() for v in f]
    x = torch.randn(N, C, H, W, generator=gen).to(torch.bfloat16).cuda()
    want = capi.conv2d_forward_bf16(x, *fd, pad=k // 2)
    odd = torch.empty(x.numel() + 1, dtype=x.dtype, device="cuda")[1:].view(x.shape)
    odd.copy_(x)
    out = torch.empty(want.numel() + 1, dtype=x.dtype, device="cuda")[1:].view(want.shape)
    capi.conv2d_forward_bf16(odd, *fd, pad=k // 2, out=out)
    assert torch.equal(out, want)


@pytest.mark.parametrize("kind", ["bf16", "f16"])
def test_a_value_that_is_not_finite_reaches_its_outputs(kind):
    dtype, _, forward, _ = TYPES[kind]
    for shape in ((8, 5, 14, 96, 84, 3, 6), (2, 2, 7, 128, 128, 3, 20)):
        N, C, T, H, W, k, R = shape
        gen, f, _ = _inputs(*shape, seed=11)
        x = torch.randn(N, C, H, W, generator=gen).to(dtype)
        x[0, 1, 40, 50] = float("nan")
        y = forward(x.cuda(), *[v.cuda() for v in f], pad=1).cpu()
        assert torch.isnan(y[0, :, 39:42, 49:52]).all()
        assert torch.isnan(y).sum() == 9 * T
