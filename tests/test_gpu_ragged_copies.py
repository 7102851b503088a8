"""Factor gradients of ragged channel counts: x, dy and the factors are copied with zero channels
appended in one launch, the gradients copied back in another.  The copies are checked through the
gradients, against float64: products of the copies are exact, sums in fp32, 1e-4 of each gradient's
largest value as elsewhere for these kernels."""
import pytest
import torch

import paralleltnnlayers_amd as cp4

pytestmark = pytest.mark.gpu


# channel counts that need copies of x, of dy, of both; rows of whole quads and not; one image and many
@pytest.mark.parametrize("shape", [
    (2, 33, 64, 8, 8, 3, 4), (3, 64, 37, 7, 9, 3, 6), (5, 157, 7, 20, 24, 3, 4), (1, 63, 1, 34, 34, 5, 25),
    (9, 45, 65, 15, 15, 3, 33), (130, 65, 35, 7, 7, 1, 3), (2, 341, 5, 41, 27, 3, 5)],
    ids=lambda s: "x".join(map(str, s)))
def test_gradients(shape):
    N, C, T, H, W, k, R = shape
    gen = torch.Generator().manual_seed(1)
    f = [torch.randn(d, R, generator=gen) * (2.0 / (C * k * k * R)) ** 0.125 for d in (T, C, k, k)]
    x, dy = torch.randn(N, C, H, W, generator=gen), torch.randn(N, T, H, W, generator=gen)
    got = cp4.conv2d_backward_filter(x.cuda(), dy.cuda(), *[v.cuda() for v in f], pad=k // 2)
    fd = [v.double().requires_grad_() for v in f]
    K = torch.einsum("tr,cr,hr,wr->tchw", *fd)
    torch.nn.functional.conv2d(x.double(), K, padding=k // 2).backward(dy.double())
    for g, w in zip(got, fd):
        err = (g.cpu().double() - w.grad).abs().max()
        assert err <= 1e-4 * w.grad.abs().max()
