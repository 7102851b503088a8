"""Dense filter gradient with dy straight from memory (bwd_filter_dense_direct.hip): the edges of its
tiles of 8 x 32 pixels and of its blocks of 16 channels and columns, against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def capi():
    import paralleltnnlayers_amd.capi as c
    c.lib()
    assert torch.cuda.is_available()
    return c


# (N, C, H, W, T, k): a plane inside one tile / rows and columns past whole tiles / one channel,
# one and four blocks of them, whole and ragged / one to five blocks of columns / many tiles a workgroup
CASES = [(3, 1, 3, 4, 1, 1), (2, 3, 9, 36, 17, 3), (1, 4, 8, 32, 64, 1), (2, 5, 17, 28, 48, 3),
         (3, 3, 33, 20, 17, 5), (2, 8, 15, 64, 33, 3), (1, 1, 40, 100, 64, 5), (5, 2, 130, 132, 16, 3),
         (2, 16, 24, 40, 64, 1), (3, 3, 257, 260, 48, 5)]
# one block of columns and many tiles a workgroup: one channel under 3x3, under 1x1, one to four blocks of rows
CASES += [(6, 1, 260, 252, 16, 3), (6, 1, 257, 252, 64, 1), (7, 1, 256, 256, 1, 3), (5, 1, 264, 260, 33, 3),
          (5, 9, 250, 244, 16, 1)]


@pytest.mark.parametrize("how", ["relu", "bias", "plain"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c)))
def test_against_float64(capi, case, how):
    N, C, H, W, T, k = case
    R = 5
    gen = torch.Generator(device="cuda").manual_seed(sum(case))
    mk = lambda *s: torch.randn(*s, device="cuda", generator=gen)
    x, dy, fac = mk(N, C, H, W), mk(N, T, H, W), [mk(d, R) for d in (T, C, k, k)]
    s = capi.shape_for(x.shape, *fac, k // 2)
    act = "relu" if how == "relu" else None
    dym = dy.double().cpu()
    if how == "plain":                                  # the tile kernel itself: variant 3
        got = capi.conv2d_backward_filter(x, dy, *fac, pad=k // 2, variant=3)
    else:
        y = capi.layer_forward(s, None, x, *fac, mk(T), act)
        if act:
            dym = dym * (y > 0).cpu()
        _, got, dbias = capi.layer_backward(s, None, x, y, dy, *fac, act, False, True, True)
        want = dym.sum((0, 2, 3))
        n = N * H * W                                   # fp32 sums: 2^-24 a step, as a random walk
        assert ((dbias.double().cpu() - want).abs()
                <= 4 * 2.0 ** -24 * ((dym ** 2).sum((0, 2, 3)) * n).sqrt() + 1e-30).all()
    f = [t.double().cpu() for t in fac]
    xd = x.double().cpu()
    dK = torch.nn.grad.conv2d_weight(xd, (T, C, k, k), dym, padding=k // 2)
    size = torch.nn.grad.conv2d_weight(xd.abs(), (T, C, k, k), dym.abs(), padding=k // 2)
    eqs = ["tcyx,cr,yr,xr->tr", "tcyx,tr,yr,xr->cr", "tcyx,tr,cr,xr->yr", "tcyx,tr,cr,yr->xr"]
    for i, (g, eq) in enumerate(zip(got, eqs)):
        others = [f[j] for j in range(4) if j != i]
        want = torch.einsum(eq, dK, *others)
        # exact products; the sums' roundings, 2^-24 of the running sum each, stay within four of the terms'
        # sizes added up (a random walk over hundreds of chains is far below)
        bound = torch.einsum(eq, size, *[o.abs() for o in others])
        assert ((g.double().cpu() - want).abs() <= 4 * 2.0 ** -24 * bound).all()


def test_repeats_bit_for_bit(capi):
    N, C, H, W, T, k, R = 4, 3, 61, 96, 40, 3, 9
    mk = lambda *s: torch.randn(*s, device="cuda")
    x, dy, fac = mk(N, C, H, W), mk(N, T, H, W), [mk(d, R) for d in (T, C, k, k)]
    runs = [capi.conv2d_backward_filter(x, dy, *fac, pad=1, variant=3) for _ in range(3)]
    assert all(torch.equal(a, b) for r in runs[1:] for a, b in zip(r, runs[0]))


@pytest.mark.parametrize("case", [(6, 1, 260, 252, 16, 3), (6, 1, 250, 252, 64, 1), (6, 1, 256, 256, 33, 3)],
                         ids=lambda c: "x".join(map(str, c)))
def test_one_block_of_columns_repeats_bit_for_bit(capi, case):
    N, C, H, W, T, k = case
    mk = lambda *s: torch.randn(*s, device="cuda")
    x, dy, fac = mk(N, C, H, W), mk(N, T, H, W), [mk(d, 7) for d in (T, C, k, k)]
    runs = [capi.conv2d_backward_filter(x, dy, *fac, pad=k // 2, variant=3) for _ in range(5)]
    assert all(torch.equal(a, b) for r in runs[1:] for a, b in zip(r, runs[0]))
