"""The input gradient beside the factor gradients of the three-launch variant, whose G1 is formed for it
alone: strips and octets that end inside a row or an image, channel groups, one rank tile and two."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def capi():
    import paralleltnnlayers_amd.capi as c
    c.lib()
    assert torch.cuda.is_available()
    return c


# (N, C, H, W, T, k, R)
CASES = [(1, 80, 4, 8, 96, 1, 1), (3, 80, 14, 14, 32, 1, 32), (2, 32, 12, 9, 48, 3, 33), (16, 64, 32, 32, 64, 3, 16),
         (3, 272, 20, 20, 16, 3, 64), (2, 48, 10, 30, 144, 5, 17), (5, 16, 22, 26, 32, 3, 5)]


@pytest.mark.parametrize("relu", [True, False], ids=["relu", "linear"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c)))
def test_against_float64(capi, case, relu):
    N, C, H, W, T, k, R = case
    gen = torch.Generator(device="cuda").manual_seed(sum(case))
    mk = lambda *s: torch.randn(*s, device="cuda", generator=gen)
    x, fac = mk(N, C, H, W), [mk(d, R) for d in (T, C, k, k)]
    s = capi.shape_for(x.shape, *fac, k // 2)
    assert capi.plan_query(s, "backward_filter")["variant"] == "mfma_fused_taps"
    act = "relu" if relu else None
    y, dy = capi.layer_forward(s, None, x, *fac, mk(T), act), mk(N, T, H, W)
    dx, grads, dbias = capi.layer_backward(s, None, x, y, dy, *fac, act)
    assert capi.lib().cp4_layer_last_backward_dx_beside() == 1
    # nothing else depends on whether dx comes along
    _, alone, bias_alone = capi.layer_backward(s, None, x, y, dy, *fac, act, False, True, True)
    assert all(torch.equal(a, b) for a, b in zip(grads, alone)) and torch.equal(dbias, bias_alone)
    d = (torch.where(y > 0, dy, torch.zeros_like(dy)) if relu else dy).double().cpu()
    f = [t.double().cpu() for t in fac]
    adjoint = lambda d, f: torch.nn.functional.conv_transpose2d(
        d, torch.einsum("tr,cr,yr,xr->tcyx", *f), padding=k // 2)
    want, terms = adjoint(d, f), adjoint(d.abs(), [t.abs() for t in f])
    # three fp32 contractions: 2^-24 a step of the terms' magnitudes, as a random walk (a factor of four to spare)
    assert ((dx.double().cpu() - want).abs() <= 4 * (T + 2 * k + R) ** 0.5 * 2.0 ** -24 * terms + 1e-30).all()


@pytest.mark.parametrize("case", CASES[1:4], ids=lambda c: "x".join(map(str, c)))
def test_without_room_for_g1(capi, case):
    """A workspace that ends where G1 would begin: dx by the pass of its own, all else bit for bit."""
    N, C, H, W, T, k, R = case
    gen = torch.Generator(device="cuda").manual_seed(sum(case))
    mk = lambda *s: torch.randn(*s, device="cuda", generator=gen)
    x, fac, dy = mk(N, C, H, W), [mk(d, R) for d in (T, C, k, k)], mk(N, T, H, W)
    s = capi.shape_for(x.shape, *fac, k // 2)
    L, F32, NONE = capi.lib(), 0, 0
    need = L.cp4_layer_backward_workspace_bytes(ctypes.byref(s), None, F32, NONE, 3)
    g1 = (N * R * H * W * 4 + 255) // 256 * 256

    def backward(bytes_):
        ws = torch.empty(need, dtype=torch.uint8, device="cuda")
        ws[bytes_:] = 0x5a
        out = [torch.empty_like(t) for t in [x] + fac]
        p = lambda t: ctypes.c_void_p(t.data_ptr())
        rc = L.cp4_layer_backward(ctypes.byref(s), None, F32, p(x), None, p(dy), *map(p, fac), NONE, *map(p, out),
                                  None, p(ws), bytes_, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        torch.cuda.synchronize()
        assert (ws[bytes_:] == 0x5a).all()
        return rc, out, L.cp4_layer_last_backward_dx_beside()

    rc, want, beside = backward(need)
    assert (rc, beside) == (capi.OK, 1)
    rc, got, beside = backward(need - g1)
    assert (rc, beside) == (capi.OK, 0)
    assert all(torch.equal(a, b) for a, b in zip(got[1:], want[1:]))
    assert torch.equal(got[0], capi.conv2d_backward_data(dy, *fac, pad=k // 2))
    assert backward(need - g1 - 256)[0] == capi.ERR_WORKSPACE
