"""Calls on a stream of their own: results are right, and outputs and scratch come from that
stream's memory, where nothing queued on another stream can still be using them."""
import pytest
import torch

pytestmark = pytest.mark.gpu

N, C, H, W, T, k, R = 8, 32, 28, 28, 48, 3, 16


@pytest.fixture(scope="module")
def data():
    gen = torch.Generator(device="cuda").manual_seed(2)
    mk = lambda *s: torch.randn(*s, device="cuda", generator=gen)
    return dict(x=mk(N, C, H, W), dy=mk(N, T, H, W), f=[mk(d, R) for d in (T, C, k, k)], b=mk(T),
                K3=[mk(C, R), mk(k, k, R), mk(R, T)], KR=[mk(4, 6, R), mk(8, 8, R), mk(k, k, R)])


def _calls(capi, d):
    x, dy, f, b = d["x"], d["dy"], d["f"], d["b"]
    s = capi.shape_for(x.shape, *f, 1)
    g = capi.geometry(s, 2, "same")
    h, dh = x.bfloat16(), dy.bfloat16()
    dy2 = dy[:, :, ::2, ::2].contiguous()
    y = capi.layer_forward(s, None, x, *f, b, "relu")
    return {
        "forward": lambda st: capi.conv2d_forward(x, *f, stream=st),
        "backward_data": lambda st: capi.conv2d_backward_data(dy, *f, stream=st),
        "backward_filter": lambda st: capi.conv2d_backward_filter(x, dy, *f, stream=st),
        "bias_act": lambda st: capi.conv2d_forward_bias_act(x, *f, b, "relu", stream=st),
        "forward_ex": lambda st: capi.conv2d_forward_ex(x, *f, g, stream=st),
        "data_ex": lambda st: capi.conv2d_backward_data_ex(dy2, (H, W), *f, g, stream=st),
        "filter_ex": lambda st: capi.conv2d_backward_filter_ex(x, dy2, *f, g, stream=st),
        "forward_bf16": lambda st: capi.conv2d_forward_bf16(h, *f, stream=st),
        "data_bf16": lambda st: capi.conv2d_backward_data_bf16(dh, *f, stream=st),
        "filter_bf16": lambda st: capi.conv2d_backward_filter_bf16(h, dh, *f, stream=st),
        "forward_f16": lambda st: capi.conv2d_forward_f16(x.half(), *f, stream=st),
        "data_f16": lambda st: capi.conv2d_backward_data_f16(dy.half(), *f, stream=st),
        "filter_f16": lambda st: capi.conv2d_backward_filter_f16(x.half(), dy.half(), *f, stream=st),
        "layer_forward": lambda st: capi.layer_forward(s, None, x, *f, b, "relu", stream=st),
        "layer_backward": lambda st: capi.layer_backward(s, None, x, y, dy, *f, "relu", stream=st),
        "filter_full": lambda st: capi.conv2d_backward_filter_full(x, dy, k, k, stream=st),
        "recompose": lambda st: capi.recompose(*f, stream=st),
        "cp3_forward": lambda st: capi.cp3_conv2d_forward(x, *d["K3"], stream=st),
        "cp3_data": lambda st: capi.cp3_conv2d_backward_data(dy, *d["K3"], stream=st),
        "cp3_filter": lambda st: capi.cp3_conv2d_backward_filter(x, dy, *d["K3"], stream=st),
        "rcp_forward": lambda st: capi.rcp_conv2d_forward(x, *d["KR"], stream=st),
        "rcp_data": lambda st: capi.rcp_conv2d_backward_data(dy, *d["KR"], stream=st),
        "rcp_filter": lambda st: capi.rcp_conv2d_backward_filter(x, dy, *d["KR"], stream=st),
    }


NAMES = ("forward backward_data backward_filter bias_act forward_ex data_ex filter_ex forward_bf16 "
         "data_bf16 filter_bf16 forward_f16 data_f16 filter_f16 layer_forward layer_backward "
         "filter_full recompose cp3_forward cp3_data cp3_filter rcp_forward rcp_data "
         "rcp_filter").split()


def _flat(result):
    if isinstance(result, torch.Tensor):
        return [result]
    return [t for r in result for t in _flat(r)]


def _stream_of_memory(t):
    for seg in torch.cuda.memory_snapshot():
        if seg["address"] <= t.data_ptr() < seg["address"] + seg["total_size"]:
            return seg["stream"]


@pytest.mark.parametrize("external", [False, True], ids=["torch", "handle"])
@pytest.mark.parametrize("name", NAMES)
def test_memory_belongs_to_the_stream(data, name, external):
    import paralleltnnlayers_amd.capi as capi
    run = _calls(capi, data)[name]
    want = _flat(run(None))
    torch.cuda.synchronize()
    side = torch.cuda.Stream()

    class Handle:                              # whatever else carries the stream's handle
        cuda_stream = side.cuda_stream

    scratch, empty = [], torch.empty
    try:                                       # what Python allocates for the call, scratch included
        torch.empty = lambda *a, **kw: (scratch.append(torch.cuda.current_stream().cuda_stream),
                                        empty(*a, **kw))[1]
        got = _flat(run(Handle() if external else side))
    finally:
        torch.empty = empty
    side.synchronize()
    assert len(got) == len(want) and all(torch.equal(a, b) for a, b in zip(got, want))
    assert {_stream_of_memory(t) for t in got} == {side.cuda_stream}
    assert set(scratch) <= {side.cuda_stream}


def test_native_scratch_belongs_to_the_stream(data):
    """backward_filter's own workspace (megabytes; its results are kilobytes)."""
    import paralleltnnlayers_amd.capi as capi
    x, dy, f = data["x"], data["dy"], data["f"]
    assert capi.backward_filter_workspace_bytes(capi.shape_for(x.shape, *f, 1)) > 2 << 20
    side = torch.cuda.Stream()
    grads = capi.conv2d_backward_filter(x, dy, *f, stream=side)
    side.synchronize()
    sizes = [seg["total_size"] for seg in torch.cuda.memory_snapshot()
             if seg["stream"] == side.cuda_stream and seg["segment_type"] == "large"]
    assert sizes and all(g.numel() < 1 << 18 for g in grads)


def test_callers_memory_stays_where_it_is(data):
    """With `out` given nothing is allocated; the current stream is no other stream."""
    import paralleltnnlayers_amd.capi as capi
    x, f = data["x"], data["f"]
    want = capi.conv2d_forward(x, *f)
    out = torch.empty_like(want)
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    assert capi.conv2d_forward(x, *f, out=out, stream=side) is out
    side.synchronize()
    assert torch.equal(out, want)
    here = torch.cuda.current_stream()
    assert _stream_of_memory(capi.conv2d_forward(x, *f, stream=here)) == here.cuda_stream
