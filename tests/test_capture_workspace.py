"""Captured launches and the workspace: a graph is replayed on any stream, beside eager launches and other graphs, so it
never uses the workspace of the stream it was captured on."""
import ctypes

import pytest
import torch

import grouped_mm_bf16_amd.kernels as K_
from grouped_mm_bf16_amd import _lib, moe

DEV = "cuda"


class _Recorder:
    """A launcher that notes the workspace it is given; `useful`: one would be of use."""

    def __init__(self, useful):
        self.useful, self.calls = useful, []

    def __call__(self, *args):
        *rest, ws, nbytes, stream = args
        self.calls.append((ws, nbytes))
        return _lib.ERR_WORKSPACE if self.useful and nbytes >= _lib.WORKSPACE_EAGER_ONLY else _lib.OK


def test_a_captured_launch_does_not_get_the_streams_workspace(monkeypatch):
    mine = torch.zeros(8192, dtype=torch.uint8)
    own = torch.zeros(8192, dtype=torch.uint8)
    device = torch.device("cuda", 0)
    monkeypatch.setattr(K_, "_workspaces", {(0, 7): mine})
    for given in (own, None):          # a capture that torch knows of, and another one
        monkeypatch.setattr(K_, "_captured_workspace", lambda d, s: given)
        launcher = _Recorder(useful=True)
        assert K_.call_with_workspace(launcher, (1, 2), device, 7) == _lib.OK
        (_, asked), (ws, nbytes) = launcher.calls
        assert asked == 8192 | _lib.WORKSPACE_EAGER_ONLY
        assert (ws, nbytes) == ((own.data_ptr(), 8192) if given is own else (None, 0))
    eager = _Recorder(useful=False)
    assert K_.call_with_workspace(eager, (), device, 7) == _lib.OK
    assert eager.calls == [(mine.data_ptr(), 8192 | _lib.WORKSPACE_EAGER_ONLY)]


# ------------------------------------------------------------------ on the GPU
def _offs(sizes):
    return torch.tensor(sizes).cumsum(0).to(torch.int32).to(DEV)


def _cases():
    """name -> launch into `out`: parts of a jagged contraction, its tile queue, cut tiles of the last round, gathered rows"""
    gen = torch.Generator(device=DEV).manual_seed(2)
    r = lambda *s: torch.randn(*s, device=DEV, dtype=torch.bfloat16, generator=gen)
    a1, b1, o1 = r(6000, 48).t(), r(6000, 64), _offs([4000, 0, 1500, 500])
    a2, b2, o2 = r(512, 6000), r(6000, 768), _offs([3000] + [10] * 190 + [1100])
    a3, b3, o3 = r(300, 8192), r(3, 8192, 256), _offs([200, 0, 100])
    idx = torch.randint(0, 300, (300,), device=DEV, dtype=torch.int32, generator=gen)
    return {
        "parts": ((4, 48, 64), lambda out: K_.grouped_mm_2d2d(a1, b1, o1, out)),
        "queue": ((192, 512, 768), lambda out: K_.grouped_mm_2d2d(a2, b2, o2, out)),
        "last round": ((300, 256), lambda out: K_.grouped_mm_2d3d(a3, b3, o3, out)),
        "gathered": ((300, 256), lambda out: moe.grouped_mm_gathered(a3, idx, b3, o3, out=out)),
    }


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["parts", "queue", "last round", "gathered"])
def test_replays_leave_the_streams_workspace_alone(name):
    """The capture stream has run the launch eagerly before.  Counters of its workspace that are not zero must not be seen
    by the graph, and replays must not change them; every replay gives the eager result's bits."""
    shape, launch = _cases()[name]
    eager, out = (torch.empty(shape, device=DEV, dtype=torch.bfloat16) for _ in range(2))
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        launch(eager)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            launch(out)
            scratch = torch.full((1 << 24,), 3, device=DEV, dtype=torch.int32)   # may take the workspace's memory
    torch.cuda.synchronize()
    ws = K_._workspaces[(torch.cuda.current_device(), stream.cuda_stream)]
    ws[:4096].fill_(1)
    try:
        for _ in range(3):
            out.fill_(float("nan"))
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out.view(torch.int16), eager.view(torch.int16))
            assert (scratch == 3).all()
        assert (ws[:4096] == 1).all()
    finally:
        ws[:4096].zero_()
        torch.cuda.synchronize()


@pytest.mark.gpu
@pytest.mark.parametrize("sizes,G,M,K,N,dtype", [
    ([10, 54], 2, 64, 64, 64, torch.bfloat16),
    # a last round of 168 tiles of 1024, of 129 of 512, and, whichever way the rows are split, of 160 to 176 of 512: too many to cut
    (None, 27, 130, 801, 2500, torch.float32), (None, 1, 81, 1601, 641 * 128 - 1, torch.bfloat16),
    ([2700, 2600], 2, 5300, 1601, 2047, torch.bfloat16)])
def test_launch_without_a_use_for_a_workspace_is_captured_as_it_is(sizes, G, M, K, N, dtype):
    a = torch.randn((G, M, K) if sizes is None else (M, K), device=DEV).to(dtype)
    b, out = torch.randn(G, K, N, device=DEV).to(dtype), torch.empty((G, M, N) if sizes is None else (M, N), device=DEV, dtype=dtype)
    offs = None if sizes is None else _offs(sizes)
    launch = lambda: K_.grouped_mm_3d3d(a, b, out) if offs is None else K_.grouped_mm_2d3d(a, b, offs, out)
    launch()
    torch.cuda.synchronize()
    before = torch.cuda.memory_reserved()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        launch()
    assert torch.cuda.memory_reserved() - before < 1 << 20


@pytest.mark.gpu
def test_capture_that_torch_does_not_know_of():
    """hipStreamBeginCapture called directly: memory allocated meanwhile would go back to the common pool, so the launch is
    recorded without a workspace."""
    shape, launch = _cases()["parts"]
    eager, out = (torch.empty(shape, device=DEV, dtype=torch.bfloat16) for _ in range(2))
    launch(eager)
    torch.cuda.synchronize()
    hip = ctypes.CDLL("libamdhip64.so")
    stream = torch.cuda.Stream()
    graph, handle = ctypes.c_void_p(), ctypes.c_void_p(stream.cuda_stream)
    with torch.cuda.stream(stream):
        launch(eager)
        torch.cuda.synchronize()
        assert hip.hipStreamBeginCapture(handle, 2) == 0        # relaxed
        try:
            assert _lib.load().gmm_stream_capture(stream.cuda_stream) > 0
            launch(out)
        finally:
            assert hip.hipStreamEndCapture(handle, ctypes.byref(graph)) == 0
    assert K_._capture[1] is False
    assert _lib.load().gmm_stream_capture(stream.cuda_stream) == 0
    exe = ctypes.c_void_p()
    assert hip.hipGraphInstantiate(ctypes.byref(exe), graph, None, None, ctypes.c_size_t(0)) == 0
    for _ in range(2):
        out.fill_(float("nan"))
        torch.cuda.synchronize()
        assert hip.hipGraphLaunch(exe, handle) == 0
        torch.cuda.synchronize()
        # the same products, summed uncut
        torch.testing.assert_close(out.float(), eager.float(), rtol=1.6e-2, atol=1e-2 * 8)
    assert hip.hipGraphExecDestroy(exe) == 0 and hip.hipGraphDestroy(graph) == 0


def _cut_cases():
    """Launches whose tiles are cut along K: aligned and few (the assembly tile's without a workspace), unaligned and few, the
    last round behind whole ones, gathered rows, and a layer whose up projection is one of them."""
    gen = torch.Generator(device=DEV).manual_seed(4)
    r = lambda *s, dtype=torch.bfloat16: torch.randn(*s, device=DEV, generator=gen).to(dtype)
    a1, b1 = r(2, 96, 2048), r(2, 2048, 1024)
    a2, b2, o2 = r(8, 2048), r(8, 2048, 1536), _offs([1] * 8)
    a3, b3 = r(2, 90, 2047), r(2, 2047, 1001)
    a4, b4 = r(26, 130, 801, dtype=torch.float32), r(26, 801, 2500, dtype=torch.float32)
    idx = torch.randint(0, 8, (8,), device=DEV, dtype=torch.int32, generator=gen)
    x, logits, w_up, w_down = r(6, 2048), r(6, 8), r(8, 2048, 1024), r(8, 512, 2048)
    return {
        "aligned": lambda: _into((2, 96, 1024), lambda out: K_.grouped_mm_3d3d(a1, b1, out)),
        "decode": lambda: _into((8, 1536), lambda out: K_.grouped_mm_2d3d(a2, b2, o2, out)),
        "unaligned": lambda: _into((2, 90, 1001), lambda out: K_.grouped_mm_3d3d(a3, b3, out)),
        "last round": lambda: _into((26, 130, 2500), lambda out: K_.grouped_mm_3d3d(a4, b4, out), torch.float32),
        "gathered": lambda: moe.grouped_mm_gathered(a2, idx, b2, o2),
        "layer": lambda: moe.moe_forward(x, logits, w_up, w_down, 2),
    }


def _into(shape, launch, dtype=torch.bfloat16):
    out = torch.empty(shape, device=DEV, dtype=dtype)
    launch(out)
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["aligned", "decode", "unaligned", "last round", "gathered", "layer"])
def test_cut_tiles_on_a_capture_stream_without_a_workspace(name):
    """torch.cuda.graph captures on a stream that no eager launch has used: the launch is recorded with the same kernel and
    the same cuts, so that every replay gives the eager result's bits."""
    call = _cut_cases()[name]
    bits = lambda t: t.view(torch.int32 if t.dtype == torch.float32 else torch.int16)
    eager = call()
    kernel = K_.last_kernel()
    assert kernel == "any" or name == "layer"
    with K_.tail_split(False):
        assert name == "layer" or not torch.equal(bits(call()), bits(eager)), "nothing was cut"
    torch.cuda.synchronize()
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    K_._workspaces.pop((torch.cuda.current_device(), stream.cuda_stream), None)      # torch hands out streams again
    with torch.cuda.graph(graph, stream=stream):
        out = call()
        assert K_.last_kernel() == kernel
    assert (torch.cuda.current_device(), stream.cuda_stream) not in K_._workspaces
    for _ in range(3):
        out.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(bits(out), bits(eager))
        assert torch.equal(bits(call()), bits(eager))
