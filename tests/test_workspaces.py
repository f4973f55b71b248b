"""Which workspace a call gets: the host side on the CPU (streams, capture and buffers stubbed), and
launches that overlap on several streams and in graphs on the GPU."""
import ctypes

import pytest
import torch

from vllm_webgpu_amd import _lib, ops


class Host:
    """A device whose current stream and capture state the test sets; buffers are CPU tensors."""

    def __init__(self, monkeypatch):
        self.stream, self.capture, self.made, self.launched = 0, False, [], []
        monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda idx: self.stream, raising=False)
        monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
        monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: self.capture)
        monkeypatch.setattr(ops, "_new_workspace", self._new)
        monkeypatch.setattr(ops, "_ws_cache", {})
        monkeypatch.setattr(ops, "_ws_side", {})

    def _new(self, nbytes, *rest):
        t = torch.empty(nbytes, dtype=torch.uint8)
        self.made.append(t)
        return t

    def get(self, stream, nbytes=1 << 20, capture=False):
        self.stream, self.capture = stream, capture
        return ops.workspace(nbytes, torch.device("cuda", 0))


@pytest.fixture
def host(monkeypatch):
    return Host(monkeypatch)


def test_a_capture_shares_no_buffer(host):
    """A graph's replays may overlap any stream's eager calls: its buffer is no stream's, nor the
    default's, nor another capture's, and the cache never holds it."""
    eager = [host.get(0), host.get(11), host.get(22)]
    seen = {t.data_ptr() for t in eager}
    for stream in (11, 33, 33):
        t = host.get(stream, capture=True)
        assert t.data_ptr() not in seen
        seen.add(t.data_ptr())
    for s, t in zip((0, 11, 22), eager):
        assert host.get(s) is t
    assert host.get(33).data_ptr() not in seen


def test_a_buffer_for_each_stream(host):
    """More streams than the cache keeps: a call never gets a buffer that another stream's may be
    using, and the buffers that are dropped are released."""
    n = 3 * ops._WS_SIDE_MAX
    kept = [host.get(s) for s in range(n)]
    assert len({t.data_ptr() for t in kept}) == n
    assert host.get(n - 1) is kept[-1]
    assert len(ops._ws_side) <= ops._WS_SIDE_MAX
    small = host.get(n - 1)
    big = host.get(n - 1, 4 << 20)
    assert big.numel() >= 4 << 20 and host.get(n - 1) is big and big is not small
    assert len(ops._ws_side) <= ops._WS_SIDE_MAX


def test_a_prepared_call_uses_the_stream_it_is_launched_on(host, monkeypatch):
    """Two prepared calls, or one, launched on streams without an order between them."""
    seen = []

    class L:
        def vws_sample(self, ref):
            a = ctypes.cast(ref, ctypes.POINTER(_lib.SampleArgs)).contents
            seen.append((a.workspace, a.workspace_bytes, a.stream, a.batch))
            return 0

        def vws_sample_workspace_size(self, *shape):
            return 4096

    monkeypatch.setattr(_lib, "lib", lambda: L())
    ws = host.get(11)
    args = _lib.SampleArgs()
    args.batch, args.workspace, args.workspace_bytes, args.stream = 5, ws.data_ptr(), ws.numel(), 11
    call = ops.PreparedSample(args, None, (ws,), 11, 4096, 0)
    for stream, capture in ((11, False), (22, False), (22, False), (11, True), (33, True), (11, False)):
        host.stream, host.capture = stream, capture
        call.launch()
    ptrs = [s[0] for s in seen]
    assert ptrs[0] == ptrs[5] == ws.data_ptr() and ptrs[1] == ptrs[2] == host.get(22).data_ptr()
    assert ws.data_ptr() not in ptrs[1:5] and len({ptrs[1], ptrs[3], ptrs[4]}) == 3
    # (a stream handle of 0 reads back as None)
    assert [s[2] for s in seen] == [11, 22, 22, 11, 33, 11] and all(s[3] == 5 and s[1] >= 4096 for s in seen)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["greedy", "plain", "history", "topk", "penalties"])
def test_graph_replays_beside_eager_streams(cuda, kind):
    """Warmed up on one stream, captured on a second, replayed on a third while the first goes on
    with the same operation (its buffer grown in between): every replay and every eager call
    returns what the call alone returns."""
    B, V = 24, 40003
    g = torch.Generator(device=cuda).manual_seed(3)
    xs = [torch.randn((B, V), generator=g, device=cuda) * 3 for _ in range(2)]
    T = torch.full((B,), 0.9, device=cuda)
    R, P = torch.full((B,), 1.2, device=cuda), torch.full((B,), 0.95, device=cuda)
    hist = torch.randint(0, V, (B, 200), generator=g, device=cuda, dtype=torch.int32)

    def call(x):
        if kind == "topk":
            return torch.cat([t.float() for t in ops.topk(x, 30)], dim=1)
        if kind == "penalties":
            return ops.apply_penalties(x.clone(), repetition_penalty=R, output_ids=hist)
        kw = {} if kind == "greedy" else {"temperature": T, "rng_key": 7}
        if kind == "history":
            kw.update(output_ids=hist, repetition_penalty=R, top_p=P)
        r = ops.sample(x, **kw)
        return torch.stack([r.sampled, r.num_kept])

    want = [call(x) for x in xs]
    warm, cap, other = (torch.cuda.Stream() for _ in range(3))
    torch.cuda.synchronize()
    with torch.cuda.stream(warm):
        call(xs[0])
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=cap):
        out = call(xs[0])
    for i in range(8):
        got = []
        with torch.cuda.stream(warm):
            if i == 3:  # (outgrows the stream's buffer)
                ops.workspace(8 << 20, cuda)
            got += [call(xs[1]) for _ in range(3)]
        with torch.cuda.stream(other):
            graph.replay()
            got += [call(xs[1])]
        with torch.cuda.stream(warm):
            got += [call(xs[1]) for _ in range(3)]
        torch.cuda.synchronize()
        assert torch.equal(out, want[0]), f"replay {i}"
        assert all(torch.equal(t, want[1]) for t in got), f"eager calls beside replay {i}"
        out.zero_()


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["greedy", "plain"])
def test_prepared_calls_on_several_streams(cuda, kind):
    """Prepared calls launched on streams without an order between them, and into a graph that is
    replayed beside them."""
    B, V, n = 24, 40003, 3
    g = torch.Generator(device=cuda).manual_seed(4)
    kw = {} if kind == "greedy" else {"temperature": torch.full((B,), 0.9, device=cuda), "rng_key": 7}
    calls = [ops.prepare_sample(torch.randn((B, V), generator=g, device=cuda) * 3, **kw) for _ in range(n)]
    want = [c.launch().sampled.clone() for c in calls]
    streams = [torch.cuda.Stream() for _ in range(n + 1)]
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=streams[n]):
        calls[0].launch()
    for i in range(8):
        for c in calls:
            c.result.sampled.fill_(-1)
        torch.cuda.synchronize()
        for _ in range(4):
            for s, c in zip(streams, calls[1:] if i % 2 else calls):
                with torch.cuda.stream(s):
                    c.launch()
        if i % 2:
            with torch.cuda.stream(streams[n - 1]):
                graph.replay()
        torch.cuda.synchronize()
        for w, c in zip(want, calls):
            assert torch.equal(c.result.sampled, w), i
