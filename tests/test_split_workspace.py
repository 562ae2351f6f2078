"""The partials of a prefill whose keys are split over work-groups belong to one call.

Such a call is two launches (the pieces, then their merge), and ctypes lets other threads run between
them: two calls that overlap on one stream, or two graphs captured on one stream and replayed on two,
must not have the same partials."""
import contextlib
import threading

import pytest
import torch

from conftest import announce
from kernels import _lib, fa2


class OnGpu(torch.Tensor):
    """A CPU tensor that says it is on a GPU, for a library whose launches are stubs."""
    is_cuda = property(lambda self: True)


def on_gpu(*shape, dtype=torch.bfloat16):
    return torch.zeros(*shape, dtype=dtype).as_subclass(OnGpu)


def padded(T, group):
    q, k = on_gpu(1, 2 * group, T, 128), on_gpu(1, 2, 4096, 128)
    return lambda: fa2.FlashAttention2Function.apply(q, k, k, T > 1, None)


def paged(T, group, max_kv_len=4096):
    q, pool = on_gpu(1, 2 * group, T, 128), on_gpu(4096, 2, 128)
    table = torch.arange(256, dtype=torch.int32)[None]
    lens = torch.tensor([4096], dtype=torch.int32)
    return lambda: fa2.fa2_paged(q, pool, pool, table, lens, max_kv_len=max_kv_len)


@pytest.mark.parametrize("T,group", [(150, 6), (2, 1), (1, 17)])
@pytest.mark.parametrize("call,entry", [(padded, "mi_fa2_fwd"), (paged, "mi_fa2_fwd_paged")])
def test_calls_that_overlap_have_their_own_partials(call, entry, T, group, monkeypatch):
    lib, seen = _lib.load(), []
    both_inside = threading.Barrier(2, timeout=30)

    class Lib:
        def __getattr__(self, name):
            return stub if name == entry else getattr(lib, name)

    def stub(*args):
        seen.append(args[-3:-1])   # workspace, its size
        both_inside.wait()         # both calls hold theirs
        return 0

    monkeypatch.setattr(_lib, "load", lambda: Lib())
    monkeypatch.setattr(_lib, "on_device", lambda dev: contextlib.nullcontext(0))
    monkeypatch.setattr(_lib, "device_index", lambda dev: 0)
    monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda i: 0, raising=False)
    fn = call(T, group)
    threads = [threading.Thread(target=fn) for _ in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    (a, n), (b, m) = seen
    assert n == m > 0 and a and b
    assert a + n <= b or b + m <= a


def test_paged_prefills_are_split_by_a_bound_that_was_given(monkeypatch):
    """Without one the table's capacity bounds the lengths, which may be far shorter."""
    lib, seen = _lib.load(), []

    class Lib:
        def __getattr__(self, name):
            return (lambda *a: seen.append(a[-3]) or 0) if name == "mi_fa2_fwd_paged" else getattr(lib, name)

    monkeypatch.setattr(_lib, "load", lambda: Lib())
    monkeypatch.setattr(_lib, "on_device", lambda dev: contextlib.nullcontext(0))
    monkeypatch.setattr(_lib, "device_index", lambda dev: 0)
    monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda i: 0, raising=False)
    for bound in (4096, None, 4096):   # each time by its own plan
        paged(150, 6, bound)()
    assert [ws is not None for ws in seen] == [True, False, True]
    seen.clear()
    paged(1, 6, None)()   # the decode needs its workspace
    assert seen[0] is not None


def test_a_call_without_memory_for_partials_runs_unsplit(monkeypatch):
    def full(*args, **kw):
        raise torch.OutOfMemoryError("full")
    monkeypatch.setattr(torch, "empty", full)
    assert fa2._own_workspace(1 << 20, torch.device("cpu")) is None


def inputs(T, seed):
    g = torch.Generator().manual_seed(seed)
    q = torch.randn(1, 12, T, 128, generator=g).bfloat16().cuda()
    k, v = (torch.randn(1, 2, 3000, 128, generator=g).bfloat16().cuda() for _ in range(2))
    return q, k, v


@pytest.mark.gpu
def test_threads_on_one_stream():
    cases = [inputs(150, 1), inputs(151, 2)]
    want = [fa2.FlashAttention2Function.apply(*c, True, None) for c in cases]
    torch.cuda.synchronize()
    announce("[gpu] split prefill: two threads on one stream")
    bad = []

    def work(c, w):
        for _ in range(100):
            if not torch.equal(fa2.FlashAttention2Function.apply(*c, True, None), w):
                bad.append(c[0].shape)

    threads = [threading.Thread(target=work, args=cw) for cw in zip(cases, want)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


@pytest.mark.gpu
def test_graphs_captured_on_one_stream_replay_on_two():
    cases = [inputs(150, 3), inputs(150, 4)]
    want = [fa2.FlashAttention2Function.apply(*c, True, None) for c in cases]
    torch.cuda.synchronize()
    graphs, outs = [], []
    for c in cases:
        graphs.append(torch.cuda.CUDAGraph())
        with torch.cuda.graph(graphs[-1]):   # torch captures every graph on one stream of its own
            for _ in range(20):
                out = fa2.FlashAttention2Function.apply(*c, True, None)
        outs.append(out)
    announce("[gpu] split prefill: two graphs replayed on two streams")
    streams = [torch.cuda.Stream() for _ in cases]
    for _ in range(5):
        for graph, stream in zip(graphs, streams):
            with torch.cuda.stream(stream):
                graph.replay()
        torch.cuda.synchronize()
        for out, w in zip(outs, want):
            assert torch.equal(out, w)
            out.zero_()
