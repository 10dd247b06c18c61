"""Calls of several host threads, and on several streams, that share or own the per-stream
workspaces (tile images, key unions and their partials): every result equals the same call made
alone, bit for bit, also where a workspace grows or is given back in between."""
import threading

import numpy as np
import pytest

from conftest import rng
from test_gpu_kv import _gpu
from test_gpu_rows import takes_rows

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def _dense(seed, L, T):
    """A row-kernel call over its own keys."""
    import qw_amd

    r = rng(seed)
    q, k, v = (_gpu(r.standard_normal(s).astype(np.float16)) for s in ((24, L, 256), (4, T, 256), (4, T, 256)))
    assert takes_rows(24, 4, 256, L, T)
    return lambda: qw_amd.causal_attention(q, k, v, 1 / 16)


def _masked(seed, L, T):
    import qw_amd

    r = rng(seed)
    q, k, v = (_gpu(r.standard_normal(s).astype(np.float16)) for s in ((24, L, 256), (4, T, 256), (4, T, 256)))
    m = torch.from_numpy(r.random((L, T)) < 0.8).cuda()
    assert takes_rows(24, 4, 256, L, T, False, 0, 0.0, 3)
    return lambda: qw_amd.attention(q, k, v, 1 / 16, m)


def _sparse(seed, L, T, W, dt):
    """Row groups over the union of their keys."""
    import qw_amd

    r = rng(seed)
    q, k, v = (_gpu(r.standard_normal(s).astype(np.float16)).to(dt) for s in ((24, L, 256), (4, T, 256), (4, T, 256)))
    lists = _gpu(np.sort(np.stack([r.permutation(T)[:W]] * L), axis=1).astype(np.int32))
    lengths = _gpu(np.full(L, W, np.int32))
    c = {torch.float16: 0, torch.bfloat16: 1, torch.float32: 2}[dt]
    assert qw_amd.lib().qw_dlsa_union_keys(c, c, L, W, 24, 4, 256, T) > 0
    f = qw_amd.sparse_attention if dt == torch.float16 else qw_amd.sparse_attention_typed
    return lambda: f(q, k, v, lists, lengths, 1 / 16)


def _calls():
    return [_dense(1, 128, 2500), _dense(2, 300, 4000), _masked(3, 25, 6000),
            _sparse(4, 128, 3000, 1700, torch.float16), _sparse(5, 300, 4000, 1800, torch.float16),
            _sparse(6, 128, 2000, 700, torch.bfloat16), _sparse(7, 70, 1500, 300, torch.float32)]


def _in_threads(work):
    """work: one list of calls and one stream a thread. Their outputs, in order."""
    outs, errors = [[] for _ in work], []
    start = threading.Barrier(len(work))

    def body(i, calls, stream):
        try:
            start.wait(30)
            with torch.cuda.stream(stream):
                outs[i].extend(c() for c in calls)
        except Exception as e:  # noqa: BLE001
            errors.append(e)

    threads = [threading.Thread(target=body, args=(i, c, s)) for i, (c, s) in enumerate(work)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    torch.cuda.synchronize()
    assert not errors, errors
    return outs


def test_threads_on_one_stream():
    calls = _calls()
    alone = [c() for c in calls]
    stream = torch.cuda.Stream()  # its workspaces are made, and grow, while the threads run
    torch.cuda.synchronize()
    order = [rng(i).permutation(12 * list(range(len(calls)))) for i in range(3)]
    outs = _in_threads([([calls[i] for i in o], stream) for o in order])
    for o, got in zip(order, outs):
        assert all(torch.equal(g, alone[i]) for i, g in zip(o, got))


def test_threads_on_streams_of_their_own():
    calls = _calls()
    alone = [c() for c in calls]
    torch.cuda.synchronize()
    order = [rng(i).permutation(8 * list(range(len(calls)))) for i in range(3)]
    outs = _in_threads([([calls[i] for i in o], torch.cuda.Stream()) for o in order])
    for o, got in zip(order, outs):
        assert all(torch.equal(g, alone[i]) for i, g in zip(o, got))


def test_two_streams_from_one_thread():
    """Calls on a side stream behind unfinished ones on another: each stream its own workspaces."""
    calls = _calls()
    alone = [c() for c in calls]
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    outs = []
    for _ in range(6):
        for i, c in enumerate(calls):
            for s in (a, b):
                with torch.cuda.stream(s):
                    outs.append((i, c()))
    torch.cuda.synchronize()
    assert all(torch.equal(g, alone[i]) for i, g in outs)


def test_workspaces_are_given_back():
    import qw_amd

    calls = [_dense(1, 128, 2500), _sparse(4, 128, 3000, 1700, torch.float16), _dense(8, 64, 60000)]
    alone = [c() for c in calls]
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        for _ in range(2):
            before = torch.cuda.mem_get_info()[0]
            outs = [c() for c in calls]
            stream.synchronize()
            used = before - torch.cuda.mem_get_info()[0]
            qw_amd.release_workspaces()
            assert used >= 60000 * 4 * 1024, used  # the last call's images, at least
            assert torch.cuda.mem_get_info()[0] >= before - (32 << 20)  # (torch's own blocks for the outputs)
            assert all(torch.equal(a, b) for a, b in zip(outs, alone))


def test_release_keeps_what_a_graph_reads():
    import qw_amd

    call = _dense(1, 128, 2500)
    want = call()
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        call()
        stream.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=stream):
            out = call()
        qw_amd.release_workspaces()
        big = _dense(9, 64, 60000)()  # grows the stream's buffer: the graph keeps its own
        qw_amd.release_workspaces()
        for _ in range(3):
            out.zero_()
            g.replay()
            stream.synchronize()
            assert torch.equal(out, want)
            del big
            big = torch.full((64 << 20,), 7, dtype=torch.uint8, device="cuda")  # whatever was freed is written
    torch.cuda.synchronize()
