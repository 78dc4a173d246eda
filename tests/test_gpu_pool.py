"""The library's device memory pool: objects of one weight version after another reuse memory, an old plan's memory is not
handed on while another stream still runs a forward of it, and threads that build and destroy objects at once each get
the right answers."""

from __future__ import annotations

import ctypes
import gc
import threading

import numpy as np
import pytest
import torch

from helpers import brain_arrays, random_params
from test_gpu_sweep import _cone, _medium, _rnn

from chessfly import _hip
from oracle import forward as F

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def _case(seed, batch):
    conn = _medium(seed)
    lg, b, al = random_params(conn, seed, gain_sd=0.1)
    in_idx, out_idx = conn.nodes("afferent"), conn.nodes("efferent")
    u = torch.randn(len(in_idx), batch, generator=torch.Generator().manual_seed(seed))
    ref = F.cone_f32(brain_arrays(conn, 4.0, lg, b, al, dtype=torch.float64), _cone(conn, in_idx, out_idx, 4), u.double(), 4)
    return conn, (lg, b, al), in_idx.to(DEV), out_idx.to(DEV), u.to(DEV), ref.numpy()


def test_new_weight_versions_on_two_streams():
    """Forwards of six weight versions alternate between two streams with no wait in between, each behind some 20 ms of
    other work: a new version's plan destroys the old one while its forward is still pending on the other stream, and
    takes arrays of the same sizes.  Every version has weights of its own and is checked against its own float64
    reference, so arrays handed on too early give a wrong answer."""
    conn, (lg, b, al), ind, outd, u, _ = _case(3, 256)
    versions = [(lg + np.float32(0.1 * i), b + np.float32(0.05 * i), al) for i in range(6)]
    cone = _cone(conn, conn.nodes("afferent"), conn.nodes("efferent"), 4)
    refs = [F.cone_f32(brain_arrays(conn, 4.0, *v, dtype=torch.float64), cone, u.cpu().double(), 4).numpy() for v in versions]
    for x, y in zip(refs, refs[1:]):
        assert np.abs(x - y).max() > 1e-2 * np.abs(x).max()
    rnn = _rnn(conn, 4.0, lg, b, al)
    params = [[torch.as_tensor(p).to(DEV) for p in v] for v in versions]
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    m = torch.randn(8192, 8192, device=DEV)
    outs, done, pending = [], [], 0
    with torch.no_grad():
        rnn.forward_io(u, ind, outd, 4)                  # the cone
        torch.cuda.synchronize()
        for i, v in enumerate(params):
            with torch.cuda.stream(streams[i % 2]):
                for p, new in zip((rnn.log_gain, rnn.bias, rnn.alpha_logit), v):
                    p.copy_(new)                         # no forward reads them: a plan holds what it needs
                pending += int(bool(done) and not done[-1].query())
                plan = rnn._cone_plan(rnn.light_cone(ind, outd, 4), 1)
                for _ in range(2):
                    m @ m
                outs.append(rnn.forward_io(u, ind, outd, 4))
                assert rnn._cone_plan(rnn.light_cone(ind, outd, 4), 1) is plan
                done.append(torch.cuda.Event())
                done[-1].record()
    torch.cuda.synchronize()
    assert pending == len(params) - 1                    # every plan was destroyed ahead of its forward's end
    for out, ref in zip(outs, refs):
        np.testing.assert_allclose(out.cpu().numpy(), ref, rtol=2e-5, atol=2e-5 * max(np.abs(ref).max(), 1.0))


def test_threads_build_and_destroy_at_once():
    cases = [_case(seed, 64) for seed in (4, 5, 6)]
    failed = []

    def work(case):
        try:
            conn, (lg, b, al), ind, outd, u, ref = case
            with torch.cuda.stream(torch.cuda.Stream()), torch.no_grad():
                for _ in range(4):
                    rnn = _rnn(conn, 4.0, lg, b, al)     # a new cone and plan each time, the old ones destroyed
                    out = rnn.forward_io(u, ind, outd, 4).cpu().numpy()
                    np.testing.assert_allclose(out, ref, rtol=2e-5, atol=2e-5 * max(np.abs(ref).max(), 1.0))
        except BaseException as e:      # noqa: BLE001  (reported by the main thread)
            failed.append(e)

    torch.cuda.synchronize()
    threads = [threading.Thread(target=work, args=(c,)) for c in cases]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed, failed


def _captured(inside, mode="global"):
    """Captures two operations with inside() between them, and replays them."""
    x = torch.ones(1000, device=DEV)
    gc.collect()                                         # what earlier tests left goes away now
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, capture_error_mode=mode):
        y = x * 2
        inside()
        z = y + 1
    for i in range(3):
        x.fill_(float(i))
        graph.replay()
        torch.cuda.synchronize()
        assert float(z[0]) == 2.0 * i + 1 and bool((z == z[0]).all())


def test_objects_released_while_a_graph_is_captured():
    """A network that goes away while a graph is being captured leaves the capture as it is, and the next network gets the
    right answers."""
    conn, (lg, b, al), ind, outd, u, ref = _case(7, 64)
    nets = [_rnn(conn, 4.0, lg, b, al), _rnn(conn, 4.0, lg, b, al)]
    with torch.no_grad():
        for i in range(2):
            nets[i].forward_io(u, ind, outd, 4)

        def drop():
            nets.pop()
            gc.collect()

        _captured(drop)
        for rnn in (nets[0], _rnn(conn, 4.0, lg, b, al)):
            out = rnn.forward_io(u, ind, outd, 4).cpu().numpy()
            np.testing.assert_allclose(out, ref, rtol=2e-5, atol=2e-5 * max(np.abs(ref).max(), 1.0))


def test_more_than_stays_idle_is_released_while_a_graph_is_captured():
    """Plans of 800 MB destroyed during a capture, beside one that lives on: what is past the bound goes back to the runtime
    at once, the rest stays idle until it is asked for."""
    lib = _hip.load()
    n, per = 2_000_000, 8
    crow = torch.arange(0, n + 1, dtype=torch.int32, device=DEV) * per
    pre = (torch.arange(n * per, dtype=torch.int32, device=DEV) * 7) % n
    w, al = torch.ones(n * per, device=DEV), torch.zeros(n, device=DEV)
    plans = []
    for _ in range(5):                                   # 200 MB each
        h = ctypes.c_void_p()
        _hip.check(lib.fly_plan_create_full(n, n * per, crow.data_ptr(), pre.data_ptr(), w.data_ptr(), al.data_ptr(), 10.0,
                                            None, _hip.stream(w.device), ctypes.byref(h)), "fly_plan_create_full")
        plans.append(h)
    del crow, pre, w, al
    _captured(lambda: [_hip.check(lib.fly_plan_destroy(h), "fly_plan_destroy") for h in plans[1:]])
    torch.cuda.empty_cache()
    held = torch.cuda.mem_get_info()[0]
    _hip.trim_memory()
    back = torch.cuda.mem_get_info()[0] - held
    _hip.check(lib.fly_plan_destroy(plans[0]), "fly_plan_destroy")
    # two of the plans' 128 MB arrays at least stayed idle; the bound on what does is checked against stand-ins
    # (test_memory_pool.py), since the runtime rounds what it reports and frees pages of its own with it
    assert back > 200 << 20, back


@pytest.mark.parametrize("mode", ["thread_local", "relaxed"])
def test_another_thread_builds_while_a_graph_is_captured(mode):
    """A network built on another thread, out of memory that must be waited for, while this one captures."""
    conn, (lg, b, al), ind, outd, u, ref = _case(8, 64)
    with torch.no_grad():
        keep = _rnn(conn, 4.0, lg, b, al)
        keep.forward_io(u, ind, outd, 4)
        _rnn(conn, 4.0, lg, b, al).forward_io(u, ind, outd, 4)        # goes away: its memory is handed on below
        fresh = _rnn(conn, 4.0, lg, b, al)
    got = []

    def build():
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream), torch.no_grad():
            got.append(fresh.forward_io(u, ind, outd, 4))
            stream.synchronize()

    def other():
        thread = threading.Thread(target=build)
        thread.start()
        thread.join()

    _captured(other, mode)
    np.testing.assert_allclose(got[0].cpu().numpy(), ref, rtol=2e-5, atol=2e-5 * max(np.abs(ref).max(), 1.0))
