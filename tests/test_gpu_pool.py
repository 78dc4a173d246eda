"""The library's device memory pool: objects of one weight version after another reuse memory, an old plan's memory is not
handed on while another stream still runs a forward of it, and threads that build and destroy objects at once each get
the right answers."""

from __future__ import annotations

import threading

import numpy as np
import pytest
import torch

from helpers import brain_arrays, random_params
from test_gpu_sweep import _cone, _medium, _rnn

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
    """Forwards of ten weight versions alternate between two streams with no wait in between: each new plan destroys the
    one that the other stream may still be running."""
    conn, (lg, b, al), ind, outd, u, ref = _case(3, 256)
    rnn = _rnn(conn, 4.0, lg, b, al)
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    outs = []
    torch.cuda.synchronize()
    with torch.no_grad():
        for i in range(10):
            with torch.cuda.stream(streams[i % 2]):
                rnn.bias.add_(0.0)                       # a new version of the same values
                outs.append(rnn.forward_io(u, ind, outd, 4))
    torch.cuda.synchronize()
    for out in outs:
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
