"""GPU parity of the small-batch state step against the CPU oracle: the narrow kernel at every width of its rows (2, 4, 16
and 32 bytes, and the first batches past them), and the staged sums of long-row steps on a graph just past the size rule,
with rows of no partner, of one more than two rounds of 16, and hubs.

Tolerances as in test_gpu_sweep.py: float32 within float32 round-off of the float64 oracle (2e-5); the float16 state within
2e-3 of the deviation's own scale, or 4e-3 of the largest activity where it holds the activity itself (six float16
roundings of the state and its sum per step)."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from helpers import brain_arrays, random_params
from test_gpu_sweep import _forward_io_both, _heavy_tailed, _rnn

from oracle import forward as F

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("batch", [1, 2, 3, 4, 5, 8, 9, 12, 16, 17, 32, 33])
def test_narrow_batches_match_the_oracle(batch):
    conn = _heavy_tailed(3)
    lg, b, al = random_params(conn, 9, gain_sd=0.1)
    rnn = _rnn(conn, 4.0, lg, b, al)
    ba = brain_arrays(conn, 4.0, lg, b, al, dtype=torch.float64)
    _forward_io_both(rnn, conn, ba, batch, 6, 200 + batch, "auto")
    u = torch.randn(conn.n_neurons, batch, generator=torch.Generator().manual_seed(batch))
    with torch.no_grad():
        h = rnn(u.clone().to(DEV), 4)
        h16 = rnn(u.half().to(DEV), 4)
    ref = F.literal(ba, u.double(), 4).numpy()
    np.testing.assert_allclose(h.cpu().numpy(), ref, rtol=2e-5, atol=2e-5 * np.abs(ref).max())
    ref = F.literal(ba, u.half().double(), 4).numpy()
    np.testing.assert_allclose(h16.double().cpu().numpy(), ref, rtol=0, atol=4e-3 * np.abs(ref).max())


def _kernels(call):
    """call()'s result, and the names of the kernels that it launched."""
    torch.cuda.synchronize()
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
        out = call()
        torch.cuda.synchronize()
    return out, " ".join(e.key for e in prof.key_averages())


def _staged_conn(n):
    """n neurons (no multiple of a row quad) of 36 partners on average: enough rows, sources and partners to be staged.
    The first and last rows are empty, some hold 33, 96 and 97 partners and three are hubs of thousands."""
    from chessfly.synthetic import degree_connectome
    rng = np.random.default_rng(5)
    deg = rng.poisson(36, n)
    deg[[0, 1, n - 1]] = 0
    deg[10:14] = [33, 96, 97, 129]
    deg[[5, 40_000, n - 2]] = [20_000, 9_193, 3_000]
    ids = rng.permutation(n)
    conn = degree_connectome(deg, np.sort(ids[:500]), np.sort(ids[500:700]), seed=6)
    return conn, random_params(conn, 4, gain_sd=0.1)


@pytest.fixture(scope="module", params=[70_001, 150_001])
def staged_net(request):
    """Graphs whose states of 2 bytes a row take 1 and 3 bands of LDS, and of 4 bytes 2 and 5."""
    conn, (lg, b, al) = _staged_conn(request.param)
    return conn, _rnn(conn, 4.0, lg, b, al), brain_arrays(conn, 4.0, lg, b, al, dtype=torch.float64)


@pytest.mark.parametrize("batch,dtype", [(1, torch.float32), (1, torch.float16), (2, torch.float16)])
def test_staged_steps_match_the_oracle(staged_net, batch, dtype):
    conn, rnn, ba = staged_net
    u = torch.randn(conn.n_neurons, batch, generator=torch.Generator().manual_seed(batch)).to(dtype)
    with torch.no_grad():
        h, kernels = _kernels(lambda: rnn(u.clone().to(DEV), 3))
    assert "k_stage_sums" in kernels, kernels
    ref = F.literal(ba, u.double(), 3).numpy()
    tol = 2e-5 if dtype == torch.float32 else 4e-3
    np.testing.assert_allclose(h.double().cpu().numpy(), ref, rtol=0, atol=tol * np.abs(ref).max())


@pytest.mark.parametrize("batch", [1, 2])
def test_staged_steps_of_the_light_cone_match_the_oracle(staged_net, batch):
    """Enough steps for the cone to reach every neuron: its middle steps are staged in both state types at one position, in
    half columns at two."""
    conn, rnn, ba = staged_net
    ind, outd = conn.nodes("afferent").to(DEV), conn.nodes("efferent").to(DEV)
    u = torch.randn(len(ind), batch, generator=torch.Generator().manual_seed(batch))
    with torch.no_grad():
        for dtype in (torch.float16, torch.float32):
            _, kernels = _kernels(lambda: rnn.forward_io(u.to(DEV, dtype), ind, outd, 8))
            assert ("k_stage_sums" in kernels) == (batch * dtype.itemsize <= 4), kernels
    _forward_io_both(rnn, conn, ba, batch, 8, batch, "auto")


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_staged_steps_of_unbounded_activity_match_the_oracle(dtype):
    conn, (lg, b, al) = _staged_conn(70_001)
    rnn = _rnn(conn, 0.5, lg, b + 20.0, al, h_max=None)       # activities past the bound that there would be
    ba = brain_arrays(conn, 0.5, lg, b + 20.0, al, h_max=float("inf"), dtype=torch.float64)
    u = torch.randn(conn.n_neurons, 1, generator=torch.Generator().manual_seed(1)).to(dtype)
    with torch.no_grad():
        h, kernels = _kernels(lambda: rnn(u.clone().to(DEV), 3))
    assert "k_stage_sums" in kernels, kernels
    ref = F.literal(ba, u.double(), 3).numpy()
    assert np.abs(ref).max() > 15
    tol = 2e-5 if dtype == torch.float32 else 4e-3
    np.testing.assert_allclose(h.double().cpu().numpy(), ref, rtol=0, atol=tol * np.abs(ref).max())


def test_stage_tables_are_built_for_plans_only():
    """Training's products sweep the same structures and never read them."""
    from chessfly import _hip
    conn, (lg, b, al) = _staged_conn(70_001)
    rnn = _rnn(conn, 4.0, lg, b, al)
    u = torch.zeros(conn.n_neurons, 1, device=DEV)
    with torch.no_grad():
        tables, kernels = _kernels(lambda: _hip.sweep_create(rnn.crow32, rnn.pre32, rnn.n, rnn.n))
        assert tables is not None and "k_band_off" in kernels and "k_stage_starts" not in kernels, kernels
        _, kernels = _kernels(lambda: rnn(u, 2))
        assert "k_stage_starts" in kernels, kernels
        rnn.bias.add_(0.0)                                      # another weight version of the same structure
        _, kernels = _kernels(lambda: rnn(u, 2))
        assert "k_stage_sums" in kernels and "k_stage_starts" not in kernels, kernels
