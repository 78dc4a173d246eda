"""The head GEMM with its K loop in parts (gemm_splits, and the automatic choice at the batches where it changes) against
float64, and against the unsplit loop: the shares of K add up, whatever their number and whether it divides the stages."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

import helpers  # noqa: F401  (puts the package on the path)

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("n_out,n_moves", [(61, 40), (700, 301)])     # 1 stage of 64; 11 stages, moves not a multiple of 4
@pytest.mark.parametrize("batch", [1, 65, 130])
def test_head_in_parts_matches_float64(n_out, n_moves, batch):
    from chessfly import _hip
    lib = _hip.load()
    rng = np.random.default_rng(n_out + batch)
    t = lambda *shape: torch.as_tensor(rng.normal(0, 1 / np.sqrt(n_out), shape).astype(np.float32), device=DEV)
    mean, var = t(n_out), t(n_out).abs() + 0.5
    w = {"policy": t(n_moves, n_out), "from": t(64, n_out), "to": t(64, n_out), "value": t(3, n_out)}
    b = {k: t(v.shape[0]) for k, v in w.items()}
    squares = [torch.as_tensor(rng.integers(0, 64, n_moves).astype(np.int32), device=DEV) for _ in range(2)]
    enc_w, enc_b = t(5, 7), t(5)
    r = torch.as_tensor(rng.normal(0, 1, (n_out, batch)).astype(np.float32), device=DEV)
    desc = _hip.HeadDesc(n_out, n_moves, mean.data_ptr(), var.data_ptr(), 1e-8, 8.0,
                         *[p.data_ptr() for k in w for p in (w[k], b[k])], *[s.data_ptr() for s in squares])
    n = ((r.double().T - mean.double()) / (var.double() + 1e-8).sqrt()).clamp(-8, 8)
    f64 = {k: n @ w[k].double().T + b[k].double() for k in w}
    want = f64["policy"] + f64["from"][:, squares[0].long()] + f64["to"][:, squares[1].long()]
    for splits in (0, 1, 2, 3, 8):
        _hip.set_tuning("gemm_splits", splits)
        try:
            handle = ctypes.c_void_p()
            _hip.check(lib.fly_dense_create(ctypes.byref(desc), enc_w.data_ptr(), 7, 7, enc_b.data_ptr(), 5,
                                            _hip.stream(r.device), ctypes.byref(handle)), "fly_dense_create")
        finally:
            _hip.set_tuning("gemm_splits", 0)
        dense = _hip.Handle(handle, "fly_dense_destroy")
        logits = torch.full((batch, n_moves), float("nan"), device=DEV)
        wdl = torch.full((batch, 3), float("nan"), device=DEV)
        ws = torch.full((max(int(lib.fly_head_workspace(dense.handle, batch)), 1),), 0xFF, dtype=torch.uint8, device=DEV)
        _hip.check(lib.fly_head(dense.handle, r.data_ptr(), batch, batch, logits.data_ptr(), wdl.data_ptr(), ws.data_ptr(),
                                ws.numel(), _hip.stream(r.device)), "fly_head")
        # 22-bit operands and float32 sums of at most 3 (n_out + 1) products of order 1 / sqrt(n_out): 1e-5 of the scale
        for got, ref in ((logits, want), (wdl, f64["value"])):
            assert float((got.double() - ref).abs().max()) < 1e-5 * max(1.0, float(ref.abs().max())), splits


def test_workspace_of_a_batch_holds_every_smaller_one():
    """A smaller batch may run in more parts than a larger one (576 boards of the full-size head in two, 640 in one): the
    last block of a forward and a caller who keeps one workspace both use a larger batch's workspace for it."""
    from chessfly import _hip
    lib = _hip.load()
    n_out, n_moves = 100, 4168
    z = lambda *shape: torch.zeros(shape, device=DEV)
    maps = [z(n_moves, n_out), z(n_moves), z(64, n_out), z(64), z(64, n_out), z(64), z(3, n_out), z(3)]
    squares = torch.zeros(n_moves, dtype=torch.int32, device=DEV)
    mean, var, enc_w, enc_b = z(n_out), z(n_out) + 1, z(5, 7), z(5)
    desc = _hip.HeadDesc(n_out, n_moves, mean.data_ptr(), var.data_ptr(), 1e-8, 8.0, *[p.data_ptr() for p in maps],
                         squares.data_ptr(), squares.data_ptr())
    handle = ctypes.c_void_p()
    _hip.check(lib.fly_dense_create(ctypes.byref(desc), enc_w.data_ptr(), 7, 7, enc_b.data_ptr(), 5,
                                    _hip.stream(mean.device), ctypes.byref(handle)), "fly_dense_create")
    dense = _hip.Handle(handle, "fly_dense_destroy")
    sizes = [int(lib.fly_head_workspace(dense.handle, b)) for b in range(1, 3000)]
    assert all(a <= b for a, b in zip(sizes, sizes[1:]))
    # room for two parts of 576 boards beside the operands (2 x 2 bytes, 128 columns): float32 rows of 4,299 values
    assert sizes[639] >= 2 * 576 * 4299 * 4
