"""The head GEMM with its K loop in parts against float64, and against the unsplit loop: forced numbers of parts, whether
they divide the stages or not, on every tile shape that the automatic choice takes; and the full-size head's automatic
choice on both sides of each change of its parts."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

import helpers  # noqa: F401  (puts the package on the path)

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


class _Head:
    """A head with random maps, its outputs in float64, and the library's under given tuning."""

    def __init__(self, n_out, n_moves, seed):
        rng = np.random.default_rng(seed)
        self.rng, self.n_out, self.n_moves = rng, n_out, n_moves
        t = lambda *shape: torch.as_tensor(rng.normal(0, 1 / np.sqrt(n_out), shape).astype(np.float32), device=DEV)
        self.mean, self.var = t(n_out), t(n_out).abs() + 0.5
        self.w = {"policy": t(n_moves, n_out), "from": t(64, n_out), "to": t(64, n_out), "value": t(3, n_out)}
        self.b = {k: t(v.shape[0]) for k, v in self.w.items()}
        self.squares = [torch.as_tensor(rng.integers(0, 64, n_moves).astype(np.int32), device=DEV) for _ in range(2)]
        self.enc = t(5, 7), t(5)

    def outputs(self, batch):
        return torch.as_tensor(self.rng.normal(0, 1, (self.n_out, batch)).astype(np.float32), device=DEV)

    def float64(self, r):
        n = ((r.double().T - self.mean.double()) / (self.var.double() + 1e-8).sqrt()).clamp(-8, 8)
        f64 = {k: n @ self.w[k].double().T.contiguous() + self.b[k].double() for k in self.w}
        return f64["policy"] + f64["from"][:, self.squares[0].long()] + f64["to"][:, self.squares[1].long()], f64["value"]

    def run(self, r, **tuning):
        from chessfly import _hip
        lib = _hip.load()
        batch = r.shape[1]
        desc = _hip.HeadDesc(self.n_out, self.n_moves, self.mean.data_ptr(), self.var.data_ptr(), 1e-8, 8.0,
                             *[p.data_ptr() for k in self.w for p in (self.w[k], self.b[k])],
                             *[s.data_ptr() for s in self.squares])
        for k, v in tuning.items():
            _hip.set_tuning(k, v)
        try:
            handle = ctypes.c_void_p()
            _hip.check(lib.fly_dense_create(ctypes.byref(desc), self.enc[0].data_ptr(), 7, 7, self.enc[1].data_ptr(), 5,
                                            _hip.stream(r.device), ctypes.byref(handle)), "fly_dense_create")
        finally:
            for k in tuning:
                _hip.set_tuning(k, 0)
        dense = _hip.Handle(handle, "fly_dense_destroy")
        logits = torch.full((batch, self.n_moves), float("nan"), device=DEV)
        wdl = torch.full((batch, 3), float("nan"), device=DEV)
        ws = torch.full((max(int(lib.fly_head_workspace(dense.handle, batch)), 1),), 0xFF, dtype=torch.uint8, device=DEV)
        _hip.check(lib.fly_head(dense.handle, r.data_ptr(), batch, batch, logits.data_ptr(), wdl.data_ptr(), ws.data_ptr(),
                                ws.numel(), _hip.stream(r.device)), "fly_head")
        return logits, wdl


def _near(got, ref, what):
    # 22-bit operands and float32 sums of at most 3 (n_out + 1) products of order 1 / sqrt(n_out): 1e-5 of the scale
    for g, r in zip(got, ref):
        assert float((g.double() - r.double()).abs().max()) < 1e-5 * max(1.0, float(r.abs().max())), what


@pytest.mark.parametrize("n_out,n_moves", [(61, 40), (700, 301)])     # 1 stage of 64; 11 stages, moves not a multiple of 4
@pytest.mark.parametrize("batch", [1, 65, 130])
def test_head_in_parts_matches_float64(n_out, n_moves, batch):
    head = _Head(n_out, n_moves, n_out + batch)
    r = head.outputs(batch)
    ref = head.float64(r)
    for tile in (22, 25, 44):
        whole = head.run(r, gemm_tile=tile, gemm_splits=1)
        _near(whole, ref, (tile, 1))
        for splits in (2, 3, 8):
            got = head.run(r, gemm_tile=tile, gemm_splits=splits)
            _near(got, ref, (tile, splits))
            _near(got, whole, (tile, splits))
            if n_out <= 64:                       # one stage: one part, whatever was asked for
                assert all(torch.equal(g, w) for g, w in zip(got, whole))
    _near(head.run(r), ref, "automatic")


def test_full_size_head_on_both_sides_of_each_change_of_parts():
    """3, 2, 3, 1, 2 and 1 parts on 64 x 64 tiles, one on 64 x 160 and on 128 x 128, and two of 128 x 128."""
    head = _Head(2333, 4168, 5)
    r_all = head.outputs(2048)
    for batch in (1, 128, 129, 192, 193, 320, 321, 448, 449, 576, 577, 1120, 1500, 2048):
        r = r_all[:, :batch].contiguous()
        got, whole = head.run(r), head.run(r, gemm_splits=1)
        _near(got, head.float64(r), batch)
        _near(got, whole, batch)


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
