"""The Muon step's descriptor pass (_pm_host.fill_muon) on CPU tensors: every
field through the ctypes layout, and the lists that it leaves to the checking
loop of patch_muon._single_tensor_muon."""
import numpy as np
import pytest
import torch

from pan2_amd import _lib
from pan2_amd.optim import patch_muon as pm


def fill(params, grads, bufs, ratios, chunks, n=None):
    arr = np.empty(len(params) * chunks if n is None else n, dtype=_lib._PM_MATRIX_NP)
    arr.view(np.uint8)[:] = 0xa5
    rc = _lib.host_ext().fill_muon(arr.ctypes.data, params, grads, bufs, ratios, chunks, hip_only=False)
    return rc, arr


@pytest.mark.parametrize("chunks", [1, 3])
def test_every_field(chunks):
    shapes = [(6, 5), (3, 8), (9, 1)]
    ps = [torch.zeros(s, dtype=torch.bfloat16) for s in shapes]
    gs = [torch.zeros(s, dtype=torch.float32) for s in shapes]
    bs = [torch.zeros(s, dtype=torch.float32) for s in shapes]
    rc, arr = fill(ps, gs, bs, [0.5, 1.5, 2.5], chunks)
    assert rc == _lib.host_ext().FILLED
    for i, (r, c) in enumerate(shapes):
        rows = r // chunks
        for k in range(chunks):
            e = arr[i * chunks + k]
            assert e["param"] == ps[i].data_ptr() + k * rows * c * 2
            assert e["grad"] == gs[i].data_ptr() + k * rows * c * 4
            assert e["momentum"] == bs[i].data_ptr() + k * rows * c * 4
            assert (e["rows"], e["cols"]) == (rows, c) and e["param_ld"] == e["grad_ld"] == e["momentum_ld"] == c
            assert (e["param_dtype"], e["grad_dtype"], e["momentum_dtype"]) == (1, 0, 0)
            assert e["reserved"] == 0 and e["adj_ratio"] == (0.5, 1.5, 2.5)[i]


class Wrapped(torch.Tensor):
    """A subclass with its own dispatch, as DTensor is."""

    @classmethod
    def __torch_dispatch__(cls, func, types, args=(), kwargs=None):
        raise NotImplementedError


def test_left_to_the_checking_loop():
    ok = lambda *s: torch.zeros(*(s or (4, 6)))  # noqa: E731
    general = _lib.host_ext().GENERAL
    sub = torch.Tensor._make_wrapper_subclass(Wrapped, (4, 6))
    cases = [
        ([ok()], [ok()], [ok()], [1.0], 3),                          # rows not a multiple of the blocks
        ([ok()], [ok(4, 5)], [ok()], [1.0], 1),                      # shapes differ
        ([ok(4)], [ok(4)], [ok(4)], [1.0], 1),                       # not a matrix
        ([ok(0, 6)], [ok(0, 6)], [ok(0, 6)], [1.0], 1),              # empty
        ([ok(6, 4).T], [ok()], [ok()], [1.0], 1),                    # not contiguous
        ([ok()], [ok().double()], [ok()], [1.0], 1),                 # dtype
        ([ok()], [ok()], [ok().half()], [1.0], 1),
        ([sub], [ok()], [ok()], [1.0], 1),                           # a subclass with its own dispatch
        ([ok(), ok()], [ok()], [ok(), ok()], [1.0, 1.0], 1),         # list lengths
        ([ok()], [ok()], [ok()], [], 1),
    ]
    for i, (p, g, b, r, k) in enumerate(cases):
        assert fill(p, g, b, r, k, n=8)[0] == general, i
    # the product path takes HIP tensors only
    assert _lib.muon_descs([ok()], [ok()], [ok()], [1.0], 1) is None


def test_group_ratio_is_the_row_blocks(monkeypatch):
    """Each shape's ratio is looked up once, with the row block's shape."""
    seen = []
    monkeypatch.setattr(pm, "_adjust_ratio", lambda fn, shape: seen.append((fn, tuple(shape))) or len(seen) * 1.0)
    got = {}
    monkeypatch.setattr(_lib, "muon_descs", lambda p, g, b, ratios, chunks: got.update(r=ratios, k=chunks) or "arr")

    class P:
        is_cuda = True

        def __init__(self, *s):
            self.shape = torch.Size(s)

    ps = [P(6, 5), P(4, 5), P(6, 5)]
    assert pm._group_descs(ps, ps, ps, "f", 2) == "arr"
    assert seen == [("f", (3, 5)), ("f", (2, 5))] and got == {"r": [1.0, 2.0, 1.0], "k": 2}
    assert pm._group_descs([P(5, 5)], None, None, "f", 2) is None
    assert pm._group_descs(ps, ps, ps, "f", 0) is None
