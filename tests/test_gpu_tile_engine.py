"""The small-tile GEMM engine (pan2_amd/csrc/pm_mid.hpp) against the 256-tile
engine and the fp64 oracle.

A lone mid-size matrix runs its stages as 64 x 64 or 128 x 128 tiles; beside a
5120 x 5120 matrix in one call every stage keeps 256 x 256 tiles. Both
accumulate each element in the same order, so the results agree bit for bit:
NS outputs, stepped params and momentum, at the tiles' edges and remainders, in
both forms, with contiguous params and with params whose rows no vector access
fits.
"""
import numpy as np
import pytest
import torch

from oracle import muon_ref
from pan2_amd import _lib
from tests.ksplit_rule import call_splits

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
COEFFS = (3.4445, -4.7750, 2.0315)
BIG = (5120, 5120)
# short sides at the edges of 64- and 128-wide tiles (3 units of k and more),
# long sides with remainders, tall and wide; none splits its K alone
SHAPES = [(129, 129), (129, 191), (192, 193), (256, 255), (257, 256), (320, 130), (383, 385), (449, 577),
          (1000, 1024), (200, 2113), (3001, 140), (640, 900)]


def seeded(shape, seed, scale=1.0):
    g = torch.Generator(DEV).manual_seed(seed)
    return torch.empty(shape, device=DEV).normal_(0.0, scale, generator=g)


@pytest.fixture(scope="module")
def big():
    return seeded(BIG, 99).bfloat16()


def test_shapes_do_not_split():
    for s in SHAPES:
        assert call_splits([s]) == [(1, 1, 1)] and call_splits([s, BIG])[0] == (1, 1, 1), s


def ns(xs, form):
    outs = [torch.full(x.shape, float("nan"), dtype=torch.bfloat16, device=DEV) for x in xs]
    _lib.newton_schulz_into(list(zip(xs, outs)), ns_form=form)
    return outs


@pytest.mark.parametrize("form", ["standard", "gram"])
@pytest.mark.parametrize("shape", SHAPES)
def test_alone_equals_beside_a_large_matrix(shape, form, big):
    print(f"ns {shape} {form}", flush=True)
    x = seeded(shape, sum(shape))
    alone = ns([x], form)[0]
    assert torch.equal(alone, ns([big, x], form)[1])
    if form == "standard":
        ref = muon_ref.ns_standard(x.cpu().numpy(), precision="fp64")
        assert np.linalg.norm(alone.float().cpu().numpy() - ref) <= 2e-2 * np.linalg.norm(ref)


def strided(t, pad):
    """t in rows of cols + pad elements, its base one element off a 16-byte line when pad is odd."""
    rows, cols = t.shape
    buf = torch.zeros(rows * (cols + pad) + 8, dtype=t.dtype, device=DEV)
    v = buf[pad % 2:][:rows * (cols + pad)].view(rows, cols + pad)[:, :cols]
    v.copy_(t)
    return v


@pytest.mark.parametrize("pdt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("pad", [0, 8, 3])
@pytest.mark.parametrize("shape", [(129, 191), (320, 130), (449, 577), (1000, 1024)])
def test_step_equals_the_step_beside_a_large_matrix(shape, pad, pdt, big):
    print(f"step {shape} pad {pad} {pdt}", flush=True)
    p0, g0, m0 = seeded(shape, 1, 0.02).to(pdt), seeded(shape, 2, 1e-3).to(pdt), seeded(shape, 3, 1e-3)
    got = []
    for beside in (False, True):
        ps, gs, ms = ([strided(t, pad)] for t in (p0, g0, m0))
        if beside:
            ps, gs, ms = ps + [big.to(pdt)], gs + [big.to(pdt)], ms + [big.float()]
        _lib.muon_step(ps, gs, ms, [0.3] * len(ps), lr=torch.tensor(0.02, device=DEV), weight_decay=0.01,
                       momentum=0.95, nesterov=True, ns_coefficients=COEFFS, ns_steps=5, eps=1e-7)
        got.append((ps[0], ms[0]))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])


@pytest.mark.parametrize("shape", [(1024, 4096), (2048, 2048), (600, 2000), (2050, 2000)])
def test_split_stages_against_the_oracle(shape):
    """Alone, these run K-split stages on small tiles (chunk partials and reduce)."""
    assert max(call_splits([shape])[0]) > 1
    x = seeded(shape, 5)
    out = ns([x], "standard")[0]
    # the reference in float64 on the device: the same quintic as the oracle's
    y = x.double() if shape[0] <= shape[1] else x.double().T.contiguous()
    y = y / y.norm()
    for _ in range(5):
        r = y @ y.T
        y = COEFFS[0] * y + (COEFFS[1] * r + COEFFS[2] * (r @ r)) @ y
    y = y if shape[0] <= shape[1] else y.T
    assert ((out.double() - y).norm() / y.norm()).item() <= 2e-2
