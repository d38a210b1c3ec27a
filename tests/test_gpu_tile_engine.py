"""The small-tile GEMM engine (pan2_amd/csrc/pm_mid.hpp) against the 256-tile
engine and the fp64 oracle.

A lone mid-size matrix runs its stages as 64 x 64 tiles, several larger ones as
128 x 128 tiles, or as those beside 256-tile stages; with 5120 x 5120 matrices
in the call every stage keeps 256 x 256 tiles. All accumulate each element in
the same order, so the results agree bit for bit: NS outputs, stepped params and
momentum, at the tiles' edges and remainders, in both forms, with contiguous
params and with params whose rows no vector access fits. Each test checks in the
launch records which tiles ran. The split stages, which no call runs on
256-tiles at the same split, are held to the fp64 Newton-Schulz.
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


def tiles_of(call):
    """call()'s result, and the tile edges that its launches of each stage ran on."""
    _lib.timing_enable(True)
    try:
        _lib.timing_read()
        out = call()
        edges = {}
        for r in _lib.timing_read():
            if r["tile"]:
                edges.setdefault(r["kind"], set()).add(r["tile"])
    finally:
        _lib.timing_enable(False)
    return out, edges


STAGES = ("gram", "poly", "update", "final")


def all_on(edge):
    return {k: {edge} for k in STAGES}


def ns(xs, form):
    outs = [torch.full(x.shape, float("nan"), dtype=torch.bfloat16, device=DEV) for x in xs]
    _lib.newton_schulz_into(list(zip(xs, outs)), ns_form=form)
    return outs


@pytest.mark.parametrize("form", ["standard", "gram"])
@pytest.mark.parametrize("shape", SHAPES)
def test_alone_equals_beside_a_large_matrix(shape, form, big):
    print(f"ns {shape} {form}", flush=True)
    x = seeded(shape, sum(shape))
    (alone,), edges = tiles_of(lambda: ns([x], form))
    (_, beside), big_edges = tiles_of(lambda: ns([big, x], form))
    assert edges == all_on(64) and big_edges == all_on(256)
    assert torch.equal(alone, beside)
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


def step(ps, gs, ms):
    _lib.muon_step(ps, gs, ms, [0.3] * len(ps), lr=torch.tensor(0.02, device=DEV), weight_decay=0.01,
                   momentum=0.95, nesterov=True, ns_coefficients=COEFFS, ns_steps=5, eps=1e-7)


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
        _, edges = tiles_of(lambda: step(ps, gs, ms))
        assert edges == all_on(256 if beside else 64)
        got.append((ps[0], ms[0]))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])


# Calls in which no stage splits, and the edge each of their stages runs on:
#   more 128-tiles of one length than CUs in every stage (persistent blocks take
#   several, the next one's copies ahead of an epilogue; the gram form's Q
#   written with Z on 128-tiles);
#   the same products beside UPDATE and FINAL on 256-tiles, which read padding;
#   128-tiles of several lengths (a block each), wide and tall;
#   a lone tall matrix whose products run on 64-tiles, its FINAL on 350 of 128.
GROUPS = {
    "persistent": ([(1536, 1530)] * 8, (128, 128, 128)),
    "beside_256": ([(1536, 1530)] * 6, (128, 128, 256)),
    "lengths": ([(1531, 1400), (1300, 2111), (2111, 1333), (1750, 1700), (1790, 1600)], (128, 128, 128)),
    "tall": ([(3100, 1700)], (64, 64, 128)),
}


def edges_of(group):
    gram, poly, full = GROUPS[group][1]
    return {"gram": {gram}, "poly": {poly}, "update": {full}, "final": {full}}


def test_groups_do_not_split():
    for shapes, _ in GROUPS.values():
        assert set(call_splits(shapes)) == {(1, 1, 1)} and set(call_splits(shapes + [BIG] * 3)) == {(1, 1, 1)}


@pytest.mark.parametrize("form", ["standard", "gram"])
@pytest.mark.parametrize("group", list(GROUPS))
def test_groups_equal_the_same_beside_large_matrices(group, form, big):
    print(f"ns group {group} {form}", flush=True)
    xs = [seeded(s, 10 + i) for i, s in enumerate(GROUPS[group][0])]
    outs, edges = tiles_of(lambda: ns(xs, form))
    beside, big_edges = tiles_of(lambda: ns([big] * 3 + xs, form))
    assert edges == edges_of(group) and big_edges == all_on(256)
    for i, (a, b) in enumerate(zip(outs, beside[3:])):
        assert torch.equal(a, b), i


@pytest.mark.parametrize("pdt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("pad", [0, 3])
@pytest.mark.parametrize("group", list(GROUPS))
def test_group_steps_equal_the_same_beside_large_matrices(group, pad, pdt, big):
    print(f"step group {group} pad {pad} {pdt}", flush=True)
    shapes = GROUPS[group][0]
    data = [(seeded(s, 3 * i, 0.02).to(pdt), seeded(s, 3 * i + 1, 1e-3).to(pdt), seeded(s, 3 * i + 2, 1e-3))
            for i, s in enumerate(shapes)]
    got = []
    for beside in (False, True):
        ps, gs, ms = ([strided(d[k], pad) for d in data] for k in range(3))
        large = [[big.to(dt, copy=True) for _ in range(3 if beside else 0)] for dt in (pdt, pdt, torch.float32)]
        _, edges = tiles_of(lambda: step(ps + large[0], gs + large[1], ms + large[2]))
        assert edges == (all_on(256) if beside else edges_of(group))
        got.append(ps + ms)
    for i, (a, b) in enumerate(zip(*got)):
        assert torch.equal(a, b), i


@pytest.mark.parametrize("shape", [(1024, 4096), (2048, 2048), (600, 2000), (2050, 2000)])
def test_split_stages_against_the_oracle(shape):
    """Alone, these run K-split stages on small tiles (chunk partials and reduce)."""
    assert max(call_splits([shape])[0]) > 1
    x = seeded(shape, 5)
    (out,), edges = tiles_of(lambda: ns([x], "standard"))
    assert not any(256 in e for e in edges.values()), edges
    # the reference in float64 on the device: the same quintic as the oracle's
    y = x.double() if shape[0] <= shape[1] else x.double().T.contiguous()
    y = y / y.norm()
    for _ in range(5):
        r = y @ y.T
        y = COEFFS[0] * y + (COEFFS[1] * r + COEFFS[2] * (r @ r)) @ y
    y = y if shape[0] <= shape[1] else y.T
    assert ((out.double() - y).norm() / y.norm()).item() <= 2e-2
