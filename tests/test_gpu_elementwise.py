"""pm_momentum_nesterov and pm_step_param over sizes around their 4096-element
blocks, at bases off any vector boundary, in every mix of dtypes, bit for bit
against the oracle's fp32 arithmetic; nothing past the last element changes."""
import itertools

import numpy as np
import pytest
import torch

from oracle import muon_ref
from pan2_amd import _lib

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
F, B = torch.float32, torch.bfloat16


def make(n, dtype, off, seed):
    """n elements starting off elements into a buffer of n + 16."""
    g = torch.Generator("cpu").manual_seed(seed)
    buf = torch.randn(n + 16, generator=g).to(dtype).to(DEV)
    return buf, buf[off:off + n]


@pytest.mark.parametrize("n", [1, 3, 1023, 4095, 4096, 4097, 8192, 12293])
@pytest.mark.parametrize("dtypes", list(itertools.product((F, B), repeat=3)))
def test_momentum(n, dtypes):
    off = n % 3  # 0, 1 or 2 elements off the allocation
    (mb, m), (_, g), (ub, u) = (make(n, dt, off, i) for i, dt in enumerate(dtypes))
    m0, tail_m, tail_u = m.clone(), mb.clone(), ub.clone()
    _lib.momentum_nesterov_into(m, g, u, 0.95, True)
    want_m, want_u = muon_ref.momentum_nesterov(m0.float().cpu().numpy(), g.float().cpu().numpy(), 0.95, True)
    assert torch.equal(m.cpu(), torch.from_numpy(want_m).to(dtypes[0]))
    assert torch.equal(u.cpu(), torch.from_numpy(want_u).to(dtypes[2]))
    for now, was in ((mb, tail_m), (ub, tail_u)):
        assert torch.equal(now[:off], was[:off]) and torch.equal(now[off + n:], was[off + n:])


@pytest.mark.parametrize("n", [1, 4095, 4096, 12293])
def test_momentum_into_the_grad(n):
    (_, m), (_, g) = (make(n, dt, 0, i) for i, dt in enumerate((F, B)))
    _, want = muon_ref.momentum_nesterov(m.cpu().numpy(), g.float().cpu().numpy(), 0.95, True)
    _lib.momentum_nesterov_into(m, g, g, 0.95, True)
    assert torch.equal(g.cpu(), torch.from_numpy(want).to(B))


@pytest.mark.parametrize("n", [1, 3, 1023, 4095, 4096, 4097, 8192, 12293])
@pytest.mark.parametrize("dtypes", list(itertools.product((F, B), repeat=2)))
def test_step(n, dtypes):
    off = n % 3
    (pb, p), (_, u) = (make(n, dt, off, 7 + i) for i, dt in enumerate(dtypes))
    p0, was = p.clone(), pb.clone()
    _lib.step_param_inplace(p, u, 0.02, 0.01, 1.5)
    want = muon_ref.step_param(p0.float().cpu().numpy(), u.float().cpu().numpy(), 0.02, 0.01, 1.5)
    assert torch.equal(p.cpu(), torch.from_numpy(np.asarray(want, dtype=np.float32)).to(dtypes[0]))
    assert torch.equal(pb[:off], was[:off]) and torch.equal(pb[off + n:], was[off + n:])


def test_step_of_more_elements_than_one_launch_holds():
    """2^36 elements are 2^24 blocks, 2^32 threads: more than a launch may
    hold. The tensor is its own update, so that one of 128 GiB does."""
    n = (1 << 36) + 4099
    if torch.cuda.mem_get_info()[0] < 2 * n + (8 << 30):
        pytest.skip("needs 136 GiB of free GPU memory")
    p = torch.ones(n, dtype=B, device=DEV)
    try:
        _lib.step_param_inplace(p, p, 0.5, 0.0, 1.0)  # p - 0.5 p, exact
        for i in range(0, n, 1 << 30):
            assert bool((p[i:i + (1 << 30)] == 0.5).all()), i
    finally:
        del p
        torch.cuda.empty_cache()
