"""Newton–Schulz over a batch (one descriptor array from the batch's strides)
equals the same call on its slices, bit for bit."""
import pytest
import torch

from pan2_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form", ["standard", "gram"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("shape", [(1, 40, 70), (3, 128, 300), (5, 301, 77), (2, 130, 260)])
def test_batch_equals_its_slices(shape, dtype, form):
    g = torch.Generator("cuda:0").manual_seed(3)
    x = torch.empty(shape, device="cuda:0").normal_(0, 1, generator=g).to(dtype)
    a, b = (torch.full(shape, float("nan"), dtype=torch.bfloat16, device="cuda:0") for _ in range(2))
    _lib.newton_schulz_batch(x, a, ns_form=form)
    _lib.newton_schulz_into([(x[i], b[i]) for i in range(shape[0])], ns_form=form)
    assert torch.equal(a, b)
