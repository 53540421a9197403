"""Masked scores are not read as values: a softmax whose masked columns hold
NaN, infinities or the largest float equals the one over the unmasked
columns (float64), and the masked columns come out exactly 0."""
import pytest
import torch

from chatterbox_amdvulkan_amd import cbxops as C

pytestmark = pytest.mark.gpu


# wave-per-row kernels (float4, float2), the one-wave and the workgroup row
# kernels for few rows, odd lengths of many rows; masks from the first column on
@pytest.mark.parametrize("heads,q,n_past", [(16, 512, 0), (16, 512, 3), (8, 250, 0), (8, 251, 0), (2, 300, 37), (1, 5, 2000),
                                            (4, 64, 0), (16, 333, 0), (300, 5, 0)])
@pytest.mark.parametrize("add", [False, True])
def test_masked_columns(cbx, heads, q, n_past, add):
    kv = q + n_past
    g = torch.Generator(device="cuda")
    g.manual_seed(heads * q + n_past)
    x = torch.randn((heads, q, kv), generator=g, device="cuda") * 4
    b = torch.randn((heads, q, kv), generator=g, device="cuda") * 4 if add else None
    seen = torch.arange(kv, device="cuda")[None] <= n_past + torch.arange(q, device="cuda")[:, None]
    junk = torch.tensor([float("nan"), float("inf"), 3.4e38, float("-inf")], device="cuda")
    x = torch.where(seen, x, junk[torch.arange(kv, device="cuda") % 4])
    y = C.add_scale_diag_mask_soft_max(x, b, 0.125, n_past) if add else C.scale_diag_mask_soft_max(x, 0.125, n_past)
    s = torch.where(seen, (x + b if add else x).double() * 0.125, float("-inf"))
    ref = torch.softmax(s, -1)
    assert not y[(~seen).expand_as(y)].any()
    # f32 scores times a power of two, expf and one product: a few 2^-23
    assert float((y.double() - ref).norm() / ref.norm()) < 1e-6
    assert torch.allclose(y.double(), ref, rtol=3e-6, atol=1e-30)
