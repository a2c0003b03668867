"""The norm kernel's projection outputs are dealt out to 4, 3, 2 or 1 workgroups per row by the batch: same bits for every row."""
import pytest
import torch

from tests import gpu_util as U

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B", [64, 65, 85, 86, 128, 129, 256, 257])
@pytest.mark.parametrize("C,n", [(512, 8), (2048, 15), (4096, 32)])
def test_shares_of_a_row(B, C, n):
    from lyra_amd.kernels import decode_fused as F

    gen = torch.Generator(device=U.dev()).manual_seed(B + C)
    x = torch.randn(B, C, device=U.dev(), generator=gen).to(torch.bfloat16)
    scale, proj, bias = (torch.randn(*s, device=U.dev(), generator=gen) for s in ((C,), (C, n), (n,)))
    h, y = F.rmsnorm_proj(x, scale, 1e-5, proj, bias)
    parts = [F.rmsnorm_proj(rows.contiguous(), scale, 1e-5, proj, bias) for rows in x.split(32)]  # (4 workgroups per row)
    assert torch.equal(h, torch.cat([p[0] for p in parts])) and torch.equal(y, torch.cat([p[1] for p in parts]))
