"""Filter gradients whose output channels lie side by side in memory (Dense "IO"): the sums over reduction slices that turn
their tiles over in LDS against the same gradient in the "OI" layout, at tile remainders on either side."""
import pytest
import torch

import phoenix_core_amd as phx
from phoenix_core_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32], ids=["f16", "f32"])
@pytest.mark.parametrize("n,ci,co", [(256, 512, 512), (264, 513, 509), (200, 129, 1030), (72, 1030, 131)])
def test_dense_filter_gradient_layouts_agree(n, ci, co, dtype):
    """Both layouts sum the same partial results and differ by the order of at most 16 fp32 additions (16 x 2^-24 of the sum
    of their absolute values, at most n x the largest products) and one rounding to the output's type.  The input gradients
    read the filter eight values a load or one by one and are equal bit for bit."""
    gen = torch.Generator(device="cuda").manual_seed(ci)
    x, grad = (torch.randn((4 * n, c), generator=gen, device="cuda").to(dtype) for c in (ci, co))
    w = torch.randn((4, ci, co), generator=gen, device="cuda").to(dtype)
    io = ops.DenseDescriptor(x.shape, w.shape, dtype=dtype)
    w_oi = w.transpose(1, 2).contiguous()
    oi = ops.DenseDescriptor(x.shape, w_oi.shape, filter_layout="OI", dtype=dtype)
    dw, dx = phx.dense_bwd(x, w, grad, io)
    dw_oi, dx_oi = phx.dense_bwd(x, w_oi, grad, oi)
    assert torch.equal(dx, dx_oi)
    assert torch.equal(phx.dense_fwd(x, w, None, io), phx.dense_fwd(x, w_oi, None, oi))
    a, b = dw.double(), dw_oi.transpose(1, 2).double()
    bound = (2.0 ** -10 if dtype == torch.float16 else 2.0 ** -23) * b.abs() + 16 * 2.0 ** -24 * 4 * n * float(x.abs().max()) * float(grad.abs().max())
    assert bool(((a - b).abs() <= bound).all())
