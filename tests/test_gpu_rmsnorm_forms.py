"""GPU parity of RMSNorm on both sides of the lines at which gamma is requested with the rows or behind them, for every number
of vectors a lane holds, with ragged widths.  Tolerance: one fp16 rounding (2^-11) and the fp32 sum: 1e-3 relative."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols", [(3072, 1024), (3073, 1024), (9000, 520), (9001, 1016), (3173, 4096), (3174, 4096), (40, 2056), (6000, 2064),
                                       (2258, 8192), (2259, 8192), (33, 4104), (4400, 4208), (700, 2048), (5, 8200), (20000, 24),
                                       (4150, 1024), (4151, 1024), (8192, 520), (8193, 520), (8192, 1016), (8193, 1016)])
@pytest.mark.parametrize("in_place", [False, True])
def test_rmsnorm_forms(rows, cols, in_place):
    from triton_amd import ops
    g = torch.Generator(device="cuda").manual_seed(rows + cols)
    x = torch.randn(rows, cols, generator=g, device="cuda").half()
    gamma = (torch.randn(cols, generator=g, device="cuda") * 0.1 + 1).half()
    f = x.float()
    want = f * (f.pow(2).mean(-1, keepdim=True) + 1e-5).rsqrt() * gamma.float()
    y = x if in_place else torch.full_like(x, 7.0)
    ops.rmsnorm(x, gamma, y, 1e-5)
    torch.cuda.synchronize()
    assert not ((y.float() - want).abs() > 1e-3 * want.abs() + 1e-6).any()
