"""GPU parity of RMSNorm on both sides of the line from which a workgroup has one row: partial last vectors of a lane, a row in place, rows at a pitch.

Tolerance against float64: the output is rounded to fp16 once, 2^-11 of it; the sum of squares and its root add a few roundings of 2^-24."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("rows,cols", [(1, 1024), (3, 1032), (400, 1032), (401, 1032), (1200, 1280), (1201, 1280), (5, 2048), (5, 2056), (2, 4096), (2, 4104), (1200, 4104),
                                       (1201, 4104), (1, 8192), (9, 8200), (4, 16384), (1, 16376)])
def test_a_row_to_a_workgroup(rows, cols, weighted):
    from triton_amd import ops
    g = torch.Generator(device="cuda").manual_seed(rows + cols)
    buf = torch.full((rows + 1, cols + 8), float("nan"), dtype=torch.half, device="cuda")
    x = buf[:rows, :cols]
    x.copy_(torch.randn(rows, cols, generator=g, device="cuda") * 3)
    gamma = torch.randn(cols, generator=g, device="cuda").half() if weighted else None
    want = x.double() * torch.rsqrt((x.double() ** 2).mean(1, keepdim=True) + 1e-5)
    if weighted:
        want = want * gamma.double()
    y = torch.full_like(x, 7.0, memory_format=torch.contiguous_format)
    ops.rmsnorm(x, gamma, y, 1e-5)
    ops.rmsnorm(x, gamma, x, 1e-5)
    assert torch.equal(x, y) and buf[rows].isnan().all() and buf[:, cols:].isnan().all()
    assert ((y.double() - want).abs() <= (2 ** -11 + 1e-6) * want.abs() + 2 ** -25).all()
