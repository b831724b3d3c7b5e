"""RMSNorm with a residual add over every pair of element types and at the
edges of the kernels' ranges of columns and rows, against float64."""
import pytest
import torch

from test_gpu_parity import say

pytestmark = pytest.mark.gpu

# unit roundoff: half the spacing, relative to the start of the binade
ROUND = {torch.float32: 2.0 ** -24, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}
# half the spacing of its subnormals
SMALL = {torch.float32: 1e-30, torch.bfloat16: 1e-30, torch.float16: 2.0 ** -25}


# 4 and 1024 columns: one register kernel; 1028 and 4096: the other; one row,
# one row per wave, and several (rows that no wave has left over included)
@pytest.mark.parametrize("rows,C", [(1, 4), (5, 1024), (2049, 64), (4099, 260), (7, 1028), (2051, 1500),
                                     (5, 4096)])
@pytest.mark.parametrize("rdt", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("ydt", [torch.float32, torch.bfloat16, torch.float16])
def test_add_rmsnorm_types(gpu_ca, rows, C, rdt, ydt):
    say(f"[case] rows={rows} C={C} res {rdt} y {ydt}")
    g = torch.Generator(device="cuda").manual_seed(rows + C)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    x, res, w = r(rows, C), r(rows, C).to(rdt), torch.rand(C, generator=g, device="cuda") + 0.5
    gy, gs = r(rows, C).to(ydt), r(rows, C)
    a = [t.clone().requires_grad_(True) for t in (x, res, w)]
    s, y = gpu_ca.decoder._AddRMSNormFn.apply(*a, 1e-6, ydt)
    got = torch.autograd.grad([s, y], a, [gs, gy])
    b = [t.double().requires_grad_(True) for t in (x, res, w)]
    s64 = b[0] + b[1]
    y64 = b[2] * s64 * torch.rsqrt(s64.square().mean(-1, keepdim=True) + 1e-6)
    want = torch.autograd.grad([s64, y64], b, [gs.double(), gy.double()])
    assert s.dtype == torch.float32 and torch.equal(s.detach(), x + res.float())
    # y: its rounding, plus fp32 rounding of the mean and three products
    assert bool(((y.double() - y64).abs() <= (ROUND[ydt] + 2.0 ** -20) * y64.abs() + SMALL[ydt]).all())
    assert got[1].dtype == rdt
    # gradients: a rounding to the type, plus fp32 rounding of terms that
    # cancel (2^-20 of the largest; dweight sums the rows)
    for d, e, dt in zip(got, want, (torch.float32, rdt, torch.float32)):
        bound = ROUND[dt] * e.abs() + 2.0 ** -20 * e.abs().max() + SMALL[dt]
        assert bool(((d.double() - e).abs() <= bound).all())
