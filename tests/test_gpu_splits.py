"""Split lengths picked by estimated time (split_cost in csrc/ca_abi.hip): the
operator under the picked splits against its own uncut work items, which sum
the same fp32 terms in another order (each sum at most ~2e-6 of the largest
element from the exact one, tests/test_gpu_parity.py; 5e-6 for the two)."""
import pytest
import torch

from test_gpu_parity import make_inputs, say

pytestmark = pytest.mark.gpu


# whole groups few (one slice), about a round, several rounds, and many
# rounds (nothing cut); each kernel family; a capped workspace (passes)
@pytest.mark.parametrize("shape,dtype,cap", [
    ((1, 1, 700, 64), torch.float32, 0), ((1, 1, 1025, 16), torch.bfloat16, 0),
    ((1, 3, 1537, 128), torch.float32, 0), ((2, 8, 768, 80), torch.float32, 0),
    ((4, 16, 1001, 64), torch.bfloat16, 0), ((8, 16, 1500, 64), torch.bfloat16, 0),
    ((1, 8, 2000, 64), torch.float32, 24 << 20), ((64, 512, 3, 8), torch.float32, 0)])
def test_picked_splits_match_whole_items(gpu_ca, shape, dtype, cap):
    say(f"[case] {shape} {dtype} cap {cap}")
    t = [x.to(dtype).cuda() for x in make_inputs(shape, 3, 1.0)[:3]]
    dy = torch.randn(shape, device="cuda").to(dtype)
    rho = torch.linspace(-0.2, 0.2, shape[1], device="cuda")

    def run():
        q, k, v, r = (x.clone().requires_grad_(True) for x in (*t, rho))
        y = gpu_ca.continuum_attention(q, k, v, r)
        return [x.detach().float() for x in (y, *torch.autograd.grad(y, (q, k, v, r), dy))]

    prev = gpu_ca.ops.workspace_cap()
    try:
        if cap:
            gpu_ca.ops.set_workspace_cap(cap)
        got = run()
        assert all(torch.equal(a, b) for a, b in zip(got, run()))  # fixed merge order
        gpu_ca.ops.set_split_override(1 << 20, 1 << 20, 1 << 20)
        whole = run()
    finally:
        gpu_ca.ops.set_split_override()
        gpu_ca.ops.set_workspace_cap(prev)
    # 16-bit outputs: a rounding of one or the other neighbour
    ulp = 0.0 if dtype == torch.float32 else 2.0 ** -7
    for i, (a, b) in enumerate(zip(got, whole)):
        step = ulp if i < 4 else 0.0
        # the gain gradient sums T^2 / 2 signed terms per slice
        tol = 5e-6 if i < 4 else 1e-4
        assert bool(((a - b).abs() <= step * b.abs() + tol * b.abs().max()).all()), i


@pytest.mark.parametrize("T,D", [(8192, 64), (4096, 32), (4096, 8), (4096, 128)])
def test_uncut_rows_as_accurate_as_short_splits(gpu_ca, T, D):
    """A row's output over n tiles in one split, against 12-tile splits.  Of the
    difference, at most half an ulp per rounding with random signs (rms 2^-24 /
    sqrt(3) of the running sum): one rounding per tile of a sum growing like
    the square root of the tiles (n / 2 in squares) and of Z, growing linearly
    (n / 3), and the split side's 12 tiles and merge of n / 12 partials (6 + n /
    24): 2^-24 sqrt(0.3 n + 2) of the output's norm, n <= T / 32."""
    q, k, v, rho, _ = make_inputs((1, 2, T, D), 17, 1.0, [0.1, -0.1])
    t = [x.cuda() for x in (q, k, v, rho)]
    out = []
    try:
        for tiles in (12, 1 << 20):
            gpu_ca.ops.set_split_override(tiles, 0, 0)
            with torch.no_grad():
                out.append(gpu_ca.continuum_attention(*t).double())
    finally:
        gpu_ca.ops.set_split_override()
    rows = slice(T // 2, T)
    err = float((out[1] - out[0])[:, :, rows].norm() / out[0][:, :, rows].norm())
    assert err <= 2.0 ** -24 * (0.3 * T / 32 + 2) ** 0.5, err
