"""Zero-padded head dims against the query-tile path, which serves the other head
dims without kernels of their own: no larger an error from the float64 oracle,
and nothing that depends on keys a row does not see."""
import numpy as np
import pytest
import torch

from oracle import ca_oracle as O
from test_gpu_parity import make_inputs, say

pytestmark = pytest.mark.gpu


def _fused(ca, t, dy):
    leaves = [x.cuda().requires_grad_(True) for x in t]
    y = ca.continuum_attention(*leaves)
    return [y.detach(), *torch.autograd.grad(y, leaves, dy.cuda())]


def _rel2(a, b):
    a = a.double().cpu().numpy()
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


@pytest.mark.parametrize("D", [12, 20, 28, 48, 80])
@pytest.mark.parametrize("scale", [1.0, 4.0])
def test_no_less_accurate_than_query_tiles(gpu_ca, D, scale):
    """Mean error in norm over three seeds per output, 3% for the spread of these
    means (the gain gradient, a handful of cancelling sums, spreads more and is
    pinned elsewhere).  ``scale`` enlarges half the heads' keys."""
    say(f"[case] D={D} scale={scale}")
    err = np.zeros((2, 4))
    for seed in range(3):
        q, k, v, rho, dy = make_inputs((1, 4, 700, D), seed, 1.0, [0.1, -0.1, 0.0, 0.2])
        k[:, 2:] *= scale
        t = (q, k, v, rho)
        n = [x.numpy() for x in t]
        ref = [O.ca_forward(*n)[0], *O.ca_backward(*n, dy.numpy())]
        g = [x.cuda() for x in t]
        tiles = [gpu_ca.ops.tiled_forward(*g, 64), *gpu_ca.ops.tiled_backward(*g, dy.cuda(), 64)]
        for row, got in enumerate((_fused(gpu_ca, t, dy), tiles)):
            err[row] += [_rel2(a, b) / 3 for a, b in zip(got[:4], ref)]
    say(str(err))
    assert (err[0] <= 1.03 * err[1]).all(), err


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
def test_rows_do_not_depend_on_later_keys(gpu_ca, dtype):
    """A NaN in a key leaves the output and dQ of the rows before its 128-query
    group bit for bit as they are."""
    T, D, bad = 400, 40, 300
    q, k, v, rho, dy = make_inputs((1, 2, T, D), 8)
    q, k, v, dy = (x.to(dtype) for x in (q, k, v, dy))
    clean = _fused(gpu_ca, (q, k, v, rho), dy)
    k = k.clone()
    k[:, :, bad] = float("nan")
    got = _fused(gpu_ca, (q, k, v, rho), dy)
    for a, b in zip(got[:2], clean[:2]):
        assert torch.equal(a[:, :, :256], b[:, :, :256])
        assert bool(a[:, :, bad:].isnan().all())
