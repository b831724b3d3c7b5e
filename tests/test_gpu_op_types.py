"""The operator in the tensors' own type and at any head dim (ca_fwd_op / ca_bwd_op).

16-bit tensors: the kernels read them as they are; on the same values the
output must be the fp32 operator's, rounded once, bit for bit, and the
gradients its gradients to one rounding.  Head dims without kernels of their
own run on zero-padded rows: checked against the float64 oracle at the edges
of each padding range, and against the next kernel dim's own operator.
"""
import numpy as np
import pytest
import torch

from oracle import ca_oracle as O
from test_gpu_parity import GRAD_TOL, OUT_TOL, make_inputs, rel, say

pytestmark = pytest.mark.gpu

HALF_ULP = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


def _typed(ca, q, k, v, rho, dy):
    t = [x.cuda().requires_grad_(True) for x in (q, k, v)]
    r = rho.cuda().requires_grad_(True)
    y = ca.continuum_attention(*t, r)
    return y.detach(), torch.autograd.grad(y, (*t, r), dy.cuda())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape", [(1, 1, 1, 64), (2, 3, 31, 8), (1, 2, 33, 16), (2, 1, 129, 32),
                                   (1, 4, 513, 64), (2, 2, 300, 128)])
def test_half_types_match_fp32_operator(gpu_ca, dtype, shape):
    say(f"[case] {shape} {dtype}")
    q, k, v, rho, dy = make_inputs(shape, 11, 1.0, [0.1 * h for h in range(shape[1])])
    q, k, v, dy = (x.to(dtype) for x in (q, k, v, dy))
    y, grads = _typed(gpu_ca, q, k, v, rho, dy)
    y32, g32 = _typed(gpu_ca, *(x.float() for x in (q, k, v)), rho, dy.float())
    assert y.dtype == dtype and all(g.dtype == dtype for g in grads[:3])
    assert torch.equal(y, y32.to(dtype))
    with torch.no_grad():  # no y kept: the same output
        assert torch.equal(gpu_ca.continuum_attention(q.cuda(), k.cuda(), v.cuda(), rho.cuda()), y)
    # fp32 rounding of a weight gradient dY.v - D, whose terms cancel where the
    # true gradient is 0 (a single key): 4 ulp of its terms, times |q| or |k|
    noise = 2.0 ** -22 * float(dy.float().norm(dim=-1).max() * v.float().norm(dim=-1).max()
                               * max(q.abs().max(), k.abs().max())) / shape[3] ** 0.5
    for a, b in zip(grads[:3], g32[:3]):
        # one rounding to the type, plus fp32 rounding of the two kernels' sums
        # (each at most ~2e-6 of the largest element, tests/test_gpu_parity.py)
        bound = HALF_ULP[dtype] * b.abs() + 5e-6 * b.abs().max() + noise
        assert bool(((a.float() - b).abs() <= bound).all())
    if shape[2] > 1:  # a single key has no gain gradient
        assert rel(grads[3].cpu(), g32[3].cpu()) < 1e-4


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_half_types_in_passes(gpu_ca, dtype):
    """Under a small workspace cap the 16-bit gradients are summed over the
    passes in fp32: each differs from the one-pass result by one rounding."""
    shape = (1, 3, 700, 64)
    q, k, v, rho, dy = make_inputs(shape, 5)
    q, k, v, dy = (x.to(dtype) for x in (q, k, v, dy))
    y, grads = _typed(gpu_ca, q, k, v, rho, dy)
    prev = gpu_ca.ops.workspace_cap()
    try:
        gpu_ca.ops.set_workspace_cap(4 << 20)
        y2, grads2 = _typed(gpu_ca, q, k, v, rho, dy)
    finally:
        gpu_ca.ops.set_workspace_cap(prev)
    for a, b in zip((y, *grads[:3]), (y2, *grads2[:3])):
        a, b = a.float(), b.float()
        assert bool(((a - b).abs() <= 2 * HALF_ULP[dtype] * b.abs() + 5e-6 * b.abs().max()).all())
    assert rel(grads2[3].cpu(), grads[3].cpu()) < 1e-5


@pytest.mark.parametrize("D,T,cap", [(1, 40, 0), (7, 65, 0), (9, 33, 0), (17, 130, 0), (31, 64, 0),
                                     (33, 97, 0), (65, 257, 0), (80, 513, 24 << 20), (127, 129, 0)])
def test_padded_head_dims_match_oracle(gpu_ca, D, T, cap):
    say(f"[case] D={D} T={T} cap={cap}")
    shape = (2, 2, T, D)
    q, k, v, rho, dy = make_inputs(shape, D, 1.0, [0.2, -0.1])
    prev = gpu_ca.ops.workspace_cap()
    try:
        if cap:
            gpu_ca.ops.set_workspace_cap(cap)
        y, grads = _typed(gpu_ca, q, k, v, rho, dy)
    finally:
        gpu_ca.ops.set_workspace_cap(prev)
    n = [x.numpy() for x in (q, k, v, rho)]
    assert rel(y.cpu(), O.ca_forward(*n)[0]) <= OUT_TOL
    for a, b in zip(grads, O.ca_backward(*n, dy.numpy())):
        assert rel(a.cpu(), b) <= GRAD_TOL
    # non-contiguous operands give the same results
    pad = [torch.cat([x, x], -1).cuda()[..., :D].requires_grad_(True) for x in (q, k, v)]
    assert torch.equal(gpu_ca.continuum_attention(*pad, rho.cuda()).detach(), y)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_padded_head_dim_equals_wider_operator(gpu_ca, dtype):
    """Padding by hand to the kernel dim, with the gain carrying the scale's
    sqrt(DP / D), is the same arithmetic."""
    T, D, DP = 200, 40, 64
    q, k, v, rho, dy = (x.to(dtype) if x.dim() == 4 else x for x in make_inputs((1, 2, T, D), 3))
    y, grads = _typed(gpu_ca, q, k, v, rho, dy)
    wide = [torch.nn.functional.pad(x, (0, DP - D)) for x in (q, k, v, dy)]
    gain = rho + 0.5 * float(np.log(DP / D))
    yw, gw = _typed(gpu_ca, *wide[:3], gain, wide[3])
    tol = 1e-6 if dtype == torch.float32 else 2 * HALF_ULP[dtype]
    assert rel(y.float().cpu(), yw[..., :D].float().cpu()) <= tol
    for a, b in zip(grads[:3], gw[:3]):
        assert rel(a.float().cpu(), b[..., :D].float().cpu()) <= max(tol, 1e-5)


@pytest.mark.parametrize("D,T", [(136, 70), (160, 33)])
def test_wide_head_dims_match_oracle(gpu_ca, D, T):
    """Head dims above 128: the query-tile structure over the weight kernels."""
    q, k, v, rho, dy = make_inputs((1, 2, T, D), D, 1.0, [0.2, -0.1])
    y, grads = _typed(gpu_ca, q, k, v, rho, dy)
    n = [x.numpy() for x in (q, k, v, rho)]
    assert rel(y.cpu(), O.ca_forward(*n)[0]) <= OUT_TOL
    for a, b in zip(grads, O.ca_backward(*n, dy.numpy())):
        assert rel(a.cpu(), b) <= GRAD_TOL


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape", [(3, 2, 300, 80), (1, 5, 201, 9)])
def test_padded_head_dims_in_sets(gpu_ca, dtype, shape):
    """Pads of everything above half of a lowered cap: sets of batches or heads
    one after another, each in one pass or (the smaller cap) several, and slices
    that start at odd addresses.  Each set is the operator on its slices, so the
    results differ by the order of the passes' sums alone."""
    B, H, T, D = shape
    q, k, v, rho, dy = make_inputs(shape, 21, 1.0, [0.1 * h for h in range(H)])
    q, k, v, dy = (x.to(dtype) for x in (q, k, v, dy))
    y, grads = _typed(gpu_ca, q, k, v, rho, dy)
    lib = gpu_ca.native.load()
    code = {torch.float32: 0, torch.bfloat16: 1, torch.float16: 2}[dtype]
    full = lib.ca_bwd_op_workspace_bytes(code, B, H, T, D)
    prev = gpu_ca.ops.workspace_cap()
    step = 0.0 if dtype == torch.float32 else 2 * HALF_ULP[dtype]
    for part in (2, 4):
        say(f"[case] {shape} {dtype} cap 1/{part} of {full}")
        try:
            gpu_ca.ops.set_workspace_cap(full // part)
            assert lib.ca_bwd_op_workspace_bytes(code, B, H, T, D) <= full // part
            y2, grads2 = _typed(gpu_ca, q, k, v, rho, dy)
        finally:
            gpu_ca.ops.set_workspace_cap(prev)
        for a, b in zip((y, *grads[:3]), (y2, *grads2[:3])):
            a, b = a.float(), b.float()
            assert bool(((a - b).abs() <= step * b.abs() + 5e-6 * b.abs().max()).all())
        assert rel(grads2[3].cpu(), grads[3].cpu()) < 1e-5
