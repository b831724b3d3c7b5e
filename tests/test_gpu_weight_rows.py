"""The weight row kernels at the edges of their row lengths (rows of at most 64
keys and past 2048 on the three-pass kernel, 256-key register chunks between,
16-byte and 4-byte accesses) against the float64 oracle."""
import numpy as np
import pytest
import torch

from oracle import ca_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [1, 4, 64, 65, 68, 255, 256, 257, 508, 513, 1024, 1025, 2047, 2048, 2049])
@pytest.mark.parametrize("misaligned", [False, True])
def test_rows_match_oracle(gpu_ca, K, misaligned):
    """The last queries of a K-key row, an early and a middle one, with a large
    common offset in the weight gradients (removed by their centring)."""
    rng = np.random.default_rng(K)
    for start, Q in {(K - min(K, 3), min(K, 3)), (0, 1), (K // 2, 1)}:
        s = (2.5 * rng.standard_normal((2, Q, K))).astype(np.float32)
        gw = (rng.standard_normal((2, Q, K)) + 3.0).astype(np.float32)
        s[:, :, start + Q:] = np.inf  # keys no query sees are not read into any result

        def dev(a):
            if not misaligned:
                return torch.from_numpy(a).cuda()
            buf = torch.empty(a.size + 1, device="cuda")  # rows off 16-byte alignment
            buf[1:] = torch.from_numpy(a.reshape(-1)).cuda()
            return buf[1:].view(a.shape)

        sd, gd = dev(s), dev(gw)
        W, stats = gpu_ca.ca_weights(sd, start)
        W2, ds = gpu_ca.ca_weights_backward(sd, gd, start, return_weights=True)
        assert torch.equal(ds, gpu_ca.ca_weights_backward(sd, gd, start))
        q = np.arange(start, start + Q)
        for b in range(2):
            sv = np.where(np.arange(K)[None, :] <= q[:, None], s[b], 0.0).astype(np.float64)
            w0 = O.ca_weights(sv, q)[0]
            d0 = O.ca_weights_vjp(sv, gw[b].astype(np.float64), qidx=q)
            # float32 segment terms (about 5e-7 of their scale, tests/test_device_math.py)
            # summed over a row
            for got in (W[b], W2[b]):
                np.testing.assert_allclose(got.cpu().numpy(), w0, rtol=2e-5, atol=2e-6)
            d0 = d0[0] if isinstance(d0, tuple) else d0
            np.testing.assert_allclose(ds[b].cpu().numpy(), d0, rtol=0,
                                       atol=3e-5 * max(np.abs(d0).max(), np.abs(w0).max()))
        assert bool((W[:, :, start + Q:] == 0).all()) and bool((ds[:, :, start + Q:] == 0).all())
