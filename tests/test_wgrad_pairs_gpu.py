"""The 16-bit pair-list weight gradient at 128-wide tiles (implicit_precomputed_gemm.py:180-230):
pair counts around its 32-pair steps, the four waves' turns and the two-stage pipeline's lead,
against the float64 oracle."""
import numpy as np
import pytest
import torch

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("cin,cout", [(128, 128), (64, 128), (128, 64), (256, 128)])
@pytest.mark.parametrize("n", [1, 31, 33, 127, 129, 256, 385, 1023, 1025, 5000])
def test_wide_weight_gradient(device, dtype, cin, cout, n):
    """m exact products summed in fp32 in any order, rounded once to fp32."""
    from sparsetriton_amd.nn.functional.conv.funcs.implicit_precomputed_gemm import wgrad
    from sparsetriton_amd.nn.functional.conv.kmap import KernelMap
    rng = np.random.default_rng(n + cin)
    K = 3
    nbr = np.stack([rng.permutation(n) for _ in range(K)], 1).astype(np.int32)
    nbr[:, 1][rng.random(n) < 0.5] = -1
    nbr[:, 2] = -1  # an offset without pairs
    X = torch.as_tensor(rng.standard_normal((n, cin)), device=device).to(dtype)
    dY = torch.as_tensor(rng.standard_normal((n, cout)), device=device).to(dtype)
    km = KernelMap.from_neighbor_indices(torch.as_tensor(nbr, device=device), n)
    dW = wgrad(X, dY, km, torch.float32).double().cpu().numpy()
    Xd, Yd = X.double().cpu().numpy(), dY.double().cpu().numpy()
    ref, mag = O.wgrad_f64_blas(Xd, Yd, nbr, K), O.wgrad_f64_blas(np.abs(Xd), np.abs(Yd), nbr, K)
    assert np.all(np.abs(dW - ref) <= (n + 2) * 2.0 ** -24 * mag)
    assert not dW[2].any()
