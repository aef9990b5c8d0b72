"""Kernels of the layers with few channels, on random maps, against the float64 oracle: the fp32
weight gradient with whole-row loads (implicit_precomputed_gemm.py:180-230)."""
import numpy as np
import pytest
import torch

from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _map(rng, n_out, n_in, K, density):
    """(n_out, K) random map in which an input row feeds at most one output per offset."""
    nbr = np.stack([rng.permutation(max(n_in, n_out))[:n_out] for _ in range(K)], 1).astype(np.int32)
    nbr[(nbr >= n_in) | (rng.random((n_out, K)) >= density)] = -1
    return nbr


def _kmap(nbr, n_in, device):
    from sparsetriton_amd.nn.functional.conv.kmap import KernelMap
    return KernelMap.from_neighbor_indices(torch.as_tensor(nbr, device=device), n_in)


@pytest.mark.parametrize("cin,cout", [(4, 16), (16, 16), (20, 36), (16, 32), (32, 32), (12, 4), (64, 16), (32, 64), (48, 80),
                                      (64, 64), (128, 20), (3, 32), (16, 5)])
@pytest.mark.parametrize("n,density", [(1, 1.0), (33, 0.9), (1000, 0.3), (5000, 0.6), (300, 0.0)])
def test_f32_weight_gradient_rows(device, cin, cout, n, density):
    """Channel tiles of 16, 32 and 64 with remainders (and odd counts, which take the element-wise
    kernel); pair counts around the 32-pair steps and the chunk size.  IEEE mode keeps 64 x 64 on
    the same fp32 kernel.  Any order of an fp32 sum of m products is off by at most m 2^-24 times
    the sum of their magnitudes (and the products' own rounding)."""
    from sparsetriton_amd.config import set_fp32_precision
    from sparsetriton_amd.nn.functional.conv.funcs.implicit_precomputed_gemm import wgrad
    set_fp32_precision("ieee")
    rng = np.random.default_rng(cin * 1000 + cout + n)
    K, n_in = 3, n + 7
    nbr = _map(rng, n, n_in, K, density)
    X = rng.standard_normal((n_in, cin)).astype(np.float32)
    dY = rng.standard_normal((n, cout)).astype(np.float32)
    dW = wgrad(torch.as_tensor(X, device=device), torch.as_tensor(dY, device=device), _kmap(nbr, n_in, device),
               torch.float32).double().cpu().numpy()
    ref, mag = O.wgrad_f64_blas(X, dY, nbr, K), O.wgrad_f64_blas(np.abs(X), np.abs(dY), nbr, K)
    pairs = int((nbr >= 0).sum(0).max())
    assert np.all(np.abs(dW - ref) <= (pairs + 2) * 2.0 ** -24 * mag)


def test_f32_weight_gradient_rows_non_finite(device):
    """A non-finite row reaches only the offsets that pair it, and only its own channels."""
    from sparsetriton_amd.config import set_fp32_precision
    from sparsetriton_amd.nn.functional.conv.funcs.implicit_precomputed_gemm import wgrad
    set_fp32_precision("ieee")
    rng = np.random.default_rng(5)
    nbr = _map(rng, 200, 200, 3, 0.5)
    X = rng.standard_normal((200, 16)).astype(np.float32)
    dY = rng.standard_normal((200, 20)).astype(np.float32)
    row = int(nbr[nbr[:, 1] >= 0, 1][0])
    nbr[(nbr == row) & (np.arange(3) != 1)[None, :]] = -1
    X[row, 5] = np.inf
    dW = wgrad(torch.as_tensor(X, device=device), torch.as_tensor(dY, device=device), _kmap(nbr, 200, device),
               torch.float32).cpu().numpy()
    assert np.isfinite(dW[[0, 2]]).all() and np.isfinite(np.delete(dW[1], 5, axis=0)).all()
    assert not np.isfinite(dW[1, 5]).any()
