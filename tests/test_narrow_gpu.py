"""Kernels of the layers with few channels, on random maps, against the float64 oracle: the fp32
weight gradient with whole-row loads (implicit_precomputed_gemm.py:180-230) and the gather-GEMM that keeps its
weights in LDS (implicit_precomputed_gemm.py:64-177)."""
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


def _tiled(nbr, n_in, device):
    """The tile plan of a (n_out, K) map, rows in the mask-sorted order."""
    from sparsetriton_amd.nn.functional.conv.kmap import TileMap, TilePlan
    n_out, K = nbr.shape
    W = (K + 31) // 32
    bits = np.zeros((n_out, W * 32), dtype=np.uint64)
    bits[:, :K] = nbr >= 0
    masks = (bits.reshape(n_out, W, 32) << np.arange(32, dtype=np.uint64)).sum(2).astype(np.uint32)
    m = torch.as_tensor(masks.view(np.int32), device=device)
    nbr_t = torch.as_tensor(np.ascontiguousarray(nbr.T), device=device)
    perm = TilePlan.build(n_out, K, m).perm
    return TileMap.build(nbr_t, n_out, 1, m, K, perm, n_out, n_in)


EPS = {torch.float32: 2.0 ** -24, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}  # unit roundoffs (24, 8, 11 bits)
GATHER = [
    # n_out, n_in, K, Kd, Nd, density
    (1, 3, 27, 4, 16, 1.0), (15, 20, 27, 16, 16, 0.5), (17, 20, 27, 32, 32, 0.2), (127, 90, 27, 8, 20, 0.3),
    (129, 200, 27, 16, 32, 0.9), (1000, 1300, 27, 20, 32, 0.15), (5000, 4000, 27, 12, 3, 0.2), (5000, 4000, 27, 32, 20, 0.2),
    (3000, 3000, 1, 32, 64, 0.9), (3000, 3000, 8, 64, 32, 0.3), (3000, 3000, 27, 64, 16, 0.1), (2000, 2500, 64, 16, 16, 0.1),
    (2000, 2500, 27, 16, 64, 0.2), (2000, 2500, 3, 24, 48, 0.4), (700, 700, 27, 40, 16, 0.3), (4000, 3000, 27, 32, 32, 0.0),
    (70000, 70000, 27, 16, 16, 0.1), (40000, 40000, 27, 4, 32, 0.2),
]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n_out,n_in,K,Kd,Nd,density", GATHER)
def test_narrow_gather(device, dtype, n_out, n_in, K, Kd, Nd, density):
    """The LDS-resident-weights gather-GEMM: row counts around its 16-row wave tiles and the plan's
    128-row tiles, offset counts, widths with padding on either side, both weight layouts (bitwise
    equal) and reversed offsets.  A sum of m exact products accumulated in fp32 and rounded once is off
    by at most (m + 2) 2^-24 of the sum of magnitudes and half a unit of the result; a split fp32
    product by 2^-15 of its magnitude."""
    from sparsetriton_amd.nn.functional.conv.funcs.implicit_precomputed_gemm import b_kn_ok, gather_gemm_tiled
    rng = np.random.default_rng(n_out + 31 * K + Kd + 7 * Nd)
    nbr = _map(rng, n_out, n_in, K, density)
    X = torch.as_tensor(rng.standard_normal((n_in, Kd)), device=device).to(dtype)
    W = torch.as_tensor(rng.standard_normal((K, Kd, Nd)), device=device).to(dtype)
    b = torch.as_tensor(rng.standard_normal(Nd), device=device).to(dtype)
    tiles = _tiled(nbr, n_in, device)
    if not b_kn_ok(X, n_out, K, Nd):  # (fp32: twice the LDS)
        assert dtype == torch.float32 and Kd > 16 and Nd >= 32
        pytest.skip("not built for fp32")
    y = gather_gemm_tiled(X, tiles, W, n_out, K, bias=b, b_kn=True)
    yt = gather_gemm_tiled(X, tiles, W.transpose(1, 2).contiguous(), n_out, K, bias=b)
    assert torch.equal(y, yt)
    yr = gather_gemm_tiled(X, tiles, W.flip(0).contiguous(), n_out, K, bias=b, reverse_k=True, b_kn=True)
    assert torch.equal(y, yr)
    Xd, Wd, bd = X.double().cpu().numpy(), W.double().cpu().numpy(), b.double().cpu().numpy()
    ref = O.fwd_f64_blas(Xd, Wd, nbr) + bd
    mag = O.fwd_f64_blas(np.abs(Xd), np.abs(Wd), nbr) + np.abs(bd)
    m = int((nbr >= 0).sum(1).max()) * Kd
    bound = ((m + 2) * 2.0 ** -24 + (2.0 ** -15 if dtype == torch.float32 else 0)) * mag + EPS[dtype] * np.abs(ref)
    assert np.all(np.abs(y.double().cpu().numpy() - ref) <= bound * 1.001 + 1e-30)


SAME_BITS = [(Kd, Nd, dt) for Kd, Nd in [(4, 16), (8, 20), (12, 32), (16, 16), (16, 64), (24, 16), (32, 32), (64, 16)]
             for dt in (torch.float32, torch.bfloat16, torch.float16) if dt != torch.float32 or Kd > 16]


@pytest.mark.parametrize("Kd,Nd,dtype", SAME_BITS)
@pytest.mark.parametrize("n,density", [(17, 0.9), (1500, 0.15), (3000, 0.6)])
def test_narrow_gather_sums_like_the_other_kernels(device, dtype, Kd, Nd, n, density):
    """Bit for bit the sums of the kernels that take rows off its alignment (a view that starts one
    element into its allocation): offsets in the tile's ascending order.  (fp32 up to 16 elements: the
    same terms in another fp32 order, bounded by test_narrow_gather.)"""
    from sparsetriton_amd.nn.functional.conv.funcs.implicit_precomputed_gemm import b_kn_ok, gather_gemm_tiled
    rng = np.random.default_rng(Kd + Nd + n)
    nbr = _map(rng, n, n, 27, density)
    tiles = _tiled(nbr, n, device)
    X = torch.as_tensor(rng.standard_normal((n, Kd)), device=device).to(dtype)
    Wt = torch.as_tensor(rng.standard_normal((27, Nd, Kd)), device=device).to(dtype)
    view = torch.zeros(n * Kd + 1, dtype=dtype, device=device)[1:].view(n, Kd).copy_(X)
    assert not b_kn_ok(view, n, 27, Nd)
    assert torch.equal(gather_gemm_tiled(X, tiles, Wt, n, 27), gather_gemm_tiled(view, tiles, Wt, n, 27))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("Kd,Nd", [(4, 16), (8, 32), (16, 20), (16, 32), (32, 32)])
def test_narrow_gather_contains_non_finite_weights(device, dtype, Kd, Nd):
    """An infinite weight slice reaches no row of a 16-row group without a source at its offset."""
    from sparsetriton_amd.nn.functional.conv.funcs.implicit_precomputed_gemm import gather_gemm_tiled
    rng = np.random.default_rng(Kd + Nd)
    n, K, k = 2000, 27, 13
    nbr = _map(rng, n, n, K, 0.3)
    nbr[rng.random(n) < 0.97, k] = -1  # few rows use offset k: whole groups lack it, their neighbours have it
    tiles = _tiled(nbr, n, device)
    perm = tiles.perm.cpu().numpy()[:n]
    has = np.add.reduceat(nbr[perm, k] >= 0, np.arange(0, n, 16)) > 0
    clean = torch.as_tensor(perm[~np.repeat(has, 16)[:n]].astype(np.int64))
    assert 16 <= len(clean) < n
    X = torch.as_tensor(rng.standard_normal((n, Kd)), device=device).to(dtype)
    W = torch.as_tensor(rng.standard_normal((K, Kd, Nd)), device=device).to(dtype)
    W[k] = 0.0
    y = gather_gemm_tiled(X, tiles, W, n, K, b_kn=True).cpu()
    W[k] = float("inf")
    y2 = gather_gemm_tiled(X, tiles, W, n, K, b_kn=True).cpu()
    assert torch.equal(y[clean], y2[clean])
    assert not torch.isfinite(y2[torch.as_tensor(nbr[:, k] >= 0)]).any()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("Kd,Nd", [(4, 16), (16, 20), (32, 32)])
def test_narrow_gather_takes_views_and_contains_non_finite_rows(device, dtype, Kd, Nd):
    """Rows that start 8 bytes (16-bit) into an allocation give the aligned rows' result; a source row
    with inf reaches only the outputs that pair it."""
    from sparsetriton_amd.nn.functional.conv.funcs.implicit_precomputed_gemm import gather_gemm_tiled
    rng = np.random.default_rng(Kd + Nd)
    n = n_in = 900
    K = 27
    nbr = _map(rng, n, n, K, 0.2)
    tiles = _tiled(nbr, n_in, device)
    X = torch.as_tensor(rng.standard_normal((n, Kd)), device=device).to(dtype)
    W = torch.as_tensor(rng.standard_normal((K, Kd, Nd)), device=device).to(dtype)
    y = gather_gemm_tiled(X, tiles, W, n, K, b_kn=True)
    buf = torch.zeros(n * Kd + 4, dtype=dtype, device=device)
    view = buf[4:].view(n, Kd)
    view.copy_(X)
    yv = gather_gemm_tiled(view, tiles, W.transpose(1, 2).contiguous(), n, K)
    assert torch.allclose(y.float(), yv.float(), rtol=2 * EPS[dtype], atol=1e-5)
    X[17, 1] = float("inf")
    hit = (nbr == 17).any(1)
    y2 = gather_gemm_tiled(X, tiles, W, n, K, b_kn=True)
    assert torch.equal(torch.isfinite(y2).all(1).cpu(), torch.as_tensor(~hit))
    assert torch.equal(y2[torch.as_tensor(~hit)], y[torch.as_tensor(~hit)])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("kw", [dict(Kd=6, Nd=16), dict(Kd=128, Nd=16), dict(Kd=16, Nd=65), dict(K=65), dict(Kd=64, Nd=64),
                                dict(Kd=32, n=262145), dict(Kd=64, n=131073)])
def test_narrow_gather_refuses_other_shapes(device, dtype, kw):
    """Host rule: shapes outside the kernel's ranges go to the other kernels."""
    from sparsetriton_amd import _lib
    a = {"K": 27, "Kd": 16, "Nd": 16, "n": 100}
    a.update(kw)
    args = (None, a["n"], a["n"], a["K"], a["Kd"], a["Nd"], _lib.compute_code(dtype))
    assert _lib.lib().st_gather_b_kn_ok(*args) == 0
    assert _lib.lib().st_gather_b_kn_ok(None, 100, 100, 27, 16, 16, _lib.compute_code(dtype)) == 1
    assert _lib.lib().st_gather_b_kn_ok(None, 1 << 27, 100, 27, 16, 16, _lib.compute_code(dtype)) == 0


# n_out, Kd, Nd, dtype: sizes at which a workgroup's waves are sixteen (weights over half a CU's LDS, above
# 32,768 rows) or take a second and third 16-row tile (above 16 rows for each of the resident waves)
SEVERAL = [
    (40003, 32, 32, torch.float32), (40003, 64, 32, torch.bfloat16), (65536, 64, 32, torch.float16),  # sixteen waves
    (70003, 32, 32, torch.float32), (131057, 32, 32, torch.float32), (70003, 16, 64, torch.float32),  # and two tiles
    (70003, 32, 32, torch.bfloat16), (100003, 16, 16, torch.float32), (140003, 4, 16, torch.bfloat16),  # two tiles
    (300001, 4, 16, torch.float32), (300001, 16, 16, torch.bfloat16), (131071, 64, 16, torch.float16)]  # three, two


def _mixed_map(rng, n, K):
    """Rows with no, few, some and all sources, in an order that mixes them."""
    nbr = np.stack([rng.permutation(n) for _ in range(K)], 1).astype(np.int32)
    nbr[rng.random((n, K)) >= rng.choice([0.0, 0.04, 0.3, 1.0], n, p=[0.1, 0.5, 0.3, 0.1])[:, None]] = -1
    return nbr


@pytest.mark.parametrize("n,Kd,Nd,dtype", SEVERAL)
@pytest.mark.parametrize("epilogue", [False, True])
def test_narrow_gather_several_tiles_a_wave(device, n, Kd, Nd, dtype, epilogue):
    """The loop over a wave's tiles (the next one's head loaded a tile ahead, its count two ahead) and the
    sixteen-wave form, plain and with a batch norm, a residual and ReLU in the store; rows from both
    ends and the middle of the tile order and at random against float64 (bound: test_narrow_gather's,
    through the affine map; its own roundings are four of the terms')."""
    from sparsetriton_amd.nn.functional.conv.funcs.implicit_precomputed_gemm import b_kn_ok, conv_forward, conv_forward_epilogue
    rng = np.random.default_rng(n + Kd + Nd)
    K = 27
    nbr = _mixed_map(rng, n, K)
    kmap = _kmap(nbr, n, device)
    X = torch.as_tensor(rng.standard_normal((n, Kd)), device=device).to(dtype)
    W = torch.as_tensor(rng.standard_normal((K, Kd, Nd)), device=device).to(dtype)
    assert b_kn_ok(X, n, K, Nd)
    mul, add, add_mag = np.ones(Nd), np.zeros(Nd), np.zeros(Nd)
    if epilogue:
        w, b, mean = (torch.as_tensor(rng.uniform(-1, 1, Nd).astype(np.float32), device=device) for _ in range(3))
        var = torch.as_tensor(rng.uniform(0.1, 2, Nd).astype(np.float32), device=device)
        R = torch.as_tensor(rng.standard_normal((n, Nd)), device=device).to(dtype)
        y = conv_forward_epilogue(X, W, kmap, None, None, None, R, True, bn=(w, b, mean, var, 1e-5))
        mul = (w.double() / torch.sqrt(var.double() + 1e-5)).cpu().numpy()
        b, mean = b.double().cpu().numpy(), mean.double().cpu().numpy()
        add, add_mag = b - mean * mul, np.abs(b) + np.abs(mean * mul)
    else:
        y = conv_forward(X, kmap, W)
    order = kmap.forward_tiles().perm.cpu().numpy()[:n]
    rows = np.r_[order[:300], order[n // 2 - 150:n // 2 + 150], order[-300:], rng.integers(0, n, 300)]
    Xd, Wd = X.double().cpu().numpy(), W.double().cpu().numpy()
    s, mag = O.fwd_f64_blas(Xd, Wd, nbr[rows]), O.fwd_f64_blas(np.abs(Xd), np.abs(Wd), nbr[rows])
    bound = ((K * Kd + 2) * 2.0 ** -24 + (2.0 ** -15 if dtype == torch.float32 else 0)) * mag
    ref = s * mul + add
    bound = bound * np.abs(mul) + (4 * 2.0 ** -24 * (np.abs(s * mul) + add_mag) if epilogue else 0)
    if epilogue:
        res = R[torch.as_tensor(rows)].double().cpu().numpy()
        ref = np.maximum(ref + res, 0)
        bound += 2.0 ** -24 * np.abs(res)
    got = y[torch.as_tensor(rows)].double().cpu().numpy()
    assert np.all(np.abs(got - ref) <= 1.001 * bound + EPS[dtype] * np.abs(ref) + 1e-30)
