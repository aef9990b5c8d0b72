"""Which gather-GEMM kernel takes a layer, and the batch norm folded in its store."""
import numpy as np
import pytest
import torch

from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _layer(device, n, cin, cout, dtype, seed):
    from sparsetriton_amd import SparseTensor
    rng = np.random.default_rng(seed)
    S = max(8, int(round((n / 0.2) ** (1 / 3))))
    lin = np.sort(rng.choice(S ** 3, n, replace=False))
    c = np.stack([0 * lin, lin // S ** 2, lin // S % S, lin % S], 1).astype(np.int32)
    X = torch.as_tensor(rng.standard_normal((n, cin)), device=device).to(dtype)
    W = torch.as_tensor(rng.standard_normal((27, cin, cout)) / np.sqrt(27 * cin), device=device).to(dtype)
    sp = SparseTensor(X, torch.as_tensor(c, device=device), spatial_shape=(S, S, S), batch_size=1)
    nbr = O.exact_kmap(c, c, O.target_offsets(3, 1, 1, False), 1, (S, S, S))
    return sp, W, nbr, rng


@pytest.mark.parametrize("cin,cout,dtype", [(128, 128, torch.bfloat16), (64, 128, torch.float32), (128, 64, torch.float32)])
@pytest.mark.parametrize("n", [40960, 40961, 49152, 49153])
def test_wide_and_ring_gathers_meet(device, cin, cout, dtype, n):
    """The row counts where the wide kernel takes over from the ring kernels: both sides agree with
    float64 within the rounding of their sums, at the first and the last rows."""
    from sparsetriton_amd.nn.functional import sparse_conv3d
    sp, W, nbr, _ = _layer(device, n, cin, cout, dtype, 3)
    y = sparse_conv3d(sp, W, 3).F
    rows = np.r_[0:500, n - 500:n]
    ref = O.fwd_f64_blas(sp.F.double().cpu().numpy(), W.double().cpu().numpy(), nbr[rows])
    mag = O.fwd_f64_blas(sp.F.double().abs().cpu().numpy(), W.double().abs().cpu().numpy(), nbr[rows])
    u = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -24
    bound = (27 * cin * 2.0 ** -24 + (2.0 ** -15 if dtype == torch.float32 else 0)) * mag + u * np.abs(ref)
    assert np.all(np.abs(y[rows].double().cpu().numpy() - ref) <= 1.001 * bound)


@pytest.mark.parametrize("cin,cout,dtype", [(16, 16, torch.float32), (32, 20, torch.bfloat16), (64, 64, torch.float16),
                                            (64, 128, torch.float32), (128, 128, torch.bfloat16)])
@pytest.mark.parametrize("affine,residual", [(True, True), (False, False), (True, False)])
def test_batch_norm_folded_in_the_store(device, cin, cout, dtype, affine, residual):
    """sparse_conv3d_fused with the batch norm's own tensors equals the one folded on the caller's
    side to the rounding of the fold (two fp32 units of mul and add)."""
    from sparsetriton_amd.nn.functional import sparse_conv3d_fused
    sp, W, _, rng = _layer(device, 1500, cin, cout, dtype, cin + cout)

    def vec(lo, hi):
        return torch.as_tensor(rng.uniform(lo, hi, cout).astype(np.float32), device=device)
    w, b = (vec(0.5, 1.5), vec(-1, 1)) if affine else (None, None)
    mean, var, eps = vec(-1, 1), vec(0.01, 2), 1e-5
    bias = vec(-1, 1).to(dtype)
    res = torch.as_tensor(rng.standard_normal((1500, cout)), device=device).to(dtype) if residual else None
    with torch.no_grad():
        got = sparse_conv3d_fused(sp, W, 3, bias=bias, residual=res, relu=True, bn=(w, b, mean, var, eps)).F
        scale = torch.rsqrt(var + eps) * (w if affine else 1.0)
        shift = -mean * scale + (b if affine else 0.0)
        want = sparse_conv3d_fused(sp, W, 3, bias=bias, scale=scale, shift=shift, residual=res, relu=True).F
    u = {torch.float32: 2.0 ** -24, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    tol = 2 * u * want.float().abs() + 8 * 2.0 ** -24 * (want.float().abs() + 40)
    assert bool(((got.float() - want.float()).abs() <= tol).all())


@pytest.mark.parametrize("transposed", [False, True])
def test_transposed_map_after_an_inference_pass(device, transposed):
    """An inference pass leaves the transposed map out of the cached build; a training pass over the
    same coordinates builds it then, with the gradients of a build that had it."""
    from sparsetriton_amd import SparseTensor
    from sparsetriton_amd.nn.functional import sparse_conv3d
    sp, _, _, rng = _layer(device, 3000, 16, 16, torch.float32, 9)
    W = torch.as_tensor(rng.standard_normal((27, 16, 16)).astype(np.float32) / 20, device=device)
    kw = dict(kernel_size=3, stride=2, padding=1, transposed=transposed, submanifold=False)
    grads = []
    for infer_first in (False, True):
        x = sp.F.clone().requires_grad_(True)
        w = W.clone().requires_grad_(True)
        t = SparseTensor(x, sp.C, spatial_shape=sp.spatial_shape, batch_size=1)
        if infer_first:
            with torch.no_grad():
                sparse_conv3d(t, w, **kw)
            (_, km, _), = t._cache.neighbor_indices.values()
            assert km.invnbr is None
        y = sparse_conv3d(t, w, **kw).F
        g = torch.sin(torch.arange(y.numel(), device=device, dtype=torch.float32)).view_as(y)
        grads.append(torch.autograd.grad(y, [x, w], g))
    assert torch.equal(grads[0][0], grads[1][0]) and torch.equal(grads[0][1], grads[1][1])


@pytest.mark.parametrize("n,cin,cout,dtype", [
    (1500, 4, 16, torch.bfloat16), (1500, 16, 32, torch.float32), (1500, 32, 20, torch.float16),  # weights in LDS
    (1500, 64, 64, torch.bfloat16), (1500, 128, 128, torch.float32), (1500, 5, 7, torch.float32),  # ring, pipelined
    (49153, 128, 128, torch.bfloat16), (98305, 64, 128, torch.float32)])  # wide
@pytest.mark.parametrize("affine", [True, False])
def test_batch_norm_in_the_store_has_the_bits_of_folded(device, n, cin, cout, dtype, affine):
    """The batch norm's own tensors give bit for bit the output of the scale and shift that
    ``SparseBatchNorm.folded`` makes of them."""
    from sparsetriton_amd.nn import SparseBatchNorm
    from sparsetriton_amd.nn.functional import sparse_conv3d_fused
    sp, W, _, rng = _layer(device, n, cin, cout, dtype, cin + cout)
    bn = SparseBatchNorm(cout, eps=1e-3, affine=affine).to(device).eval()
    with torch.no_grad():
        for t in [bn.running_mean, bn.running_var] + list(bn.parameters()):
            t.copy_(torch.as_tensor(rng.uniform(0.05, 1.5, cout)))
        kw = dict(bias=torch.as_tensor(rng.standard_normal(cout), device=device).to(dtype),
                  residual=torch.as_tensor(rng.standard_normal((n, cout)), device=device).to(dtype), relu=True)
        got = sparse_conv3d_fused(sp, W, 3, bn=bn.running_affine(), **kw).F
        scale, shift = bn.folded()
        want = sparse_conv3d_fused(sp, W, 3, scale=scale, shift=shift, **kw).F
    assert torch.equal(got, want)


def test_wide_gather_contains_non_finite_weights(device):
    """An infinite weight slice reaches no row of a 64-row group (a wave's rows) without a source at its
    offset."""
    from sparsetriton_amd.nn.functional.conv.funcs.implicit_precomputed_gemm import gather_gemm_tiled
    from sparsetriton_amd.nn.functional.conv.kmap import TileMap, TilePlan
    rng = np.random.default_rng(2)
    n, K, k = 70001, 27, 13
    nbr = np.stack([rng.permutation(n) for _ in range(K)], 1).astype(np.int32)
    nbr[rng.random((n, K)) >= 0.2] = -1
    nbr[rng.random(n) < 0.9, k] = -1  # few rows use offset k
    masks = ((nbr >= 0).astype(np.uint64) << np.arange(K, dtype=np.uint64)).sum(1).astype(np.uint32)
    m = torch.as_tensor(masks.view(np.int32)[:, None].copy(), device=device)
    nbr_t = torch.as_tensor(np.ascontiguousarray(nbr.T), device=device)
    perm = TilePlan.build(n, K, m).perm
    tiles = TileMap.build(nbr_t, n, 1, m, K, perm, n, n)
    order = perm.cpu().numpy()[:n]
    has = np.add.reduceat(nbr[order, k] >= 0, np.arange(0, n, 64)) > 0
    clean = torch.as_tensor(order[~np.repeat(has, 64)[:n]].astype(np.int64))
    assert 64 <= len(clean) < n // 2
    X = torch.as_tensor(rng.standard_normal((n, 128)), device=device).bfloat16()
    Wt = torch.as_tensor(rng.standard_normal((K, 128, 128)), device=device).bfloat16()
    out = []
    for v in (0.0, float("inf")):
        Wt[k] = v
        out.append(gather_gemm_tiled(X, tiles, Wt, n, K).cpu())
    assert torch.equal(out[0][clean], out[1][clean])
    assert not torch.isfinite(out[1][torch.as_tensor(nbr[:, k] >= 0)]).any()


@pytest.mark.parametrize("cin,cout,dtype,last_ring", [
    (128, 128, torch.bfloat16, 49152), (128, 128, torch.float16, 49152), (64, 128, torch.float32, 98304),
    (128, 64, torch.float32, 40960)])
@pytest.mark.parametrize("beyond", [0, 1])
def test_wide_and_ring_gathers_meet_with_an_epilogue_and_reversed_offsets(device, cin, cout, dtype, last_ring, beyond):
    """The last row count of the ring kernels and the first of the wide ones: batch norm, residual and ReLU
    in the store against float64 at the first and last rows (the plain sum's bound through the affine
    map, and four fp32 roundings of its terms), and reversed offsets, bit for bit those of a reversed
    copy of the weights."""
    from sparsetriton_amd import _lib
    from sparsetriton_amd.nn.functional import sparse_conv3d_fused
    from sparsetriton_amd.nn.functional.conv.funcs.implicit_precomputed_gemm import gather_gemm_tiled, weight_prep
    n = last_ring + beyond
    sp, W, nbr, rng = _layer(device, n, cin, cout, dtype, 4)
    w, b, mean, var = (torch.as_tensor(rng.uniform(lo, 1.5, cout).astype(np.float32), device=device)
                       for lo in (-1.5, -1.5, -1.5, 0.1))
    R = torch.as_tensor(rng.standard_normal((n, cout)), device=device).to(dtype)
    with torch.no_grad():
        y = sparse_conv3d_fused(sp, W, 3, residual=R, relu=True, bn=(w, b, mean, var, 1e-5)).F
    w, b, mean, var = (t.double().cpu().numpy() for t in (w, b, mean, var))
    mul = w / np.sqrt(var + 1e-5)
    rows = np.r_[0:500, n - 500:n]
    Xd, Wd, res = sp.F.double().cpu().numpy(), W.double().cpu().numpy(), R[rows].double().cpu().numpy()
    s, mag = O.fwd_f64_blas(Xd, Wd, nbr[rows]), O.fwd_f64_blas(np.abs(Xd), np.abs(Wd), nbr[rows])
    ref = np.maximum(s * mul + (b - mean * mul) + res, 0)
    u = {torch.float32: 2.0 ** -24, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    bound = (27 * cin * 2.0 ** -24 + (2.0 ** -15 if dtype == torch.float32 else 0)) * mag * np.abs(mul) + u * np.abs(ref)
    bound += 4 * 2.0 ** -24 * (np.abs(s * mul) + np.abs(b) + np.abs(mean * mul) + np.abs(res))
    assert np.all(np.abs(y[rows].double().cpu().numpy() - ref) <= 1.001 * bound)
    (_, km, _), = sp._cache.neighbor_indices.values()
    assert km.symmetric
    Bt = weight_prep(W, _lib.W_TRANSPOSE)
    rev = gather_gemm_tiled(sp.F, km.forward_tiles(), Bt, n, 27, reverse_k=True)
    assert torch.equal(rev, gather_gemm_tiled(sp.F, km.forward_tiles(), Bt.flip(0).contiguous(), n, 27))


def test_batch_norm_in_the_store_at_extreme_variances(device):
    """Variances from subnormal to huge, zero and infinite (eps 0): the bits of ``folded``."""
    from sparsetriton_amd.nn import SparseBatchNorm
    from sparsetriton_amd.nn.functional import sparse_conv3d_fused
    n, C = 300, 64
    sp, W, _, rng = _layer(device, n, 16, C, torch.float32, 11)
    bn = SparseBatchNorm(C, eps=0.0, affine=False).to(device).eval()
    for round_ in range(40):
        var = (10.0 ** rng.uniform(-37, 38, C)).astype(np.float32)
        if round_ == 0:
            var[:4] = (0.0, np.inf, 1e-40, np.float32(2.0) ** -126)
        bn.running_var.copy_(torch.as_tensor(var))
        with torch.no_grad():
            got = sparse_conv3d_fused(sp, W, 3, bn=bn.running_affine()).F
            scale, shift = bn.folded()
            want = sparse_conv3d_fused(sp, W, 3, scale=scale, shift=shift).F
        assert torch.equal(torch.nan_to_num(got), torch.nan_to_num(want)) and torch.equal(got.isnan(), want.isnan())
