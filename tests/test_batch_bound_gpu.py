"""Layers on new coordinates hold their batch indices against the tensor's batch size in every pass
(the constructor's check, tensor.py:55-138), whatever was assigned or written since the tensor was made."""
import numpy as np
import pytest
import torch

from sparsetriton_amd import SparseTensor, _lib
from sparsetriton_amd.config import ConvAlgo, set_conv_algo
from sparsetriton_amd.utils.hash import HostWords
from sparsetriton_amd.nn.functional import sparse_conv3d, sparse_pooling, sparse_upsample

pytestmark = pytest.mark.gpu


def _tensor(device, n=600, S=16):
    lin = torch.randperm(2 * S ** 3, generator=torch.Generator().manual_seed(1))[:n].sort().values
    c = torch.stack([lin // S ** 3, lin // S ** 2 % S, lin // S % S, lin % S], 1)
    return SparseTensor(torch.ones((n, 16), device=device), c.to(device), spatial_shape=(S, S, S), batch_size=2)


def _conv(transposed, algo):
    def run(t):
        set_conv_algo(algo)
        try:
            w = torch.ones((27, 16, 8), device=t.F.device)
            return sparse_conv3d(t, w, 3, stride=2, padding=1, transposed=transposed, submanifold=False)
        finally:
            set_conv_algo(ConvAlgo.PrecomputedNeighborGEMM)
    return run


MAP, FLY = ConvAlgo.PrecomputedNeighborGEMM, ConvAlgo.ImplicitHashFlyGEMM
LAYERS = {"strided": _conv(False, MAP), "transposed": _conv(True, MAP), "strided_fly": _conv(False, FLY),
          "pool": lambda t: sparse_pooling(t, 2, 0, 2, "max"), "upsample": lambda t: sparse_upsample(t, 2)}


@pytest.mark.parametrize("layer", LAYERS)
@pytest.mark.parametrize("how", ["batch_size", "batch_size_after_a_pass", "data", "in_place", "assigned", "replaced"])
def test_a_batch_index_beyond_the_batch_is_refused(device, layer, how):
    run = LAYERS[layer]
    t = _tensor(device)
    if how == "batch_size_after_a_pass":  # the coordinates' maps are cached
        assert run(t).batch_size == 2
    if how.startswith("batch_size"):
        t.batch_size = 1
    elif how == "data":
        t.C.data[-1, 0] = 7
    elif how == "in_place":
        t.C[-1, 0] = 7
    elif how == "assigned":
        c = t.C.clone()
        c[-1, 0] = 7
        t.C = c
    else:
        t.C.data[-1, 0] = 7
        t = t.replace(t.F)
    with pytest.raises(AssertionError, match="must be > max batch index"):
        run(t)


@pytest.mark.parametrize("layer", LAYERS)
def test_coordinates_within_the_batch_are_taken(device, layer):
    run = LAYERS[layer]
    t = _tensor(device)
    first, again = run(t), run(t)
    assert torch.equal(first.C, again.C) and torch.equal(first.F, again.F) and again.batch_size == 2
    t.batch_size = 5
    wide = run(t)
    assert wide.batch_size == 5 and torch.equal(first.C, wide.C)
    empty = SparseTensor(t.F[:0], t.C[:0], spatial_shape=(16, 16, 16), batch_size=2)
    assert run(empty).F.shape[0] == 0


@pytest.mark.parametrize("dtype", [torch.int16, torch.int32, torch.int64])
@pytest.mark.parametrize("n", [0, 1, 63, 257, 100003])
def test_batch_index_max(device, dtype, n):
    rng = np.random.default_rng(n)
    c = torch.as_tensor(rng.integers(-9, 30000, (n, 4)), dtype=dtype, device=device)
    c[:, 1:] = 32000
    parts = torch.empty((64,), dtype=torch.int32, device=device)
    _lib.call("st_batch_index_max", _lib.ptr(c), _lib.coord_code(dtype), n, _lib.ptr(parts), 64, _lib.stream_of(c.device))
    want = int(c[:, 0].max()) if n else -2 ** 31
    assert int(parts.max()) == want
    host = HostWords(64, c.device, lambda ptr: _lib.call("st_batch_index_max", _lib.ptr(c), _lib.coord_code(dtype), n,
                                                         ptr, 64, _lib.stream_of(c.device)))
    assert max(host.values()) == want == max(host.values())


def test_layers_over_cached_maps_can_be_captured(device):
    """A graph takes a strided convolution over a cached map and an upsampling (the eager pass before it
    checked their batch indices); every replay equals the eager result."""
    t = _tensor(device)
    w = torch.ones((27, 16, 8), device=device)
    x = torch.randn_like(t.F)

    def run():
        with torch.no_grad():
            y = sparse_conv3d(t.replace(x), w, 3, stride=2, padding=1, submanifold=False)
            return sparse_upsample(y, 2).F
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        run()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = run()
    for seed in range(3):
        x.copy_(torch.randn(x.shape, generator=torch.Generator().manual_seed(seed)))
        want = run()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
