"""kNN pooling on channel planes (unit point stride): the planes kernels give the bits of the
any-stride kernels, which tests/test_knnpool.py checks against the oracle. A view with point
stride 2 of the same values takes the latter."""
import pytest
import torch

from fovi_amd import _lib
from fovi_amd.arch.knn import KNNPoolingLayer
from fovi_amd.sensing.coords import SamplingCoords


@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["max", "avg", "sum", "gaussian"])
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("res_in,res_out,k,c,batch", [
    (12, 8, 9, 8, 3),       # one group of channels, pad ring
    (12, 5, 16, 13, 2),     # an odd number of channels, the longest list
    (7, 4, 1, 40, 5),       # one neighbour, fewer points than a wave
    (20, 16, 9, 24, 2),     # more than 256 input points
])
def test_planes_equal_the_any_stride_kernels(mode, dt, res_in, res_out, k, c, batch):
    ci = SamplingCoords(16, 0.5, res_in, style="isotropic")
    co = SamplingCoords(16, 0.5, res_out, style="isotropic")
    layer = KNNPoolingLayer(k, ci, co, mode=mode, device="cuda")
    n_in, n_out = ci.shape[0], co.shape[0]
    assert n_out >= 16
    g = torch.Generator().manual_seed(c)
    x = torch.randn(batch, c, n_in, generator=g).to(dt)
    x = torch.where(torch.rand(x.shape, generator=g) < 0.1, torch.full_like(x, float("nan")), x)
    x = torch.where(torch.rand(x.shape, generator=g) < 0.1, torch.full_like(x, 0.5), x)      # ties
    x = torch.where(torch.rand(x.shape, generator=g) < 0.02, torch.full_like(x, float("-inf")), x).cuda()
    strided = torch.empty(batch, c, n_in, 2, dtype=dt, device="cuda")[..., 0]
    strided.copy_(x)
    got, want = layer(x), layer(strided)
    assert got.stride(2) == 1 and strided.stride(2) == 2
    assert torch.equal(got.nan_to_num(7.0), want.nan_to_num(7.0)) and torch.equal(got.isnan(), want.isnan())
    dy = torch.randn(batch, c, n_out, generator=g).to(got.dtype).cuda()
    # the any-stride gradient: dx of a strided x is laid out as planes, so force its kernel with
    # channels-last x and dx (point stride c)
    rows = x.transpose(1, 2).contiguous().transpose(1, 2)
    ref = layer._backward(rows, dy)
    assert ref.stride(1) == 1 and ref.stride(2) == c
    for d in (dy, dy.transpose(1, 2).contiguous().transpose(1, 2)):
        dx = layer._backward(x, d)
        assert dx.stride(2) == 1
        assert torch.equal(dx.nan_to_num(7.0), ref.nan_to_num(7.0)) and torch.equal(dx.isnan(), ref.isnan())


@pytest.mark.gpu
@pytest.mark.parametrize("mode,want", [(_lib.POOL_MAX, float("-inf")), (_lib.POOL_AVG, float("nan")),
                                       (_lib.POOL_SUM, 0.0), (_lib.POOL_GAUSSIAN, 0.0)])
def test_no_input_point_reads_nothing(mode, want):
    """Every neighbour is a pad token and there is no input 0 to read in its place: the kernels that
    look at the index first take it."""
    x, y = torch.zeros(1, device="cuda"), torch.full((2, 3, 20), 5.0, device="cuda")
    nbr = torch.zeros(20, 4, dtype=torch.int32, device="cuda")
    w = torch.ones(20, 4, device="cuda")
    a = _lib.KnnPoolArgs()
    a.x, a.x_dtype, a.y, a.y_dtype = x.data_ptr(), _lib.F32, y.data_ptr(), _lib.F32
    a.batch, a.channels, a.n_in, a.n_out, a.k = 2, 3, 0, 20, 4
    a.x_stride[:], a.y_stride[:] = [0, 0, 1], [60, 20, 1]
    a.nbr, a.weights, a.mode = nbr.data_ptr(), w.data_ptr(), mode
    _lib.check(_lib.load().fovi_knnpool_fwd(a, _lib.stream_handle(y.device)), "fovi_knnpool_fwd")
    assert torch.equal(y.nan_to_num(7.0), torch.full_like(y, want).nan_to_num(7.0))
