"""Calls under a default device other than the host: host tables and staging buffers are host memory
whatever ``torch.device`` context or ``torch.set_default_device`` says."""
import numpy as np
import pytest
import torch

from fovi_amd.arch import knn_tables as T
from fovi_amd.arch.knn import KNNConvLayer
from fovi_amd.sensing.coords import SamplingCoords
from fovi_amd.sensing.samplers import GridSampler

_SIZE = np.array([[64, 64]] * 3)


def test_host_tables_stay_on_the_host():
    coords = SamplingCoords(16, 2.78, 8, style="logpolar")
    layer = KNNConvLayer(2, 2, 9, coords, coords, device="cpu")
    tables = lambda: T.image_row_tables(layer.slot_ptr, layer.nbr_sorted, layer.slot_order, layer._point_order(), 4)
    want = tables()
    with torch.device("meta"):
        got = tables()
    assert all(torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.gpu
def test_calls_under_a_cuda_default_device():
    sampler = GridSampler(16, 2.78, 16, device="cuda", mode="bilinear", style="logpolar")
    coords = SamplingCoords(16, 2.78, 16, style="logpolar")
    g = torch.Generator().manual_seed(2)
    img, fix = torch.randn(3, 3, 64, 64, generator=g).cuda(), torch.rand(3, 2, generator=g)
    want = sampler.sample_views(img, fix, _SIZE)
    x = torch.randn(9, 256, 32, generator=g).cuda().transpose(1, 2)
    few = torch.randn(9, 256, 3, generator=g).cuda().transpose(1, 2)

    def grads():
        torch.manual_seed(3)
        out = []
        for c, xin, dt in ((32, x, torch.float32), (3, few, torch.bfloat16)):
            layer = layers[c]
            xg = xin.detach().requires_grad_(True)
            with torch.autocast("cuda", dtype=torch.bfloat16, enabled=dt == torch.bfloat16):
                y = layer(xg)
            layer.weight.grad = None
            y.backward(torch.ones(y.shape, dtype=y.dtype, device="cuda"))
            out += [y.detach(), xg.grad, layer.weight.grad]
        return out

    layers = {c: KNNConvLayer(c, 48, 9, coords, coords, device="cuda") for c in (32, 3)}
    with torch.device("cuda"):
        assert torch.equal(sampler.sample_views(img, fix, _SIZE), want)
        assert torch.equal(sampler(img, fix_loc=fix, fixation_size=_SIZE), want)
        got = grads()          # the first calls: packing, transposed layers, pair lists
    assert all(torch.equal(a, b) for a, b in zip(got, grads()))
