"""``fovi_knnconv_dw`` over its channel tiles (128 or 256 output and input channels) and image
splits, against float64: dW[o, c V + v] = sum over images and (n, i) pairs of slot v of
dy[b, n, o] x[b, i, c]. Products of bf16 values are exact in fp32, so the error is that of the fp32
sums: below 1e-5 of the result's norm for the few thousand terms here."""
import pytest
import torch

from fovi_amd import _lib
from fovi_amd.arch.knn import KNNConvLayer
from fovi_amd.sensing.coords import SamplingCoords
from tests.helpers import assert_close_rel


def _dw64(layer, x, dy):
    b, c, n_in = x.shape
    idx, v = layer.knn_indices.t().cpu(), layer.ref_coords.shape[0]
    slots = layer.slots.cpu()
    dw = torch.zeros(dy.shape[1], c, v, dtype=torch.float64)
    for s in range(v):
        n, j = torch.nonzero((slots == s) & (idx < n_in), as_tuple=True)
        if len(n):
            dw[:, :, s] = torch.einsum("bop,bcp->oc", dy[:, :, n].double(), x[:, :, idx[n, j]].double())
    return dw.reshape(dy.shape[1], c * v)


@pytest.mark.gpu
@pytest.mark.parametrize("c_in,c_out", [(8, 8), (128, 128), (136, 128), (128, 136), (96, 256), (256, 104), (264, 136)])
def test_dw_tiles_and_splits_against_float64(c_in, c_out):
    coords = SamplingCoords(16, 0.5, 10, style="isotropic")
    layer = KNNConvLayer(c_in, c_out, 9, coords, coords, device="cuda", ref_frame_side_length=6)
    n, batch = coords.shape[0], 7
    g = torch.Generator().manual_seed(c_in + c_out)
    x = torch.randn(batch, n, c_in, generator=g).bfloat16()
    dy = torch.randn(batch, n, c_out, generator=g).bfloat16()
    ref = _dw64(layer, x.transpose(1, 2), dy.transpose(1, 2))
    xd, dyd = x.cuda().transpose(1, 2), dy.cuda().transpose(1, 2)
    for ipg in (None, 1, 3, 7):
        layer.dw_images_per_group = ipg
        got = layer._dw_fused(xd, dyd)
        assert_close_rel(got.double().cpu(), ref, 1e-5, f"images per group {ipg}")


def test_split_covers_the_batch_and_grows_with_many_slots():
    coords = SamplingCoords(16, 0.5, 10, style="isotropic")
    layer = KNNConvLayer(96, 256, 9, coords, coords, device="cpu", ref_frame_side_length=6)
    for batch in (1, 2, 63, 64, 1000):
        assert 1 <= layer._dw_split(batch, 36) <= batch
    assert layer._dw_split(1000, 36) > 1         # many images: several per workgroup
    wide = KNNConvLayer(256, 256, 25, SamplingCoords(16, 2.78, 64, style="logpolar"),
                        SamplingCoords(16, 2.78, 64, style="logpolar"), device="cpu")
    assert wide._dw_split(4, 25) == 1            # few images, long lists: one each


@pytest.mark.gpu
@pytest.mark.parametrize("n_ref,c_in,c_out", [(512, 40, 8), (16384, 16, 8), (16385, 24, 16), (41000, 8, 8)])
def test_dw_of_many_slots(n_ref, c_in, c_out):
    """Through the C entry: reduction blocks of 32, one and part of one channel's slots."""
    g = torch.Generator().manual_seed(n_ref)
    n_in, n_out, batch, n_pairs = 50, 60, 2, 4000
    v = torch.randint(0, n_ref, (n_pairs,), generator=g).sort().values
    v[0], v[-1] = 0, n_ref - 1
    n, i = torch.randint(0, n_out, (n_pairs,), generator=g), torch.randint(0, n_in, (n_pairs,), generator=g)
    off = torch.zeros(n_ref + 1, dtype=torch.int32)
    off[1:] = torch.bincount(v, minlength=n_ref).cumsum(0)
    x = torch.randn(batch, n_in, c_in, generator=g).bfloat16()
    dy = torch.randn(batch, n_out, c_out, generator=g).bfloat16()
    prod = torch.einsum("bpo,bpc->poc", dy[:, n].double(), x[:, i].double())
    want = torch.zeros(n_ref, c_out, c_in, dtype=torch.float64).index_add_(0, v, prod).permute(1, 2, 0)
    dev = [t.cuda() for t in (x, dy, off, torch.stack([n, i], 1).to(torch.int32).contiguous())]
    lib = _lib.load()
    nbytes = lib.fovi_knnconv_dw_workspace_bytes(batch, 2, 1, c_in, c_out, n_ref)
    ws = torch.empty(nbytes // 4, dtype=torch.float32, device="cuda")
    dw = torch.full((c_out, c_in, n_ref), float("nan"), device="cuda")
    a = _lib.KnnConvDwArgs()
    a.x, a.dy = dev[0].data_ptr(), dev[1].data_ptr()
    a.x_stride[:] = [n_in * c_in, 1, c_in]
    a.dy_stride[:] = [n_out * c_out, 1, c_out]
    a.batch, a.c_in, a.c_out, a.n_in, a.n_out, a.n_ref = batch, c_in, c_out, n_in, n_out, n_ref
    a.pair_off, a.pairs, a.n_chunks, a.images_per_group = dev[2].data_ptr(), dev[3].data_ptr(), 1, 2
    a.workspace, a.workspace_bytes, a.dw = ws.data_ptr(), nbytes, dw.data_ptr()
    _lib.check(lib.fovi_knnconv_dw(a, _lib.stream_handle(ws.device)), "fovi_knnconv_dw")
    assert_close_rel(dw.double().cpu(), want, 1e-5, f"{n_ref}")
