"""Image-row kernel (``knnconv_img.hip``) on points without a neighbour: inputs that no output reads (a
strided layer's input gradient) and all -1 columns (an empty group of a partition). A group of such
points visits no slot; its outputs are the bias, and nobody else's are touched."""
import pytest
import torch

from fovi_amd import _lib
from fovi_amd.arch import knn_tables as T
from fovi_amd.arch.knn import KNNConvLayer, _TransposedKnnConv, get_in_out_coords
from fovi_amd.sensing.coords import SamplingCoords
from oracle import knnconv_ref
from tests.helpers import assert_close_rel


def _strided(style, res, stride, k, c_in, c_out, device):
    cin, cout, _ = get_in_out_coords(res, 16, 2.78 if style == "logpolar" else 0.5, stride, style=style,
                                     auto_match_cart_resources=0, device=device)
    layer = KNNConvLayer(c_in, c_out, k, cin, cout, device=device)
    g = torch.Generator().manual_seed(1)
    with torch.no_grad():
        layer.weight.copy_(torch.randn(layer.weight.shape, generator=g) * (1.0 / (c_in * layer._k)) ** 0.5)
    return layer


def _unread(layer):
    read = torch.zeros(layer.in_coords.shape[0] + 1, dtype=torch.bool)
    read[layer.knn_indices_pad_token.cpu().flatten()] = True
    return ~read[:-1]


def _empty_groups(layer, batch):
    """Groups of the plan for ``batch`` images that visit no slot."""
    _, (rb, ib, _) = layer._image_plan(batch)
    _, points, nact = T.image_row_tables(layer.slot_ptr, layer.nbr_sorted, layer.slot_order, layer._point_order(),
                                         rb * 32 // ib)
    used = (layer.slot_ptr.cpu() & 0xFFFF).sum(1) > 0
    for g in torch.nonzero(nact == 0).flatten().tolist():
        pts = points[g][points[g] >= 0].long()
        assert len(pts) and not used[pts].any()
    return int((nact == 0).sum())


_STRIDED = [("logpolar", 32, 4, 9), ("logpolar", 13, 2, 9), ("isotropic", 32, 4, 9)]


@pytest.mark.parametrize("style,res,stride,k", _STRIDED)
def test_strided_layers_have_groups_without_a_slot(style, res, stride, k):
    layer = _strided(style, res, stride, k, 96, 64, "cpu")
    t = _TransposedKnnConv(layer, torch.device("cpu"))
    assert int(_unread(layer).sum()) > 0
    assert sum(_empty_groups(t, b) for b in (8, 32, 128)) > 0


@pytest.mark.gpu
@pytest.mark.parametrize("style,res,stride,k", _STRIDED)
@pytest.mark.parametrize("batch", [8, 32, 128])
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_input_gradient_of_inputs_nothing_reads(style, res, stride, k, batch, dt):
    """96 input channels: three waves of a dx workgroup own columns, and only the first writes the
    group's points."""
    layer = _strided(style, res, stride, k, 96, 64, "cuda")
    g = torch.Generator().manual_seed(2)
    x = torch.randn(batch, layer.in_coords.shape[0], 96, generator=g).to(dt)
    dy = torch.randn(batch, 64, layer.out_coords.shape[0], generator=g).to(dt)
    xg = x.cuda().transpose(1, 2).requires_grad_(True)
    layer(xg).backward(dy.cuda())
    t = layer._transposed_conv
    assert t.last_weight_layout == "image"
    unread = _unread(layer)
    assert torch.equal(xg.grad.cpu()[:, :, unread], torch.zeros(batch, 96, int(unread.sum()), dtype=dt))
    w = layer.weight.detach().cpu()
    xr = x.float().transpose(1, 2).requires_grad_(True)
    knnconv_ref.knnconv_forward(xr, layer.knn_indices.cpu(), layer.in_coords.shape[0], layer.local_rf.cpu(),
                                w if dt == torch.float32 else w.bfloat16().float()).backward(dy.float())
    assert_close_rel(xg.grad.float().cpu(), xr.grad, 1e-5 if dt == torch.float32 else 1e-2, f"{batch}")


def _with_empty_columns(device, c_in, c_out):
    """16 x 16 points, nine neighbours; every third column and a run of 100 all -1."""
    coords = SamplingCoords(16, 2.78, 16, style="logpolar")
    whole = KNNConvLayer(c_in, c_out, 9, coords, coords, device="cpu")
    idx = whole.knn_indices.clone()
    empty = torch.zeros(256, dtype=torch.bool)
    empty[::3] = True
    empty[100:200] = True
    idx[:, empty] = -1
    layer = KNNConvLayer.from_tables(c_in, c_out, coords, coords, idx, slots=whole.slots, device=device, bias=True)
    g = torch.Generator().manual_seed(3)
    with torch.no_grad():
        layer.weight.copy_(torch.randn(layer.weight.shape, generator=g) * (1.0 / (c_in * 9)) ** 0.5)
        layer.bias.copy_(torch.randn(c_out, generator=g))
    return layer, empty


@pytest.mark.gpu
@pytest.mark.parametrize("batch", [8, 17, 130])
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16, torch.float8_e4m3fn])
def test_all_minus_one_columns_give_the_bias(batch, dt):
    layer, empty = _with_empty_columns("cuda", 64, 320)
    x = torch.randn(batch, 256, 64, generator=torch.Generator().manual_seed(4))
    x = (x if dt == torch.float32 else x.bfloat16()).cuda().transpose(1, 2)
    fp8 = dt == torch.float8_e4m3fn
    xq = layer.quantize_input(x) if fp8 else x
    seen = 0
    with torch.no_grad():
        for plan in (None, (4, 128, 2), (4, 16, 1), (2, 32, 2), (1, 16, 1)):
            if plan is not None:
                layer._img.plans[batch] = (0.0, plan)
            seen += _empty_groups(layer, batch)
            y = layer(xq)
            assert layer.last_weight_layout == "image"
            bias = layer.bias.detach().to(y.dtype).cpu()
            assert torch.equal(y.cpu()[:, :, empty], bias.view(1, -1, 1).expand(batch, -1, int(empty.sum())))
            layer.image_rows = False
            want = layer(xq)
            layer.image_rows = True
            assert_close_rel(y.float().cpu(), want.float().cpu(), 1e-5 if dt == torch.float32 else 1e-2, f"{plan}")
    assert seen > 0
    path = {torch.float32: "f32", torch.bfloat16: "bf16"}.get(dt, "fp8")
    layer(xq)
    assert _lib.knnconv_last_path() == f"{path} image rows"
