"""``fovi_knnconv_dw_few``: the weight gradient of layers with at most 8 input channels from a bf16
output gradient, against float64 over the same operands. The products are exact in fp32 (fp32 x
enters as three bf16 parts that add up to it), so the error is that of fp32 sums: below 1e-5 of
the result's norm for the few thousand terms here."""
import pytest
import torch

from fovi_amd import _lib
from fovi_amd.arch.knn import KNNConvLayer
from fovi_amd.sensing.coords import SamplingCoords
from tests.helpers import assert_close_rel
from tests.test_dw_tiles import _dw64


def _layer(res_in, res_out, k, c_in, c_out, side, device="cuda"):
    return KNNConvLayer(c_in, c_out, k, SamplingCoords(16, 0.5, res_in, style="isotropic"),
                        SamplingCoords(16, 0.5, res_out, style="isotropic"), device=device, ref_frame_side_length=side)


_SHAPES = [
    (12, 6, 25, 3, 96, 10, 16),      # V = 100, pad ring, one tile of 96 rows
    (10, 8, 9, 1, 33, None, 5),      # one channel (32 slots per block, V = 9), images padded to 16
    (8, 8, 30, 4, 128, 3, 33),       # several neighbours per slot, two tiles of 64 rows
    (8, 5, 16, 5, 8, 7, 17),         # 30 of 32 columns used
    (6, 3, 4, 8, 200, None, 1),      # one image, three row tiles
]


@pytest.mark.gpu
@pytest.mark.parametrize("res_in,res_out,k,c_in,c_out,side,batch", _SHAPES)
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("layout", ["planes", "rows"])
def test_dw_few_against_float64(res_in, res_out, k, c_in, c_out, side, batch, dt, layout):
    layer = _layer(res_in, res_out, k, c_in, c_out, side)
    g = torch.Generator().manual_seed(c_in)
    x = torch.randn(batch, c_in, layer.in_coords.shape[0], generator=g).to(dt)
    dy = torch.randn(batch, c_out, layer.out_coords.shape[0], generator=g).bfloat16()
    rows = lambda t: t.transpose(1, 2).contiguous().transpose(1, 2) if layout == "rows" else t
    got = layer._dw_few(rows(x.cuda()), rows(dy.cuda()))
    assert_close_rel(got.double().cpu(), _dw64(layer, x, dy), 1e-5, f"{dt} {layout}")


@pytest.mark.gpu
def test_dw_few_is_as_exact_as_the_fp32_path():
    """fp32 x over six orders of magnitude: no further from float64 than the slot sums and the fp32
    GEMM it replaces (both rounded sums of the same products; twice for the difference of their
    orders)."""
    layer = _layer(16, 8, 49, 3, 64, 14)
    g = torch.Generator().manual_seed(5)
    x = torch.randn(64, 3, layer.in_coords.shape[0], generator=g)
    x = x * torch.pow(10.0, 6 * torch.rand(x.shape, generator=g) - 3)
    dy = torch.randn(64, 64, layer.out_coords.shape[0], generator=g).bfloat16()
    ref = _dw64(layer, x, dy)
    got = layer._dw_few(x.cuda(), dy.cuda())
    layer.dw_fused = False
    _, old = layer._backward(x.cuda(), layer.weight, dy.cuda(), False, True)
    e = [float((t.double().cpu() - ref).norm() / ref.norm()) for t in (got, old)]
    assert e[0] <= 2 * e[1] and e[0] < 1e-6, e


@pytest.mark.gpu
def test_autocast_training_step_takes_it_and_non_finite_gradients_show():
    layer = _layer(12, 6, 25, 3, 64, 10)
    x = torch.randn(9, 3, layer.in_coords.shape[0], generator=torch.Generator().manual_seed(6)).cuda()
    with torch.autocast("cuda", dtype=torch.bfloat16):
        y = layer(x)
    assert y.dtype == torch.bfloat16
    dy = torch.randn(y.shape, generator=torch.Generator().manual_seed(7)).bfloat16().cuda()
    y.backward(dy)
    assert torch.equal(layer.weight.grad, layer._dw_few(x, dy))
    dy[2, 5, 3] = float("inf")
    bad = layer._dw_few(x, dy)
    layer.dw_fused = False
    _, want = layer._backward(x, layer.weight, dy, False, True)
    # inf times the zeros of the slots that point 3 does not use, as in the dense product
    assert torch.equal(torch.isfinite(bad), torch.isfinite(want))


@pytest.mark.gpu
@pytest.mark.parametrize("res_in,res_out,k,c_in,c_out,side,batch", [(12, 6, 25, 3, 96, 10, 9), (8, 8, 30, 4, 128, 3, 33),
                                                                    (10, 8, 9, 1, 33, None, 5)])
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_non_finite_gradients_as_in_the_product_with_the_slot_sums(res_in, res_out, k, c_in, c_out, side, batch, dt):
    """dW = dy^T a over the matrix a of slot sums (fp32; bf16 for a bf16 x): an infinite dy gives
    infinities of the right sign, and NaN only where a is zero or infinities meet. x has values of few
    significant bits (zero middle and low parts) beside ordinary ones, an infinity and a NaN. The values
    that stay finite keep the fp32 sums' bound."""
    layer = _layer(res_in, res_out, k, c_in, c_out, side)
    n_in, n_out, v = layer.in_coords.shape[0], layer.out_coords.shape[0], layer.ref_coords.shape[0]
    g = torch.Generator().manual_seed(8)
    x = torch.randn(batch, c_in, n_in, generator=g).to(dt)
    x[:, :, ::2] = x[:, :, ::2].bfloat16().to(dt)
    x[0, 0, 1], x[1, 0, 2] = float("inf"), float("nan")
    dy = torch.randn(batch, c_out, n_out, generator=g).bfloat16()
    dy[2, 5, 3], dy[3, 6, 3], dy[4, 5, 7], dy[1, 7, 0] = (float(t) for t in ("inf", "-inf", "inf", "nan"))
    got = layer._dw_few(x.cuda(), dy.cuda()).cpu()
    sp, nbr = layer.slot_ptr.cpu().long(), layer.nbr_sorted.cpu().long()
    a = torch.zeros(batch, c_in, n_out, v)
    for r in range(int((sp & 0xFFFF).max())):            # in list order, as the slot-sum kernel
        n, s = torch.nonzero((sp & 0xFFFF) > r, as_tuple=True)
        a[:, :, n, s] += x[:, :, nbr[n, (sp[n, s] >> 16) + r]].float()
    a = (a if dt == torch.float32 else a.bfloat16()).double()
    want = torch.einsum("bon,bcnv->ocv", dy.double(), a).reshape(c_out, c_in * v)
    if k == 30:
        assert (torch.isinf(want[5]) & (want[5] > 0)).any() and (torch.isinf(want[6]) & (want[6] < 0)).any()
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    assert torch.equal(torch.isposinf(got), torch.isposinf(want))
    assert torch.equal(torch.isneginf(got), torch.isneginf(want))
    fin = torch.isfinite(want)
    assert fin.any() and not fin.all()
    assert_close_rel(got.double()[fin], want[fin], 1e-5, f"{dt}")


def test_dw_few_sizes():
    lib = _lib.load()
    assert lib.fovi_knnconv_dw_few_workspace_bytes(128, 3, 96, 4085, 964, 484, _lib.F32) > 0
    for args in ((0, 3, 96, 4, 4, 9, 0), (8, 9, 96, 4, 4, 9, 0), (8, 3, 96, 4, 4, 9, 2), (8, 3, 0, 4, 4, 9, 0)):
        assert lib.fovi_knnconv_dw_few_workspace_bytes(*args) == -1
    assert lib.fovi_knnconv_dw_few(_lib.KnnConvDwFewArgs(), None) != 0
    assert b"null pointer" in lib.fovi_last_error()


def test_dw_few_is_taken_where_it_pays():
    """Few images of a large layer are padded to 16: slot sums and a GEMM are faster there."""
    layer = _layer(48, 24, 49, 3, 96, 14, device="cpu")
    n_in = layer.in_coords.shape[0]
    for dt in (torch.float32, torch.bfloat16):
        pays = [layer._dw_few_pays(torch.zeros(b, 3, n_in, dtype=dt)) for b in (1, 2, 128)]
        assert pays == [False, False, True]
    small = _layer(8, 4, 9, 3, 32, None, device="cpu")          # below the host's own time
    assert small._dw_few_pays(torch.zeros(1, 3, small.in_coords.shape[0]))
    assert small._few_lists is not None and _layer(8, 4, 9, 9, 32, None, device="cpu")._few_lists is None
    eight = _layer(48, 24, 49, 8, 96, 14, device="cpu")         # channels-last bf16: the pair lists
    rows = lambda b: torch.zeros(b, eight.in_coords.shape[0], 8, dtype=torch.bfloat16).transpose(1, 2)
    assert not eight._dw_few_pays(rows(1)) and eight._dw_few_pays(rows(128))
    lib = _lib.load()
    assert lib.fovi_knnconv_dw_few_us(8, 9, 96, 4, 4, 9, _lib.F32, 1.0) == -1.0
    assert lib.fovi_knnconv_dw_few_us(128, 3, 96, 4085, 964, 484, _lib.F32, 2.0) > 100.0


@pytest.mark.gpu
@pytest.mark.parametrize("batch,few", [(1, False), (2, False), (128, True)])
def test_the_backward_follows_the_rule(batch, few, monkeypatch):
    layer = _layer(48, 24, 49, 3, 96, 14)
    g = torch.Generator().manual_seed(9)
    x = torch.randn(batch, 3, layer.in_coords.shape[0], generator=g)
    dy = torch.randn(batch, 96, layer.out_coords.shape[0], generator=g).bfloat16()
    calls = []
    inner = layer._dw_few
    monkeypatch.setattr(layer, "_dw_few", lambda *a: calls.append(1) or inner(*a))
    _, dw = layer._backward(x.cuda(), layer.weight, dy.cuda(), False, True)
    assert bool(calls) == few
    assert_close_rel(dw.double().cpu(), _dw64(layer, x, dy), 1e-5, f"{batch}")
