"""Image-row kernel (``knnconv_img.hip``): groups of points x images that visit only the slots the
group uses. CPU: its tables replayed against the CSR lists. GPU: bit-identical to the kernels that
visit every slot where those accumulate in the same order, else against the oracle."""
import pytest
import torch

from fovi_amd import _lib
from fovi_amd.arch import knn_tables as T
from fovi_amd.arch.knn import KNNConvLayer, _TransposedKnnConv
from fovi_amd.sensing.coords import SamplingCoords
from oracle import knnconv_ref
from tests.helpers import assert_close_rel


def _layer(res_in, res_out, k, c_in, c_out, side=None, style="logpolar", bias=True, seed=1, device="cuda"):
    a = 2.78 if style == "logpolar" else 0.5
    layer = KNNConvLayer(c_in, c_out, k, SamplingCoords(16, a, res_in, style=style),
                         SamplingCoords(16, a, res_out, style=style), device=device, bias=bias,
                         ref_frame_side_length=side)
    g = torch.Generator().manual_seed(seed)
    with torch.no_grad():
        layer.weight.copy_(torch.randn(layer.weight.shape, generator=g) * (1.0 / (c_in * layer._k)) ** 0.5)
        if bias:
            layer.bias.copy_(torch.randn(c_out, generator=g))
    return layer


def _oracle(layer, x, w):
    b = None if layer.bias is None else layer.bias.detach().cpu()
    return knnconv_ref.knnconv_forward(x.float(), layer.knn_indices.cpu(), layer.in_coords.shape[0],
                                       layer.local_rf.cpu(), w, b)


@pytest.mark.parametrize("res_in,res_out,k,side,style,pp", [
    (24, 12, 25, None, "logpolar", 1), (24, 12, 25, None, "logpolar", 8), (16, 8, 30, None, "isotropic", 4),
    (12, 12, 9, 6, "isotropic", 2), (20, 20, 9, None, "logpolar", 3)])
def test_tables_replay_the_csr_lists(res_in, res_out, k, side, style, pp):
    layer = _layer(res_in, res_out, k, 2, 2, side, style, device="cpu")
    n, v = layer.slot_ptr.shape
    order = torch.randperm(v, generator=torch.Generator().manual_seed(3)).tolist()
    for slot_order, point_order in ((None, None), (order, layer._point_order())):
        ent, points, nact = T.image_row_tables(layer.slot_ptr, layer.nbr_sorted, slot_order, point_order, pp)
        assert sorted(points[points >= 0].tolist()) == list(range(n))
        unions = []
        for g in range(points.shape[0]):
            used = set()
            for row in range(v):
                pos = ent[g, row, :, 3]
                assert (pos == pos[0]).all()
                slot = int(pos[0]) if slot_order is None else slot_order[int(pos[0])]
                for q in range(pp):
                    pt = int(points[g, q])
                    word = int(layer.slot_ptr[pt, slot]) if pt >= 0 else 0
                    cnt, begin = word & 0xFFFF, word >> 16
                    e = ent[g, row, q]
                    assert int(e[2]) == (cnt << 16 | begin) or cnt == 0 and int(e[2]) >> 16 == 0
                    lst = layer.nbr_sorted[pt, begin:begin + cnt].tolist() if cnt else []
                    none = -2 ** 31
                    assert [int(e[0]), int(e[1])] == (lst[:2] + [none, none])[:2]
                    if cnt:
                        assert row < int(nact[g])
                        used.add(slot)
            assert len(used) == int(nact[g])
            # the used slots in visit order, then the others in visit order: each slot once
            seq = ent[g, :, 0, 3].tolist()
            na = int(nact[g])
            assert seq[:na] == sorted(seq[:na]) and seq[na:] == sorted(seq[na:]) and sorted(seq) == list(range(v))
            unions.append(na)
        if n <= T.IMG_WINDOW:
            got = T.image_row_union(layer.slot_ptr, point_order, pp)
            assert got == pytest.approx(sum(unions) / len(unions))


def test_spatial_order_is_a_permutation_of_compact_runs():
    c = SamplingCoords(16, 2.78, 64, style="logpolar")
    order = T.spatial_order(c.cortical)
    assert sorted(order.tolist()) == list(range(4096))
    pts = c.cortical[order.long()].reshape(16, 256, -1)
    area = (pts.amax(1) - pts.amin(1)).prod(1)
    whole = (c.cortical.amax(0) - c.cortical.amin(0)).prod()
    assert float(area.max()) < 0.12 * float(whole)       # 1 / 16 each, but for the lattice's rounding


def test_group_tables_refuse_bad_arguments():
    lib = _lib.load()
    layer = _layer(8, 8, 9, 2, 2, device="cpu")
    bad = torch.full((64,), 64, dtype=torch.int32)
    sp = layer.slot_ptr.contiguous()
    assert lib.fovi_knnconv_img_tables(_lib.ptr(sp), None, 64, 9, 9, None, _lib.ptr(bad), 1, 256, 1, None, None,
                                       None, None) == -1
    assert b"point_order" in lib.fovi_last_error()
    assert lib.fovi_knnconv_img_tables(None, None, 64, 9, 9, None, None, 1, 256, 1, None, None, None, None) == -1
    assert lib.fovi_knnconv_weight_img_elems(33, 21, 9, _lib.BF16) == 32 * 9 * 64
    assert lib.fovi_knnconv_weight_img_elems(33, 21, 9, 7) == -1


# rows per workgroup / 32, images per point, column blocks per wave
_PLANS = [None, (4, 128, 2), (4, 16, 1), (2, 32, 1), (1, 16, 2), (1, 32, 1)]


@pytest.mark.gpu
@pytest.mark.parametrize("res_in,res_out,k,c_in,c_out,batch", [
    (16, 16, 9, 32, 256, 8),        # one channel chunk, half a block of images
    (24, 12, 25, 64, 200, 33),      # strided, partial column block, odd batch
    (16, 16, 9, 96, 512, 17),       # three chunks (an odd number of stages), two column tiles
    (32, 16, 25, 64, 192, 130),     # a batch past one block of 128
    (20, 20, 25, 128, 256, 16),     # long lists at the fovea
])
def test_bf16_equals_the_wide_layer_kernel(res_in, res_out, k, c_in, c_out, batch):
    """Same slot sums (fp32, list order, one rounding), same order of slots and chunks; the skipped
    slots would add products of zeros: bit-identical, whatever the plan."""
    layer = _layer(res_in, res_out, k, c_in, c_out)
    x = torch.randn(batch, res_in * res_in, c_in, generator=torch.Generator().manual_seed(2)).bfloat16().cuda()
    x = x.transpose(1, 2)
    with torch.no_grad():
        layer.image_rows = False
        want = layer.forward_fused(x, "relu")
        assert layer.last_weight_layout == "mfma"
        layer.image_rows = True
        for plan in _PLANS:
            if plan is not None:
                layer._img.plans[batch] = (0.0, plan)
            got = layer.forward_fused(x, "relu")
            assert _lib.knnconv_last_path() == "bf16 image rows"
            assert torch.equal(got, want), plan


@pytest.mark.gpu
@pytest.mark.parametrize("res_in,res_out,k,c_in,c_out,side,style,batch,layout", [
    (16, 8, 30, 40, 33, None, "isotropic", 9, "rows"),        # pad ring, partial chunk, odd columns
    (12, 12, 9, 21, 65, 6, "logpolar", 12, "planes"),         # odd channels: padded copy; V = 36
    (16, 4, 64, 16, 96, 2, "logpolar", 40, "rows"),           # 64 neighbours in 4 slots: long lists
    (16, 16, 9, 72, 300, None, "logpolar", 8, "view-major"),  # rows of one point for all images adjacent
    (12, 6, 25, 48, 8, 10, "isotropic", 20, "expanded"),      # one image expanded over the batch
])
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_against_the_oracle(res_in, res_out, k, c_in, c_out, side, style, batch, layout, dt):
    layer = _layer(res_in, res_out, k, c_in, c_out, side, style)
    n = layer.in_coords.shape[0]
    x = torch.randn(batch, c_in, n, generator=torch.Generator().manual_seed(4)).to(dt)
    if layout == "expanded":
        x = x[:1].expand(batch, -1, -1)
    if layout == "rows":
        xd = x.cuda().transpose(1, 2).contiguous().transpose(1, 2)
    elif layout == "view-major":
        xd = x.cuda().permute(2, 0, 1).contiguous().permute(1, 2, 0)
    elif layout == "expanded":
        xd = x[:1].cuda().transpose(1, 2).contiguous().transpose(1, 2).expand(batch, -1, -1)
    else:
        xd = x.cuda()
    w = layer.weight.detach().cpu()
    ref = _oracle(layer, x, w if dt == torch.float32 else w.bfloat16().float())
    with torch.no_grad():
        for plan in _PLANS:
            if plan is not None:
                layer._img.plans[batch] = (0.0, plan)
            y = layer(xd)
            assert layer.last_weight_layout == "image"
            assert_close_rel(y.float().cpu(), ref, 1e-5 if dt == torch.float32 else 1e-2, f"{plan}")


@pytest.mark.gpu
@pytest.mark.parametrize("res_in,res_out,k,c_in,c_out,batch", [(16, 16, 9, 64, 256, 9), (24, 12, 25, 128, 96, 33)])
def test_e4m3_equals_the_other_kernels(res_in, res_out, k, c_in, c_out, batch):
    """Saturating e4m3 slot sums included: planted 448s whose sums overflow, and NaN bytes."""
    layer = _layer(res_in, res_out, k, c_in, c_out)
    layer.set_slot_order(None)
    x = torch.randn(batch, c_in, res_in * res_in, generator=torch.Generator().manual_seed(5)).bfloat16().cuda()
    xq = layer.quantize_input(x)
    raw = xq.data.view(torch.uint8)
    raw[0, 5, ::3] = 0x7E
    raw[1, 9, ::5] = 0x7F
    with torch.no_grad():
        got = layer(xq)
        assert _lib.knnconv_last_path() == "fp8 image rows"
        layer.image_rows = False
        want = layer(xq)
    assert torch.isnan(want).any() and torch.equal(torch.isnan(got), torch.isnan(want))
    keep = ~torch.isnan(want)
    assert torch.equal(got[keep], want[keep])


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_non_finite_weights_reach_the_points_with_empty_slots(dt):
    """0 * inf is NaN: with a non-finite weight every slot is visited, as in the other kernels."""
    layer = _layer(16, 16, 25, 32, 256)
    x = torch.randn(8, 256, 32, generator=torch.Generator().manual_seed(6)).to(dt).cuda().transpose(1, 2)
    with torch.no_grad():
        layer.weight[3, 7 * 25] = float("inf")
        layer.weight[9, 11 * 25 + 24] = float("nan")
        got = layer(x)
        assert layer.last_weight_layout == "image"
        layer.image_rows = False
        want = layer(x)
    assert torch.isnan(want[:, 3]).any() and torch.isfinite(want[:, 4]).all()
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    assert torch.equal(torch.isinf(got), torch.isinf(want))


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_gradients_through_the_image_row_kernel(dt):
    """The input gradient runs the same kernel on the inverse tables, from a channel-planes
    output gradient too; both gradients against those of the other kernels."""
    layer = _layer(16, 12, 9, 32, 96, side=6)
    x = torch.randn(10, 256, 32, generator=torch.Generator().manual_seed(7)).to(dt).cuda().transpose(1, 2)
    dy = torch.randn(10, 96, 144, generator=torch.Generator().manual_seed(8)).to(dt).cuda()

    def grads(image):
        layer.image_rows = image
        layer._transposed(x.device).image_rows = image
        xg = x.detach().requires_grad_(True)
        layer.weight.grad = layer.bias.grad = None
        layer(xg).backward(dy)
        return xg.grad.float(), layer.weight.grad.float(), layer.bias.grad.float()

    got, want = grads(True), grads(False)
    assert isinstance(layer._transposed_conv, _TransposedKnnConv)
    assert layer._transposed_conv.last_weight_layout == "rows"
    tol = 2e-5 if dt == torch.float32 else 1e-2
    for a, b, what in zip(got, want, ("dx", "dW", "db")):
        assert_close_rel(a.cpu(), b.cpu(), tol, what)


def test_input_layouts_the_kernel_reads():
    buf = torch.zeros(2, 9, 96, dtype=torch.uint8).view(torch.float8_e4m3fn)
    e4m3 = torch.float8_e4m3fn
    ready = KNNConvLayer._image_input_ready
    assert ready(buf[:, :, :64].transpose(1, 2), e4m3) and ready(buf[:, :, 16:80].transpose(1, 2), e4m3)
    assert not ready(buf[:, :, 8:72].transpose(1, 2), e4m3)         # rows not 16-byte aligned
    assert not ready(buf[:, :, :56].transpose(1, 2), e4m3)          # rows not a multiple of 16 bytes
    assert not ready(buf[:, :, :64].permute(0, 2, 1).contiguous(), e4m3)
    x = torch.zeros(2, 9, 12).transpose(1, 2)
    assert KNNConvLayer._image_input(x, torch.float32) is x


@pytest.mark.gpu
def test_unaligned_e4m3_rows_are_not_copied(monkeypatch):
    """They run the kernels that read them as they are: the answer, or the refusal, of those."""
    layer = _layer(16, 16, 9, 64, 256)
    x = torch.randn(9, 64, 256, generator=torch.Generator().manual_seed(9)).bfloat16().cuda()
    xq = layer.quantize_input(x)
    want = layer(xq)
    assert layer.last_weight_layout == "image"

    def never(*a):
        raise AssertionError("copied")
    monkeypatch.setattr(KNNConvLayer, "_image_input", staticmethod(never))
    buf = torch.zeros(9, 256, 96, dtype=torch.uint8, device="cuda").view(torch.float8_e4m3fn)
    buf.view(torch.uint8)[:, :, 8:72] = xq.data.view(torch.uint8).transpose(1, 2)
    xq = xq._replace(data=buf[:, :, 8:72].transpose(1, 2))
    try:
        got = layer(xq)
    except RuntimeError as e:
        assert "fovi_knnconv_fwd" in str(e)
        layer.image_rows = False
        with pytest.raises(RuntimeError, match="fovi_knnconv_fwd"):
            layer(xq)
        return
    assert layer.last_weight_layout != "image"
    assert_close_rel(got.float().cpu(), want.float().cpu(), 1e-2, "unaligned")
