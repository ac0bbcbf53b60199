"""The image-row kernel's group tables belong to the layer: built with its other tables for every group
size a plan may take, moved with it, and never by a call."""
import copy
import io

import pytest
import torch

from fovi_amd import _lib
from fovi_amd.arch import knn_tables as T
from fovi_amd.arch.knn import KNNConvLayer, _ImageRows, _TransposedKnnConv, get_in_out_coords


def _layer(c_in, c_out, device, res=32, stride=2, k=9):
    cin, cout, _ = get_in_out_coords(res, 16, 2.78, stride, style="logpolar", auto_match_cart_resources=0, device=device)
    return KNNConvLayer(c_in, c_out, k, cin, cout, device=device)


def test_no_call_builds_tables(monkeypatch):
    layer = _layer(16, 24, "cpu")
    layers = [layer, _TransposedKnnConv(layer, torch.device("cpu"))]
    want = {pp: T.image_row_tables(layer.slot_ptr, layer.nbr_sorted, layer.slot_order, layer._point_order(), pp)
            for pp in (1, 2, 4, 8)}

    def never(*a, **k):
        raise AssertionError("tables built by a call")
    for name in ("image_row_tables", "image_row_union", "spatial_order"):
        monkeypatch.setattr(T, name, never)
    taken = set()
    for la in layers + [copy.deepcopy(layer)]:
        for batch in (8, 9, 15, 16, 17, 31, 40, 64, 100, 128, 256, 1000):
            _, (rb, ib, _) = la._image_plan(batch)
            la._image_tables_of(rb * 32 // ib, torch.device("cpu"))
            taken.add(rb * 32 // ib)
    assert len(taken) > 1
    for pp, tables in want.items():
        assert all(torch.equal(a, b) for a, b in zip(layer._image_tables_of(pp, torch.device("cpu")), tables))
    assert layer.to("meta")._img.tables[2][0].device.type == "meta"


def test_a_new_slot_order_and_few_channels():
    layer = _layer(16, 24, "cpu")
    before = layer._img.tables[4][0].clone()
    layer.set_slot_order([8, 7, 6, 5, 4, 3, 2, 1, 0])
    assert sorted(layer._img.tables) == [1, 2, 4, 8] and not torch.equal(layer._img.tables[4][0], before)
    assert not _layer(8, 24, "cpu")._img.tables          # never run by this kernel


def test_very_large_layers_keep_to_two_group_sizes():
    img = _ImageRows(torch.zeros(1, 9, dtype=torch.int32), torch.zeros(1, 9, dtype=torch.int32))
    assert img.groups() == (1, 2, 4, 8)
    img.slot_ptr = torch.zeros(1, 1, dtype=torch.int32).expand(1 << 17, 65)
    assert img.groups() == (1, 2)
    layer = _layer(16, 24, "cpu")
    layer._img.groups = lambda: (1, 2)
    for batch in (8, 16, 17, 33, 256):
        _, (rb, ib, _) = layer._image_plan(batch)
        assert rb * 32 // ib in (1, 2)


def test_layers_pickled_with_the_device_in_front_of_their_tables():
    layer = _layer(16, 24, "cpu")
    layer._img.tables = {pp: (torch.device("cpu"),) + t for pp, t in layer._img.tables.items() if pp == 2}
    f = io.BytesIO()
    torch.save(layer, f)
    f.seek(0)
    layer = torch.load(f, weights_only=False)
    assert len(layer._img.tables[2]) == 3
    assert layer._image_tables_of(8, torch.device("cpu"))[1].shape == (32, 8)     # built when asked for


def test_group_tables_of_many_windows_equal_those_of_one_thread():
    """Windows are shared out to threads; each window's groups alone give the same rows."""
    layer = _layer(16, 4, "cpu", res=64, stride=1)            # 4096 points: 16 windows
    order = layer._point_order()
    for pp in (1, 3, 8):
        ent, points, nact = T.image_row_tables(layer.slot_ptr, layer.nbr_sorted, None, order, pp)
        per = -(-T.IMG_WINDOW // pp)
        for q in (0, 7, 15):
            part = order[q * T.IMG_WINDOW:(q + 1) * T.IMG_WINDOW].long()
            e, p, n = T.image_row_tables(layer.slot_ptr[part], layer.nbr_sorted[part], None, None, pp)
            rows = slice(q * per, (q + 1) * per)
            assert torch.equal(ent[rows], e) and torch.equal(nact[rows], n)
            assert torch.equal(points[rows], torch.where(p < 0, p, part[p.clamp(min=0).long()].to(p.dtype)))


def test_point_orders_of_another_length_are_refused():
    layer = _layer(16, 4, "cpu")
    for bad in (layer._point_order()[:-1], layer._point_order().long()):
        with pytest.raises(ValueError, match="point_order"):
            T.image_row_tables(layer.slot_ptr, layer.nbr_sorted, None, bad, 2)
        with pytest.raises(ValueError, match="point_order"):
            T.image_row_union(layer.slot_ptr, bad, 2)


@pytest.mark.gpu
def test_a_capture_takes_the_kernel_an_eager_call_takes():
    """Batches whose plans take other group sizes than the one eager call before the capture."""
    layer = _layer(32, 48, "cuda")
    x = torch.randn(256, 1024, 32, generator=torch.Generator().manual_seed(1)).cuda().transpose(1, 2)
    side = torch.cuda.Stream()
    with torch.no_grad():
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            layer(x[:256])                      # packs the weight
        torch.cuda.current_stream().wait_stream(side)
        sizes = set()
        for batch in (8, 20, 100):
            sizes.add(layer._image_plan(batch)[1])
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                y = layer(x[:batch])
            assert _lib.knnconv_last_path() == "f32 image rows"
            want = layer(x[:batch])
            for _ in range(3):
                y.zero_()
                graph.replay()
                torch.cuda.synchronize()
                assert torch.equal(y, want)
        assert len(sizes) > 1
