"""Fixations under stream capture: host arguments are refused (their copy would be replayed from a host
block that has been given back), prepared views are captured."""
import numpy as np
import pytest
import torch

from fovi_amd.sensing.samplers import GridSampler

_SIZE = np.array([[64, 64]] * 2)


def test_host_fixations_are_refused_while_capturing(monkeypatch):
    sampler = GridSampler(16, 2.78, 16, device="cpu", style="logpolar")
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    for device in ("cuda", "cuda:0"):
        for blocking in (False, True):
            with pytest.raises(RuntimeError, match="prepare_views before the capture"):
                sampler._make_views(torch.full((2, 2), 0.5), _SIZE, 2, device, None, blocking)


@pytest.mark.gpu
def test_captured_sampling_takes_prepared_views():
    sampler = GridSampler(16, 2.78, 16, device="cuda", mode="bilinear", style="logpolar")
    g = torch.Generator().manual_seed(1)
    img = torch.randn(2, 3, 64, 64, generator=g).cuda()
    fix = torch.rand(2, 2, generator=g)
    views = sampler.prepare_views(fix, _SIZE, 2, img.device)
    want = sampler.sample_views(img, fix, _SIZE)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        sampler.sample_views(img, views=views)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        with pytest.raises(RuntimeError, match="prepare_views before the capture"):
            sampler.sample_views(img, fix, _SIZE)
        with pytest.raises(RuntimeError, match="prepare_views before the capture"):
            sampler.prepare_views(fix, _SIZE, 2, img.device)
        out = sampler.sample_views(img, views=views)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        torch.empty(1 << 16, pin_memory=True).fill_(7.0)      # host blocks written in between
