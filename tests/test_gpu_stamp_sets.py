"""Stamp words of plans and captured graphs: a plan made inside a capture gets its
words like any other, however many plans there are, and a graph that outlives its plan
does not stamp the words of a later one."""
import time

import pytest

pytestmark = pytest.mark.gpu


def test_plan_made_inside_a_capture(gpu):
    """More plans than a block of stamp words holds, all but the first made while the stream is captured."""
    import torch
    import hpxfft_amd
    x = torch.randn(16, 32, dtype=torch.float64, device="cuda")
    out = torch.empty(16, 17, dtype=torch.complex128, device="cuda")
    s = torch.cuda.Stream()
    plans = [hpxfft_amd.Plan(16, 32, ld_in=32, stream=s)]   # the device's tables
    plans[0].exec(x.data_ptr(), out.data_ptr())
    torch.cuda.synchronize()
    ref = out.clone()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        plans += [hpxfft_amd.Plan(16, 32, ld_in=32, stream=s) for _ in range(140)]
        plans[-1].exec(x.data_ptr(), out.data_ptr())
    for _ in range(3):
        out.fill_(float("nan"))
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ref)
    assert plans[-1].measurement("total") > 0.0
    for p in plans:
        p.close()


def test_graph_that_outlives_its_plan(gpu):
    """Its replays (a grid of 2^24 points) do not show in the times of the next plan (16 x 32)."""
    import torch
    import hpxfft_amd
    x = torch.randn(1024, 16384, dtype=torch.float64, device="cuda")
    out = torch.empty(1024, 8193, dtype=torch.complex128, device="cuda")
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    p = hpxfft_amd.Plan(1024, 16384, ld_in=16384, stream=s)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        p.exec(x.data_ptr(), out.data_ptr())
    p.close()
    q = hpxfft_amd.Plan(16, 32, ld_in=32, stream=s)
    torch.cuda.synchronize()
    t = time.perf_counter()
    q.exec(x.data_ptr(), out.data_ptr())
    torch.cuda.synchronize()
    wall = time.perf_counter() - t
    for _ in range(3):
        g.replay()
    torch.cuda.synchronize()
    assert 0.0 < q.measurement("total") <= wall
    assert q.measurement("first_fftw") + q.measurement("second_fftw") <= wall
    q.close()
