"""Phase times of an exec (get_measurement), stamped by its launches: forward
and backward, one- and two-launch column passes, general lengths, two-level,
16-bit storage through the FP32 workspace, batched plans.  Times are positive,
the phases fill the total, and the total lies within the host's own clock
around the exec; a graph replay stamps its own."""
import time

import pytest

pytestmark = pytest.mark.gpu


def _check(p, wall, split):
    total, first, second = (p.measurement(k) for k in ("total", "first_fftw", "second_fftw"))
    assert first > 0.0 and second > 0.0
    assert abs(total - first - second) <= 1e-8   # one tick of the 100 MHz clock
    assert total <= wall, (total, wall)
    a, b = p.measurement("column_a"), p.measurement("column_b")
    assert (a > 0.0 and b > 0.0) if split else (a == 0.0 and b == 0.0)
    if split:
        assert abs(a + b - (second if p.forward else first)) <= 2e-8


def _timed(torch, f):
    torch.cuda.synchronize()
    t = time.perf_counter()
    f()
    torch.cuda.synchronize()
    return time.perf_counter() - t


@pytest.mark.parametrize("nx,ny,prec,split", [(8, 14, "f64", False), (256, 16384, "f64", False),
                                              (2048, 512, "f32", False), (8192, 64, "f64", True),
                                              (300, 210, "f32", False), (18000, 16, "f64", False),
                                              (8209, 8, "f64", False), (8, 2 * 18000, "f32", False)])
def test_times(gpu, nx, ny, prec, split):
    import torch
    import hpxfft_amd
    rdt, cdt = (torch.float64, torch.complex128) if prec == "f64" else (torch.float32, torch.complex64)
    p = hpxfft_amd.Plan(nx, ny, precision=prec, ld_in=ny, stream=torch.cuda.current_stream())
    assert p.measurement("total") == 0.0
    x = torch.randn(nx, ny, dtype=rdt, device="cuda")
    out = torch.empty(nx, ny // 2 + 1, dtype=cdt, device="cuda")
    for _ in range(2):
        p.forward = True
        _check(p, _timed(torch, lambda: p.exec(x.data_ptr(), out.data_ptr())), split)
        p.forward = False
        p.exec_c2r(out.data_ptr(), x.data_ptr())
        _check(p, _timed(torch, lambda: p.exec_adjoint(out.data_ptr(), x.data_ptr())), split)
    p.close()


def test_times_16bit_workspace_batched_and_graph(gpu):
    import torch
    import hpxfft_amd
    s = torch.cuda.Stream()
    p = hpxfft_amd.Plan(20000, 16, precision="f16", stream=s)
    p.forward = True
    x = torch.zeros(20000, 18, dtype=torch.float16, device="cuda")
    ce = torch.empty(9, dtype=torch.int32, device="cuda")
    _check(p, _timed(torch, lambda: p.exec_scaled(x.data_ptr(), x.data_ptr(), None, ce.data_ptr())), False)
    p.close()

    b = hpxfft_amd.BatchedPlan([64, 2048], [128, 64], stream=s)
    b.forward = True
    g = [torch.zeros(64, 130, device="cuda"), torch.zeros(2048, 66, device="cuda")]
    _check(b, _timed(torch, lambda: b.exec([t.data_ptr() for t in g])), False)
    b.close()

    q = hpxfft_amd.Plan(2048, 2048, stream=s)
    q.forward = True
    d = torch.zeros(2048, 2050, dtype=torch.float64, device="cuda")
    out = torch.empty(2048, 1025, dtype=torch.complex128, device="cuda")
    q.exec(d.data_ptr(), out.data_ptr())
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        q.exec(d.data_ptr(), out.data_ptr())
    for _ in range(3):
        _check(q, _timed(torch, graph.replay), False)
    q.close()


def test_more_plans_than_the_stamp_pool(gpu):
    """Each plan has stamp words of its own, from the device's pool of 64 or allocated; both are given back."""
    import torch
    import hpxfft_amd
    x = torch.zeros(16, 32, dtype=torch.float64, device="cuda")
    out = torch.empty(16, 17, dtype=torch.complex128, device="cuda")
    for _ in range(2):
        plans = [hpxfft_amd.Plan(16, 32, ld_in=32, stream=torch.cuda.current_stream()) for _ in range(70)]
        for p in plans[::23]:
            p.exec(x.data_ptr(), out.data_ptr())
        torch.cuda.synchronize()
        times = [p.measurement("total") for p in plans]
        for p in plans:
            p.close()
        assert all((t > 0.0) == (i % 23 == 0) for i, t in enumerate(times)), times
