"""The host entry point reads its run's phase times once; a later exec of the same plan
reports its own, and a plan with a captured exec reads them from the device each time."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

KEYS = ("total", "first_fftw", "second_fftw")


@pytest.mark.parametrize("captured", [False, True])
def test_times_follow_the_last_exec(gpu, captured):
    import torch
    import hpxfft_amd
    nx, ny = 256, 512
    print(f"host times, captured exec {captured}", flush=True)
    x = oracle.fill(nx, ny, seed=3, dist="upm1")
    d = torch.from_numpy(x).cuda()
    stream = torch.cuda.Stream()
    p = hpxfft_amd.Plan(nx, ny, precision="f64", stream=stream)
    g = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    if captured:
        with torch.cuda.graph(g, stream=stream):
            p.exec(d.data_ptr(), d.data_ptr())
    h = x.copy()
    p.exec_host(h)
    host = [p.measurement(k) for k in KEYS]
    assert all(v > 0 for v in host) and host == [p.measurement(k) for k in KEYS]
    assert p.measurement("h2d") > 0
    assert oracle.rel_l2(h.view(np.complex128), oracle.r2c_2d(x, ny)) <= 1e-12
    seen = set()
    for _ in range(8):   # the stamps resolve 10 ns: eight runs do not all repeat the host run's times
        if captured:
            g.replay()
        else:
            p.exec(d.data_ptr(), d.data_ptr())
        torch.cuda.synchronize()
        seen.add(tuple(p.measurement(k) for k in KEYS))
    assert seen != {tuple(host)}
    p.close()
