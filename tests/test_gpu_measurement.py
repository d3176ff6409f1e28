"""get_measurement reads an exec's stamps once and leaves a captured stream alone."""
import time

import pytest

pytestmark = pytest.mark.gpu

KEYS = ("total", "first_fftw", "second_fftw", "column_a", "column_b")


def _plan(torch, stream):
    import hpxfft_amd
    x = torch.randn(256, 512, dtype=torch.float64, device="cuda")
    out = torch.empty(256, 257, dtype=torch.complex128, device="cuda")
    p = hpxfft_amd.Plan(256, 512, ld_in=512, stream=stream)
    torch.cuda.synchronize()
    p.exec(x.data_ptr(), out.data_ptr())
    torch.cuda.synchronize()
    return p, x, out


@pytest.mark.parametrize("read_before", [False, True])
def test_inside_a_capture(gpu, read_before):
    """Times read before the capture are given again; others are refused.  Either way the
    capture stays valid and its replays hold the caller's work alone."""
    import torch
    import hpxfft_amd
    from hpxfft_amd._lib import HpxfftError
    s = torch.cuda.Stream()
    p, x, out = _plan(torch, s)
    before = [p.measurement(k) for k in KEYS] if read_before else None
    a = torch.ones(1024, device="cuda")
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    refused = None
    with torch.cuda.graph(g, stream=s):
        a.mul_(2)
        try:
            inside = [p.measurement(k) for k in KEYS]
        except HpxfftError as e:
            refused = str(e)
        a.add_(1)
    if read_before:
        assert refused is None and inside == before
    else:
        assert refused is not None and "being captured" in refused
    want = 1.0
    for _ in range(3):
        g.replay()
        torch.cuda.synchronize()
        want = 2 * want + 1
        assert bool((a == want).all())
    after = [p.measurement(k) for k in KEYS]
    assert after[0] > 0.0 and (before is None or after == before)
    p.close()


def test_one_read_serves_all_keys(gpu):
    """The second key does not wait for work queued after the first was read; a new exec is read anew."""
    import torch
    s = torch.cuda.Stream()
    p, x, out = _plan(torch, s)
    total = p.measurement("total")
    with torch.cuda.stream(s):
        torch.cuda._sleep(100_000_000)   # some 40 ms or more
        done = torch.cuda.Event()
        done.record(s)
    first, second = p.measurement("first_fftw"), p.measurement("second_fftw")
    assert not done.query()
    assert abs(total - first - second) <= 1e-8
    t = time.perf_counter()
    p.exec(x.data_ptr(), out.data_ptr())
    assert p.measurement("total") > 0.0 and done.query()
    assert p.measurement("total") <= time.perf_counter() - t
    p.close()


def test_every_kind_of_exec_is_read_anew(gpu):
    """Forward, backward, host, batched, and 16-bit through the FP32 workspace: after each
    of eight execs the times are that exec's, not one kept from before."""
    import numpy as np
    import torch
    import hpxfft_amd
    s = torch.cuda.Stream()
    p, x, out = _plan(torch, s)
    h = hpxfft_amd.Plan(256, 512, stream=s)
    xh = np.zeros((256, 514))
    b = hpxfft_amd.BatchedPlan([64, 512], [128, 64], stream=s)
    grids = [torch.zeros(64, 130, device="cuda"), torch.zeros(512, 66, device="cuda")]
    w = hpxfft_amd.Plan(20000, 16, precision="f16", stream=s)
    x16 = torch.zeros(20000, 18, dtype=torch.float16, device="cuda")
    ce = torch.empty(9, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    ptrs = [t.data_ptr() for t in grids]
    for q, run in ((p, lambda: p.exec(x.data_ptr(), out.data_ptr())),
                   (p, lambda: p.exec_adjoint(out.data_ptr(), x.data_ptr())),
                   (h, lambda: h.exec_host(xh)), (b, lambda: b.exec(ptrs)),
                   (w, lambda: w.exec_scaled(x16.data_ptr(), x16.data_ptr(), None, ce.data_ptr()))):
        seen = set()
        for _ in range(8):   # 10 ns steps: eight runs do not all take the same
            run()
            seen.add(tuple(q.measurement(k) for k in KEYS))
        assert len(seen) > 1, seen
    for q in (p, h, b, w):
        q.close()
