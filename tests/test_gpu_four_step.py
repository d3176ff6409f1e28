"""The FP64 / FP32 four-step columns (Nx >= 2^13) where its scratch is shared or replayed:
the allocation-free entry point's static array, the per-grid slices of a strided batch
forward and backward, and graph replays.  (2^11 and 2^12 rows run as one launch and use
no scratch.)  Every plan's text must say four-step.  Against the oracle: FP64 <= 1e-12,
FP32 <= 1e-5, the bounds of the other parity tests."""
import ctypes

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

TOL = {"f64": 1e-12, "f32": 1e-5}


def _dt(prec):
    import torch
    return (torch.float64, torch.complex128) if prec == "f64" else (torch.float32, torch.complex64)


def _four_step_plan(*args, **kw):
    import hpxfft_amd
    p = hpxfft_amd.Plan(*args, **kw)
    text = p.describe()
    assert "column c2c four-step" in text and "in registers" not in text, text
    return p


def _noalloc(nx, ny, ld_in, ld_out, prec, d_in, d_out, stream=0):
    import hpxfft_amd
    return hpxfft_amd.lib().hpxfft_exec_r2c_2d_noalloc(nx, ny, ld_in, ld_out, 0 if prec == "f64" else 1,
                                                       ctypes.c_void_p(d_in), ctypes.c_void_p(d_out),
                                                       ctypes.c_void_p(stream))


@pytest.mark.parametrize("prec", ["f64", "f32"])
def test_noalloc_calls_in_a_row(gpu, prec):
    """8192 x 1024 takes 71 MB (FP64) of the static scratch; the next calls find its contents there."""
    import torch
    import hpxfft_amd
    rdt, cdt = _dt(prec)
    for i, (nx, ny) in enumerate([(8192, 1024), (8192, 64), (16384, 32), (8192, 1024)]):
        print(f"noalloc four-step {prec} {nx}x{ny} (call {i + 1})", flush=True)
        nc = ny // 2 + 1
        x = oracle.fill(nx, ny, seed=60 + i, dist="upm1")
        d = torch.from_numpy(x).to(device="cuda", dtype=rdt)
        got = torch.full((nx, nc), float("nan"), dtype=cdt, device="cuda")
        assert _noalloc(nx, ny, 2 * nc, nc, prec, d.data_ptr(), got.data_ptr()) == 0, hpxfft_amd.last_error()
        want = torch.empty_like(got)
        p = _four_step_plan(nx, ny, precision=prec)
        p.exec(d.data_ptr(), want.data_ptr())
        assert _noalloc(nx, ny, 2 * nc, nc, prec, d.data_ptr(), d.data_ptr()) == 0, hpxfft_amd.last_error()
        torch.cuda.synchronize()
        p.close()
        assert torch.equal(got, want) and torch.equal(d.view(cdt), want)
        assert oracle.rel_l2(got.cpu().numpy().astype(np.complex128), oracle.r2c_2d(x, ny)) <= TOL[prec]


@pytest.mark.parametrize("prec", ["f64", "f32"])
def test_noalloc_refuses_beyond_the_scratch(gpu, prec):
    """8192 x 4096: 273 MB (FP64) and 138 MB (FP32)."""
    import torch
    import hpxfft_amd
    from hpxfft_amd import _lib
    d = torch.zeros(16, dtype=torch.float64, device="cuda")
    assert _noalloc(8192, 4096, 4098, 2049, prec, d.data_ptr(), d.data_ptr()) == _lib.UNSUPPORTED_SIZE
    assert "holds 134217728 bytes" in hpxfft_amd.last_error()


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("entry", ["plan", "c2r", "noalloc"])
def test_graph_replays(gpu, entry, prec):
    import torch
    import hpxfft_amd
    nx, ny = 8192, 130
    nc = ny // 2 + 1
    if entry == "noalloc":
        ny, nc = 128, 65   # powers of two only
    rdt, cdt = _dt(prec)
    x = oracle.fill(nx, ny, seed=71, dist="upm1")
    d = torch.from_numpy(x).to(device="cuda", dtype=rdt)
    spec = torch.from_numpy(oracle.r2c_2d(x, ny)).to(device="cuda", dtype=cdt)
    s = torch.cuda.Stream()
    p = _four_step_plan(nx, ny, precision=prec, stream=s)
    if entry == "c2r":
        out = torch.zeros_like(d)
        run = lambda: p.exec_c2r(spec.data_ptr(), out.data_ptr())   # noqa: E731
    else:
        out = torch.empty((nx, nc), dtype=cdt, device="cuda")
        run = lambda: p.exec(d.data_ptr(), out.data_ptr())   # noqa: E731
    if entry == "noalloc":
        def run():
            rc = _noalloc(nx, ny, 2 * nc, nc, prec, d.data_ptr(), out.data_ptr(), s.cuda_stream)
            assert rc == 0, hpxfft_amd.last_error()
    torch.cuda.synchronize()
    run()
    torch.cuda.synchronize()
    ref = out.clone()
    host = ref.cpu().numpy()
    if entry == "c2r":
        want = oracle.c2r_2d(spec.cpu().numpy().astype(np.complex128), ny)
        assert oracle.rel_l2(host[:, :ny].astype(np.float64), want) <= TOL[prec]
    else:
        assert oracle.rel_l2(host.astype(np.complex128), oracle.r2c_2d(x, ny)) <= TOL[prec]
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        run()
    for r in range(3):
        out[:, :ny] = float("nan")
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ref), r
        d.mul_(1.0)   # eager work between replays
    p.close()


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("nx,ny,batch", [(8192, 64, 3), (16384, 30, 2)])
def test_strided_batch(gpu, nx, ny, batch, prec):
    """Grids apart by more than their size, each with its own slice of the scratch: forward, adjoint, c2r."""
    import torch
    rdt, cdt = _dt(prec)
    print(f"four-step {prec} {batch} x {nx}x{ny}", flush=True)
    nc = ny // 2 + 1
    xs = [oracle.fill(nx, ny, seed=80 + b, dist="normal") for b in range(batch)]
    ld_out, dist_out = nc + 2, (nx + 1) * (nc + 2)
    d = torch.zeros((batch, nx + 2, 2 * nc), dtype=rdt, device="cuda")
    d[:, :nx] = torch.from_numpy(np.stack(xs)).to(device="cuda", dtype=rdt)
    out = torch.full((batch, nx + 1, ld_out), complex(7, 7), dtype=cdt, device="cuda")
    p = _four_step_plan(nx, ny, batch=batch, precision=prec, ld_in=2 * nc, dist_in=(nx + 2) * 2 * nc, ld_out=ld_out,
                        dist_out=dist_out)
    p.exec(d.data_ptr(), out.data_ptr())
    torch.cuda.synchronize()
    for b in range(batch):
        got = out[b, :nx, :nc].cpu().numpy().astype(np.complex128)
        assert oracle.rel_l2(got, oracle.r2c_2d(xs[b], ny)) <= TOL[prec], b
    Y = torch.randn((batch, nx + 1, ld_out), dtype=torch.complex128, device="cuda").to(cdt)
    Yr = Y[:, :nx, :nc].cpu().numpy().astype(np.complex128)
    for run, ref in ((p.exec_adjoint, oracle.adjoint_r2c_2d), (p.exec_c2r, oracle.c2r_2d)):
        r = torch.full((batch, nx + 2, 2 * nc), 7.0, dtype=rdt, device="cuda")
        run(Y.data_ptr(), r.data_ptr())
        torch.cuda.synchronize()
        for b in range(batch):
            got = r[b, :nx, :ny].cpu().numpy().astype(np.float64)
            assert oracle.rel_l2(got, ref(np.ascontiguousarray(Yr[b]), ny)) <= TOL[prec], b
        assert bool((r[:, nx:] == 7).all()) and bool((r[:, :nx, ny:] == 7).all())
    out[:, :nx, :nc] = complex(7, 7)
    assert bool((out == complex(7, 7)).all())   # nothing beyond the grids
    p.close()
