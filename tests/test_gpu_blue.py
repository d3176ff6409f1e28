"""Bluestein's algorithm in registers: one length for each convolution length
2^8 .. 2^13 (FP64) / 2^14 (FP32), as rows and as columns.

The lengths lie at the edges: the largest prime below half of the convolution
length (only there do the padded halves meet) and the smallest composite with a
factor above 61 past the previous one (the most padding).  The other dimension
makes rows and strips that do not fill a workgroup.  Forward in place and out of
place in a pitch of its own, strided batches, the adjoint and c2r, against the FP64
oracle (FP64 <= 1e-12, FP32 <= 1e-5, the bounds of the other parity tests).
"""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

TOL = {"f64": 1e-12, "f32": 1e-5}
LENGTHS = [67, 127, 131, 251, 262, 509, 514, 1021, 1028, 2039, 2053, 4093]
CASES = [(n, p) for n in LENGTHS for p in ("f64", "f32")] + [(4099, "f32"), (8191, "f32")]


def _dt(prec):
    import torch
    return (torch.float64, torch.complex128) if prec == "f64" else (torch.float32, torch.complex64)


def _check(nx, ny, prec, batch=1):
    import torch
    import hpxfft_amd
    print(f"blue {prec} {nx}x{ny} batch {batch}", flush=True)
    rdt, cdt = _dt(prec)
    nc = ny // 2 + 1
    xs = [oracle.fill(nx, ny, seed=nx + ny + b, dist="normal") for b in range(batch)]
    d = torch.from_numpy(np.stack(xs)).to(device="cuda", dtype=rdt)
    out = torch.full((batch, nx + 1, nc + 3), complex(7, 7), dtype=cdt, device="cuda")
    p = hpxfft_amd.Plan(nx, ny, batch=batch, precision=prec, ld_in=2 * nc, ld_out=nc + 3,
                        dist_out=(nx + 1) * (nc + 3))
    p.exec(d.data_ptr(), out.data_ptr())
    q = hpxfft_amd.Plan(nx, ny, batch=batch, precision=prec)
    assert "Bluestein" in q.describe() and "in registers" in q.describe()
    q.exec(d.data_ptr(), d.data_ptr())
    torch.cuda.synchronize()
    got = d.view(cdt)
    for b in range(batch):
        assert oracle.rel_l2(got[b].cpu().numpy().astype(np.complex128), oracle.r2c_2d(xs[b], ny)) <= TOL[prec], b
    assert torch.equal(out[:, :nx, :nc], got)
    out[:, :nx, :nc] = complex(7, 7)
    assert bool((out == complex(7, 7)).all())   # nothing beyond the grids
    # backward, reals in the padded pitch
    Y = torch.randn((batch, nx, nc), dtype=torch.complex128, device="cuda").to(cdt)
    Yr = Y.cpu().numpy().astype(np.complex128)
    for exec_, ref in ((q.exec_adjoint, oracle.adjoint_r2c_2d), (q.exec_c2r, oracle.c2r_2d)):
        r = torch.full((batch, nx, 2 * nc), 7.0, dtype=rdt, device="cuda")
        exec_(Y.data_ptr(), r.data_ptr())
        torch.cuda.synchronize()
        for b in range(batch):
            assert oracle.rel_l2(r[b, :, :ny].cpu().numpy().astype(np.float64), ref(Yr[b], ny)) <= TOL[prec], b
        assert bool((r[:, :, ny:] == 7).all())
    p.close()
    q.close()


@pytest.mark.parametrize("n,prec", CASES)
def test_rows(gpu, n, prec):
    _check(5, 2 * n, prec)


@pytest.mark.parametrize("n,prec", CASES)
def test_columns(gpu, n, prec):
    _check(n, 34, prec)   # 18 columns


@pytest.mark.parametrize("nx,ny,batch,prec", [(67, 134, 3, "f64"), (131, 1018, 2, "f32"), (1021, 134, 2, "f64"),
                                              (17, 254, 3, "f32")])
def test_both_and_batched(gpu, nx, ny, batch, prec):
    _check(nx, ny, prec, batch)
