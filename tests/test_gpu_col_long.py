"""Columns of 2^11 and 2^12 points in one launch (FP64 / FP32).

Shapes sit where the kernel can go wrong: one column, strips of W - 1, W and
W + 1 columns (W = 4 for FP64 and 8 for FP32 at 2^11 rows; 2 / 4 or 4 / 8 at
2^12, by the launch's thread count), and numbers of strips on both sides of
the rule that picks 512 or 1024 threads.  Forward in place and out of place,
strided batches, the adjoint and c2r, against the FP64 oracle (FP64 <= 1e-12,
FP32 <= 1e-5, the bounds of the other parity tests); the four-step that
hpxfft_plan_set_column_split forces on the same plan gives the same.
"""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

TOL = {"f64": 1e-12, "f32": 1e-5}


def _dt(prec):
    import torch
    return (torch.float64, torch.complex128) if prec == "f64" else (torch.float32, torch.complex64)


@pytest.mark.parametrize("prec", ["f64", "f32"])
# ny / 2 + 1 columns: 2, 4, 5, 8, 9, 17; 4096 x 770 (386 columns: 97 FP64 strips, the first 1024-thread FP64
# grid), 4096 x 768 (385), 4096 x 2048 (1025: 257 wide FP64 strips), 4096 x 2310 (1156: 289)
@pytest.mark.parametrize("nx,ny", [(2048, 2), (2048, 6), (2048, 8), (2048, 14), (2048, 16), (4096, 2), (4096, 8),
                                   (4096, 14), (4096, 16), (4096, 32), (4096, 768), (4096, 770), (4096, 2048),
                                   (4096, 2310)])
def test_forward(gpu, nx, ny, prec):
    import torch
    import hpxfft_amd
    print(f"long columns {prec} {nx}x{ny}", flush=True)
    rdt, cdt = _dt(prec)
    x = oracle.fill(nx, ny, seed=nx + ny, dist="normal")
    ref = oracle.r2c_2d(x, ny)
    nc = ny // 2 + 1
    d = torch.from_numpy(x).to(device="cuda", dtype=rdt)
    out = torch.full((nx, nc + 3), complex(7, 7), dtype=cdt, device="cuda")   # a pitch of its own
    p = hpxfft_amd.Plan(nx, ny, precision=prec, ld_in=d.shape[1], ld_out=nc + 3)
    p.exec(d.data_ptr(), out.data_ptr())
    q = hpxfft_amd.Plan(nx, ny, precision=prec)
    assert "columns x all rows in registers" in q.describe()
    assert q.measurement("column_a") == 0.0
    q.exec(d.data_ptr(), d.data_ptr())
    torch.cuda.synchronize()
    p.close()
    q.close()
    inplace = d.view(cdt)[:, :nc]
    err = oracle.rel_l2(inplace.cpu().numpy().astype(np.complex128), ref)
    print(f"  rel-L2 {err:.2e}", flush=True)
    assert err <= TOL[prec]
    assert torch.equal(out[:, :nc], inplace)
    assert bool((out[:, nc:] == complex(7, 7)).all())   # nothing beyond the columns


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("nx,ny,batch", [(2048, 6, 3), (4096, 14, 2), (4096, 514, 2)])
def test_batch_and_backward(gpu, nx, ny, batch, prec):
    import torch
    import hpxfft_amd
    print(f"long columns {prec} {batch} x {nx}x{ny} backward", flush=True)
    rdt, cdt = _dt(prec)
    rng = np.random.default_rng(nx + ny)
    nc = ny // 2 + 1
    Y = rng.standard_normal((batch, nx, nc)) + 1j * rng.standard_normal((batch, nx, nc))
    Yd = torch.from_numpy(Y).to(device="cuda", dtype=cdt)
    Yr = Yd.cpu().numpy().astype(np.complex128)
    x = rng.standard_normal((batch, nx, ny))
    xd = torch.from_numpy(x).to(device="cuda", dtype=rdt)
    xr = xd.cpu().numpy().astype(np.float64)
    X = hpxfft_amd.rfft2(xd).cpu().numpy().astype(np.complex128)
    adj = hpxfft_amd.rfft2_adjoint(Yd, ny).cpu().numpy().astype(np.float64)
    inv = hpxfft_amd.c2r_2d(Yd, ny).cpu().numpy().astype(np.float64)
    hpxfft_amd.clear_plan_cache()
    for b in range(batch):
        assert oracle.rel_l2(X[b], oracle.r2c_2d(xr[b])) <= TOL[prec]
        assert oracle.rel_l2(adj[b], oracle.adjoint_r2c_2d(Yr[b], ny)) <= TOL[prec]
        assert oracle.rel_l2(inv[b], oracle.c2r_2d(Yr[b], ny)) <= TOL[prec]


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("nx,lg", [(2048, 5), (2048, 6), (4096, 5), (4096, 7)])
def test_forced_split(gpu, nx, lg, prec):
    import torch
    import hpxfft_amd
    ny = 66
    rdt, cdt = _dt(prec)
    x = oracle.fill(nx, ny, seed=9, dist="normal")
    d = torch.from_numpy(x).to(device="cuda", dtype=rdt)
    p = hpxfft_amd.Plan(nx, ny, precision=prec)
    p.set_column_split(lg)
    assert "in registers" not in p.describe()
    p.exec(d.data_ptr(), d.data_ptr())
    torch.cuda.synchronize()
    assert p.measurement("column_a") > 0.0
    p.close()
    assert oracle.rel_l2(d.view(cdt).cpu().numpy().astype(np.complex128), oracle.r2c_2d(x, ny)) <= TOL[prec]
