"""The four-step scratch of plans whose columns run as one launch (2^11 and 2^12
rows, FP64 / FP32): none until a split is set, and none kept by the measure effort
when it chooses the one launch.  Device memory is read around the planning call,
with every per-device table in place."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

MIB = 1 << 20


def _used(torch):
    torch.cuda.synchronize()
    free, total = torch.cuda.mem_get_info()
    return total - free


@pytest.mark.parametrize("effort", ["estimate", "measure"])
@pytest.mark.parametrize("nx,ny,batch,prec", [(2048, 2048, 8, "f64"), (4096, 4096, 4, "f32")])
def test_scratch_only_where_the_four_step_runs(gpu, nx, ny, batch, prec, effort):
    import torch
    import hpxfft_amd
    print(f"scratch {prec} {batch} x {nx}x{ny} {effort}", flush=True)
    spectrum = batch * nx * (ny // 2 + 1) * (16 if prec == "f64" else 8)   # 269 and 269 MB
    warm = hpxfft_amd.Plan(nx, 64, precision=prec)
    before = _used(torch)
    p = hpxfft_amd.Plan(nx, ny, batch=batch, precision=prec, effort=effort)
    planned = _used(torch) - before
    one_launch = effort == "estimate" or "in registers" in p.describe()
    assert planned < 32 * MIB if one_launch else planned >= spectrum, planned
    p.set_column_split(6)
    assert _used(torch) - before >= spectrum
    p.close()
    warm.close()


@pytest.mark.parametrize("prec,tol", [("f64", 1e-12), ("f32", 1e-5)])
def test_split_set_after_an_exec(gpu, prec, tol):
    """The scratch comes with the first split: an exec before it, and one after, give the same transform."""
    import torch
    import hpxfft_amd
    nx, ny = 4096, 66
    x = oracle.fill(nx, ny, seed=11, dist="normal")
    ref = oracle.r2c_2d(x, ny)
    cdt, rdt = (torch.complex128, torch.float64) if prec == "f64" else (torch.complex64, torch.float32)
    p = hpxfft_amd.Plan(nx, ny, precision=prec)
    for split in (None, 5, 6):
        if split is not None:
            p.set_column_split(split)
        d = torch.from_numpy(x).to(device="cuda", dtype=rdt)
        p.exec(d.data_ptr(), d.data_ptr())
        torch.cuda.synchronize()
        assert (p.measurement("column_a") > 0.0) == (split is not None)
        assert oracle.rel_l2(d.view(cdt).cpu().numpy().astype(np.complex128), ref) <= tol
    p.close()
