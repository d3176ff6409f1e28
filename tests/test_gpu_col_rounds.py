"""The width of one-launch columns of 4096 rows: 512 threads with half the columns where
the wide form's last round over the 256 CUs is the first and at most half full, or the
second and at most an eighth (FP64) or half (FP32) full.  Numbers of wide strips (4 FP64
or 8 FP32 columns) on both sides of each edge: the plan text, and the transform against
the oracle (FP64 <= 1e-12, FP32 <= 1e-5, the bounds of the other parity tests)."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

EDGES = [(1, 512), (128, 512), (129, 1024), (256, 1024), (257, 512), (513, 1024)]
CASES = [(s, t, p) for s, t in EDGES for p in ("f64", "f32")] + [
    (288, 512, "f64"), (289, 1024, "f64"), (384, 512, "f32"), (385, 1024, "f32")]


@pytest.mark.parametrize("strips,threads,prec", CASES)
def test_width(gpu, strips, threads, prec):
    import torch
    import hpxfft_amd
    nx, wide = 4096, 4 if prec == "f64" else 8
    ny = 2 * (strips * wide - 1)
    print(f"long columns {prec} {nx}x{ny}: {strips} wide strips", flush=True)
    p = hpxfft_amd.Plan(nx, ny, precision=prec)
    text = p.describe()
    w = wide * threads // 1024
    assert f"4096-point, {w} adjacent columns x all rows in registers, {threads} threads" in text, text
    x = oracle.fill(nx, ny, seed=strips, dist="normal")
    rdt, cdt = (torch.float64, torch.complex128) if prec == "f64" else (torch.float32, torch.complex64)
    d = torch.from_numpy(x).to(device="cuda", dtype=rdt)
    p.exec(d.data_ptr(), d.data_ptr())
    torch.cuda.synchronize()
    p.close()
    err = oracle.rel_l2(d.view(cdt).cpu().numpy().astype(np.complex128), oracle.r2c_2d(x, ny))
    assert err <= (1e-12 if prec == "f64" else 1e-5), err


@pytest.mark.parametrize("strips,batch,threads", [(32, 4, 512), (43, 3, 1024), (96, 3, 512), (97, 3, 1024)])
def test_width_counts_the_batch(gpu, strips, batch, threads):
    import hpxfft_amd
    p = hpxfft_amd.Plan(4096, 2 * (strips * 4 - 1), batch=batch, precision="f64")
    text = p.describe()
    p.close()
    assert f"in registers, {threads} threads" in text, text
