"""Batched column tasks of 32 points per thread (grids of 1024 and 2048 rows, task
shape 0): 33 to 1025 columns, one past a whole number of the tasks' 16 or 8, among
grids whose tasks hold 16 points per thread, against the FP64 oracle (FP32 <= 1e-5,
the bound of the other parity tests)."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [([1024], [64]), ([2048], [64]), ([1024, 512, 2048, 64], [2048, 256, 128, 64]),
                                   ([512, 1024, 2048], [64, 128, 2048])])
def test_long_columns(gpu, nx, ny):
    import torch
    import hpxfft_amd
    print(f"batched long columns {nx} {ny}", flush=True)
    xs = [oracle.fill(a, b, seed=a + b, dist="normal") for a, b in zip(nx, ny)]
    ds = [torch.from_numpy(x).to(device=gpu, dtype=torch.float32) for x in xs]
    plan = hpxfft_amd.BatchedPlan(nx, ny)
    plan.set_config(0, 0)
    plan.exec([d.data_ptr() for d in ds])
    torch.cuda.synchronize()
    plan.close()
    for x, d, b in zip(xs, ds, ny):
        got = d.cpu().numpy().astype(np.float64).view(np.complex128)
        assert oracle.rel_l2(got, oracle.r2c_2d(x, b)) <= 1e-5
