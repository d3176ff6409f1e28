"""rfft2_scaled reads the caller's grid where the kernels can, and copies it where they
cannot: the input stays as it was, and strided, offset, lazily negated and
gradient-carrying inputs give bit for bit what the contiguous grid gives."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
# power-of-two kernels (one launch of columns, four-step), general, Bluestein, beyond one workgroup
@pytest.mark.parametrize("nx,ny", [(64, 128), (1024, 32), (48, 60), (67, 134), (4, 2 * 20000)])
def test_inputs(gpu, nx, ny, dtype):
    import torch
    import hpxfft_amd
    print(f"scaled input {dtype} {nx}x{ny}", flush=True)
    dt = getattr(torch, dtype)
    gen = torch.Generator(device="cuda").manual_seed(nx + ny)
    ld = ny + 2
    x = torch.randn((nx, ld), dtype=dt, device="cuda", generator=gen)
    x[:, ny:] = 0
    keep = x.clone()
    ref, exp = hpxfft_amd.rfft2_scaled(x)
    assert torch.equal(x, keep)
    assert ref.data_ptr() != x.data_ptr() and not ref.requires_grad
    offset = torch.empty(nx * ld + 1, dtype=dt, device="cuda")[1:].view(nx, ld).copy_(x)   # half a complex element in
    wide = torch.empty((nx, ld + 6), dtype=dt, device="cuda")[:, :ld].copy_(x)
    neg = torch._neg_view(x.neg())
    for other in (offset, wide, neg, x.t().contiguous().t(), x.clone().requires_grad_(True)):
        got, e = hpxfft_amd.rfft2_scaled(other)
        assert got.shape == (nx, ld // 2, 2) and got.requires_grad == other.requires_grad
        assert torch.equal(got, ref) and torch.equal(e, exp)
