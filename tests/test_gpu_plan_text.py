"""The plan text gives the shapes of the kernels that are launched: a Bluestein length
that runs in registers (the in-LDS form it replaces named as such), batched column tasks."""
import pytest

pytestmark = pytest.mark.gpu


# length, convolution length, last radix (1: none), rows and columns per workgroup with their threads.  A thread
# holds 16 points (FP64) or, of long FP32 sequences, 32; columns of 2^8 (FP64) fill a 128-byte segment
@pytest.mark.parametrize("n,prec,conv,last,rows,row_nt,cols,col_nt", [
    (2039, "f64", 4096, 1, 1, 256, 2, 512), (2039, "f32", 4096, 1, 1, 256, 4, 512),
    (67, "f64", 256, 1, 8, 128, 8, 128), (1021, "f32", 2048, 8, 1, 128, 8, 512),
    (4093, "f64", 8192, 2, 1, 512, 2, 1024), (8191, "f32", 16384, 4, 1, 512, 2, 1024)])
def test_plan_text(gpu, n, prec, conv, last, rows, row_nt, cols, col_nt):
    import hpxfft_amd
    p = hpxfft_amd.Plan(n, 2 * n, precision=prec)
    text = p.describe()
    p.close()
    how = (f"{n}-point Bluestein in registers (two {conv}-point transforms, radix 16" +
           (f", last stage radix {last}" if last > 1 else "") + ", LDS exchange in re/im halves)")
    row, col = (next(l for l in text.splitlines() if l.startswith(k)) for k in ("  row r2c", "  column c2c"))
    assert f"{how}, {row_nt} threads, {rows} row(s)/workgroup + r2c split; the in-LDS form it replaces: " in row, text
    assert f"{how}, {col_nt} threads, {cols} adjacent columns/workgroup; the in-LDS form it replaces: " in col, text


@pytest.mark.parametrize("cfg,text", [(0, "(8192 points per task, 16384 on grids of 1024 and 2048 rows, "),
                                      (1, "(4096 points per task, 34 tasks"), (3, "(16384 points per task, 10 tasks")])
def test_batched_column_tasks(gpu, cfg, text):
    """One grid of 64 x 2048 and one of 1024 x 128: 1025 and 65 columns."""
    import hpxfft_amd
    p = hpxfft_amd.BatchedPlan([64, 1024], [2048, 128])
    p.set_config(0, cfg)
    line = next(l for l in p.describe().splitlines() if l.startswith("  column phase"))
    p.close()
    assert text in line, line
    tasks = {0: 9 + 5, 1: 17 + 17, 3: 5 + 5}[cfg]   # strips of PTS / rows columns, 16 of 1024 rows in shape 0
    assert f"{tasks} tasks" in line, line
