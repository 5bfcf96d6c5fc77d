"""The partial sums' shifted rows of odd widths below 513 whole vectors
(hprms.hip, shift_phase): on both sides of the first width, the widest, and
widths whose last slots lie past the row; several rows per workgroup, each
with a shift of its own.  Against the oracle, at the usual bar, with nothing
written outside the rows."""
import pytest
import torch

from helpers import DT, assert_output_close, assert_residual_exact, bits, make_inputs
from oracle import oracle
from test_gpu_unaligned import View, abi  # noqa: F401  (the fixture)

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
EPS = 1e-6


@pytest.mark.parametrize("hidden", [951, 961, 967, 1441, 1921, 2503, 3079, 4095, 4103])
@pytest.mark.parametrize("dtype,rows,off,pad", [(torch.bfloat16, 5, 0, 0), (torch.float16, 1300, 0, 0),
                                                (torch.bfloat16, 300, 3, 5)])
def test_partial_sums_shift_narrow_rows_of_odd_widths(abi, hidden, dtype, rows, off, pad):  # noqa: F811
    print("narrow shifted rows", rows, hidden, dtype, off, pad, flush=True)
    x, r, w = make_inputs(rows, hidden, dtype, seed=hidden + rows)
    th = min(16, oracle.max_threads())
    st = torch.cuda.current_stream().cuda_stream
    wd = w.to(DEV)
    z = torch.zeros_like(x)

    def view(t):
        return View(t, off, pad)

    parts = [torch.randn((rows, hidden), generator=torch.Generator().manual_seed(i)).to(dtype) for i in range(3)]
    pvs, rv, ov = [view(p) for p in parts], view(r), view(z)
    abi.reduce_add_rmsnorm(ov.ptr, [p.ptr for p in pvs], wd.data_ptr(), rv.ptr, rows, hidden, ov.stride,
                           pvs[0].stride, rv.stride, DT[dtype], EPS, st)
    torch.cuda.synchronize()
    p_out, p_res = oracle.reduce_add_rmsnorm([bits(p) for p in parts], bits(w), bits(r), EPS, DT[dtype], threads=th)
    assert_residual_exact(bits(rv.view), p_res, dtype)
    assert_output_close(bits(ov.view), p_out, dtype)
    for v in (ov, rv):
        v.check_outside("rows")
