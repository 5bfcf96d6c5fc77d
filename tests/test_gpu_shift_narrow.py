"""The partial sums' shifted rows of odd widths below 513 whole vectors
(hprms.hip, shift_phase): on both sides of the first width, the widest, and
widths whose last slots lie past the row; several rows per workgroup, each
with a shift of its own.  With every stream at one phase (shifted) and at
phases of their own (not shifted), 3 and 8 parts.  Against the oracle, at the
usual bar, with nothing written outside the rows."""
import pytest
import torch

from helpers import DT, assert_output_close, assert_residual_exact, bits, make_inputs
from oracle import oracle
from test_gpu_unaligned import View, abi  # noqa: F401  (the fixture)

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
EPS = 1e-6


def run_case(abi, rows, hidden, dtype, nparts, out_at, res_at, parts_at):  # noqa: F811
    """`*_at`: (element offset, row padding) of a stream; parts_at: of each part
    (one row padding for all)."""
    x, r, w = make_inputs(rows, hidden, dtype, seed=hidden + rows)
    th = min(16, oracle.max_threads())
    st = torch.cuda.current_stream().cuda_stream
    wd = w.to(DEV)
    parts = [torch.randn((rows, hidden), generator=torch.Generator().manual_seed(i)).to(dtype) for i in range(nparts)]
    pad = max(off + p for off, p in parts_at)
    pvs = [View(p, off, pad - off) for p, (off, _) in zip(parts, parts_at)]
    rv, ov = View(r, *res_at), View(torch.zeros_like(x), *out_at)
    assert len({v.stride for v in pvs}) == 1
    abi.reduce_add_rmsnorm(ov.ptr, [p.ptr for p in pvs], wd.data_ptr(), rv.ptr, rows, hidden, ov.stride,
                           pvs[0].stride, rv.stride, DT[dtype], EPS, st)
    torch.cuda.synchronize()
    p_out, p_res = oracle.reduce_add_rmsnorm([bits(p) for p in parts], bits(w), bits(r), EPS, DT[dtype], threads=th)
    assert_residual_exact(bits(rv.view), p_res, dtype)
    assert_output_close(bits(ov.view), p_out, dtype)
    for v in (ov, rv):
        v.check_outside("rows")


HIDDENS = [951, 961, 967, 1441, 1921, 2503, 3079, 4095, 4103]


@pytest.mark.parametrize("hidden", HIDDENS)
@pytest.mark.parametrize("dtype,rows,off,pad", [(torch.bfloat16, 5, 0, 0), (torch.float16, 1300, 0, 0),
                                                (torch.bfloat16, 300, 3, 5)])
def test_partial_sums_shift_narrow_rows_of_odd_widths(abi, hidden, dtype, rows, off, pad):  # noqa: F811
    print("narrow shifted rows", rows, hidden, dtype, off, pad, flush=True)
    for nparts in (3, 8):
        run_case(abi, rows, hidden, dtype, nparts, (off, pad), (off, pad), [(off, pad)] * nparts)


@pytest.mark.parametrize("hidden", HIDDENS)
@pytest.mark.parametrize("dtype,rows", [(torch.bfloat16, 5), (torch.float16, 300), (torch.bfloat16, 1300)])
def test_partial_sums_of_narrow_rows_at_phases_of_their_own(abi, hidden, dtype, rows):  # noqa: F811
    """The residual, one part or the row pitch away from the output's phase."""
    print("narrow rows, unequal phases", rows, hidden, dtype, flush=True)
    for nparts in (3, 8):
        at = [(0, 0)] * nparts
        run_case(abi, rows, hidden, dtype, nparts, (0, 0), (3, 5), [(0, 8)] * nparts)
        run_case(abi, rows, hidden, dtype, nparts, (0, 8), (0, 8), at[:-1] + [(5, 3)])
        run_case(abi, rows, hidden, dtype, nparts, (0, 0), (0, 0), [(0, 2)] * nparts)
