"""The quantised outputs at the edges of their table's rows from 12K up: the
first and last width of each lane shape (slots wholly past the row, slots
partly past it, exact fits), one row, and a row count past one per CU.  Bit
for bit against the quantisation of the 16-bit op's own output and within the
oracle's bar, as in the forms' own test files, whose checks this runs.  The
tail and unaligned variants of the same shapes (odd widths, rows off the
128-byte grid) against the oracle, with nothing written outside the rows."""
import pytest
import torch

import test_gpu_fp8
import test_gpu_fp8_group
import test_gpu_mx
import test_gpu_random_fp8_forms
import test_gpu_random_shapes
from oracle import oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    assert torch.cuda.is_available(), "the gpu tests need a HIP device"
    import hp_rms_norm_amd
    return hp_rms_norm_amd


WIDTHS = [12416, 14336, 14464, 16256, 16384, 16512, 20480, 20608, 24704]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("hidden", WIDTHS)
@pytest.mark.parametrize("rows", [1, 300])
def test_quantised_outputs_at_the_edges_of_their_shapes(ops, rows, hidden, dtype):
    print("quant edges", rows, hidden, dtype, flush=True)
    test_gpu_fp8.run_case(ops, rows, hidden, dtype, seed=hidden + rows)
    test_gpu_fp8_group.run_case(ops, rows, hidden, dtype, seed=hidden + rows)
    test_gpu_mx.run_case(ops, rows, hidden, dtype, oracle.MXFP8, seed=hidden + rows)
    test_gpu_mx.run_case(ops, rows, hidden, dtype, oracle.MXFP4, seed=hidden + rows)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("rows,hidden", [(769, 3200), (768, 4096), (769, 4096), (257, 4224), (257, 5120), (256, 5248),
                                         (257, 5248), (300, 8064), (4096, 8192)])
def test_quantised_outputs_with_the_weight_loaded_with_the_row(ops, rows, hidden, dtype):
    """3K-8K: the first and last widths and the first row counts of the shapes
    that load the weight early, and the last of those that load it late."""
    test_quantised_outputs_at_the_edges_of_their_shapes(ops, rows, hidden, dtype)


# odd widths and rows off the grid at the first and last width of 512 x 4, 5
# and 6, and the LDS tier's first: (element offsets, row padding) per stream
LAYOUTS = [([0] * 6, [0] * 6), ([1, 3, 8, 13, 0, 1], [5, 1, 0, 120, 8, 0])]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("hidden", [12297, 14337, 16383, 16391, 18433, 20487, 20489, 22529, 24583, 24585])
@pytest.mark.parametrize("rows", [1, 300])
def test_fp8_rows_of_odd_widths(ops, rows, hidden, dtype):
    from hp_rms_norm_amd import abi
    print("quant odd width", rows, hidden, dtype, flush=True)
    for k, (offs, pads) in enumerate(LAYOUTS):
        test_gpu_random_shapes.run_case(abi, hidden + rows + k, dict(
            hidden=hidden, rows=rows, dtype=dtype, offs=offs, pads=pads, mode=2, eps=1e-6, dist="bench"))
        test_gpu_random_fp8_forms.run_case(abi, hidden + rows + k, dict(
            form="static", hidden=hidden, rows=rows, dtype=dtype, offs=offs, pads=pads, eps=1e-6, special=False,
            scale=0.01))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("hidden", WIDTHS)
@pytest.mark.parametrize("rows", [1, 300])
def test_quantised_outputs_off_the_grid(ops, rows, hidden, dtype):
    from hp_rms_norm_amd import abi
    print("quant off grid", rows, hidden, dtype, flush=True)
    offs, pads = LAYOUTS[1]
    for mode in (2, 5, 6):
        test_gpu_random_shapes.run_case(abi, hidden + rows + mode, dict(
            hidden=hidden, rows=rows, dtype=dtype, offs=offs, pads=pads, mode=mode, eps=1e-6, dist="bench"))
    test_gpu_random_fp8_forms.run_case(abi, hidden + rows, dict(
        form="group", hidden=hidden, rows=rows, dtype=dtype, offs=offs, pads=pads, eps=1e-6, special=False, scale=1.0))
