"""The quantised outputs at the edges of their table's rows from 12K up: the
first and last width of each lane shape (slots wholly past the row, slots
partly past it, exact fits), one row, and a row count past one per CU.  Bit
for bit against the quantisation of the 16-bit op's own output and within the
oracle's bar, as in the forms' own test files, whose checks this runs."""
import pytest
import torch

import test_gpu_fp8
import test_gpu_fp8_group
import test_gpu_mx
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
