"""Batched one-token launches of the streaming int4 kernel whose activations are read in whole chunks (one shared source row) or row by
row (a source row of its own for each matrix): one chunk, the last of a step's 64, the first of a second step, full and
ragged second and third steps, both strip widths.  Group-wise scales always come with whole chunks of K-slices (the launcher asks for
them), so the number of source rows is what chooses."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from test_gpu_batch_ids import check, run_device
from test_oracle_fc import make_batch_ids_case


# strips of 64 channels from 192 strips x rows on, half strips below; groups of 32 (the reference's one output group: never the strip kernel)
@pytest.mark.parametrize("rows,src_rows,k,n,batch", [(1, 1, 32, 64, 2), (1, 1, 64, 64, 2), (3, 1, 2016, 96, 4), (2, 1, 2048, 160, 3), (4, 1, 2080, 72, 5), (4, 4, 2080, 72, 5),
                                                     (2, 1, 4160, 104, 3), (48, 1, 2112, 256, 3), (48, 48, 2112, 256, 3), (48, 1, 64, 256, 4)])
@pytest.mark.parametrize("zp", [False, True])
def test_whole_rows(oracle, rows, src_rows, k, n, batch, zp):
    print("whole rows", rows, src_rows, k, n, batch, zp, flush=True)
    c = make_batch_ids_case(rows + k, rows, 1, src_rows, k, n, batch, 4, k // 32, zp)
    ops = []
    got, name = run_device(c, np.float16, ops=ops)
    # (one group is per-channel scales, whose kernels mask every load)
    assert (name, ops[0].kernel_whole) == ("fc_w4_stream_kernel", src_rows == 1 and k > 32), name
    check(c, np.float16, got, oracle)


# K that ends inside a chunk, which only per-channel scales allow: their kernels mask every load
@pytest.mark.parametrize("k", [36, 2060])
def test_ragged_chunk(oracle, k):
    c = make_batch_ids_case(k, 3, 1, 1, k, 96, 4, 4, 1, False)
    ops = []
    got, name = run_device(c, np.float16, ops=ops)
    assert (name, ops[0].kernel_whole) == ("fc_w4_stream_kernel", False), name
    check(c, np.float16, got, oracle)
