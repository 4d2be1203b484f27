"""Batched one-token launches of the streaming int4 kernel whose activations are read in whole chunks (one shared source row) or row by
row (a source row of its own for each matrix): one chunk, the last of a step's 64, the first of a second step, full and
ragged second and third steps, K-slices that are no whole chunk, both strip widths."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from test_gpu_batch_ids import check, run_device
from test_oracle_fc import make_batch_ids_case


# strips of 64 channels from 192 strips x rows on, half strips below; groups of 32 (the reference's one output group: never the strip kernel)
@pytest.mark.parametrize("rows,src_rows,k,n,batch", [(1, 1, 32, 64, 2), (3, 1, 2016, 96, 4), (2, 1, 2048, 160, 3), (4, 1, 2080, 72, 5), (4, 4, 2080, 72, 5),
                                                     (2, 1, 4160, 104, 3), (48, 1, 2112, 256, 3), (48, 48, 2112, 256, 3), (48, 1, 64, 256, 4)])
@pytest.mark.parametrize("zp", [False, True])
def test_whole_rows(oracle, rows, src_rows, k, n, batch, zp):
    print("whole rows", rows, src_rows, k, n, batch, zp, flush=True)
    c = make_batch_ids_case(rows + k, rows, 1, src_rows, k, n, batch, 4, k // 32, zp)
    got, name = run_device(c, np.float16)
    assert name == "fc_w4_stream_kernel", name
    check(c, np.float16, got, oracle)


# K that ends inside a chunk stays on the masked loads
@pytest.mark.parametrize("k", [36, 2060])
def test_ragged_chunk(oracle, k):
    c = make_batch_ids_case(k, 3, 1, 1, k, 96, 4, 4, 1, False)
    got, name = run_device(c, np.float16)
    assert name == "fc_w4_stream_kernel", name
    check(c, np.float16, got, oracle)
