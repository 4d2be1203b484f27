"""Batched one-token launches over uint4 weights: the rule between the contiguous-strip kernel and the streaming one."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from test_gpu_batch_ids import check as check_batch, run_device
from test_oracle_fc import make_batch_ids_case


# one token, 128 strips x rows and more: the contiguous-strip kernel; fewer: the streaming one
@pytest.mark.parametrize("rows,src_rows,k,n,batch", [(2, 1, 2048, 4096, 8), (1, 1, 512, 8192, 2), (8, 8, 768, 1024, 4), (3, 3, 4096, 2816, 5),
                                                     (127, 1, 96, 64, 7)])
def test_batched_strips(oracle, rows, src_rows, k, n, batch):
    c = make_batch_ids_case(rows + k, rows, 1, src_rows, k, n, batch, 4, k // 32, False)
    got, name = run_device(c, np.float16, group=16)
    assert name == ("fc_w4_strip_kernel" if n // 64 * rows >= 128 else "fc_w4_stream_kernel"), name
    check_batch(c, np.float16, got, oracle)


# the streaming kernel's half strips, two of a 64-channel strip on one XCD: one half, an odd count, one strip per row, more pairs
# than XCDs, output groups of 16 slices and one group, channels that end inside a half
@pytest.mark.parametrize("rows,src_rows,k,n,batch,group", [(1, 1, 256, 32, 3, 0), (5, 1, 256, 96, 4, 0), (7, 7, 512, 64, 8, 16), (9, 1, 2080, 160, 3, 0),
                                                           (3, 3, 96, 1000, 4, 0), (8, 1, 2048, 768, 16, 16), (11, 1, 64, 72, 5, 0)])
@pytest.mark.parametrize("zp", [False, True])
def test_batched_half_strips(oracle, rows, src_rows, k, n, batch, group, zp):
    c = make_batch_ids_case(rows + k, rows, 1, src_rows, k, n, batch, 4, k // 32, zp)
    got, name = run_device(c, np.float16, **({"group": group} if group else {}))
    assert name == "fc_w4_stream_kernel", name
    check_batch(c, np.float16, got, oracle)
