"""GPU parity of the packed-groups GEMM's tile numbering and wave counts: a launch has one token tile for every
tile's worth of tokens plus one per group, found on the device from the group sizes, and 1, 2, 4 or 8 waves
share the K of a tile.  More groups than a wave counts at a time, empty ones between, one group with nearly every
token, sizes around the tile edges, and shapes that reach every (token tile, wave count) pair; against the
per-matrix float64 product."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

import mldhip as M
import workloads as W
from test_gpu_packed_groups import run_device
from test_oracle_fc import batch_ids_float_weights, make_packed_groups_case


def run(oracle, sizes, k, n, bits=4, groups=1, zp=False, max_group=None, group=None, seed=1, gap=0):
    sizes = np.asarray(sizes, np.int32)
    offsets = (np.cumsum(sizes) - sizes + gap * np.arange(len(sizes))).astype(np.int32)
    tokens = int(sizes.sum()) + gap * len(sizes)
    c = make_packed_groups_case(seed, tokens, 1, k, n, len(sizes), bits, groups, zp)
    got = run_device(c, np.float16, sizes=sizes, offsets=offsets, max_group_size=max_group or tokens, fill=7.0, group=group)
    wf = batch_ids_float_weights(oracle, c).astype(np.float64)
    src = c["packed_src"].astype(np.float16).astype(np.float64)
    limit = max_group or tokens
    for g, (s, off) in enumerate(zip(sizes, offsets)):
        live = slice(int(off), int(off) + min(int(s), limit))
        ref = src[live] @ wf[:, g, :].T
        # weights are rounded to fp16 (2^-11 relative, twice with a zero point), results once more; sums in fp32
        tol = 2.0 ** -10 * (np.abs(src[live]) @ np.abs(wf[:, g, :]).T) / np.sqrt(k) * 4 + 2.0 ** -10 * np.abs(ref) + 1e-6
        assert np.all(np.abs(got[live] - ref) <= tol), (g, s)
        assert np.all(got[live.stop:int(off) + int(s)] == 7.0)
    if gap:
        for g in range(len(sizes)):
            end = int(offsets[g] + sizes[g])
            assert np.all(got[end:end + gap] == 7.0), g


@pytest.mark.parametrize("sizes", [
    [0] * 66 + [1, 0, 31, 32, 33, 0, 64, 65],                       # the first 64 groups are empty
    [1] * 130,                                                      # three countings, every group one tile
    [3, 700, 0, 2, 1],                                              # nearly everything in one group
    list(range(40, 140)),                                           # one and two (128-token: one and two) tiles each
    [600, 1, 520, 640],                                             # 128-token tiles
])
@pytest.mark.parametrize("gap", [0, 1])
def test_tile_numbering(oracle, sizes, gap):
    run(oracle, sizes, 64, 132, seed=len(sizes), gap=gap)


# 64, 256, 1024 and 8192 input channels: 1, 2, 4 and 8 waves where tiles are few
@pytest.mark.parametrize("sizes,k,n", [
    ([18, 0, 20, 5], 64, 128), ([16] * 20, 256, 388), ([9, 12], 1024, 256), ([20, 3], 8192, 128),  # 32-token tiles
    ([40] * 12, 64, 256), ([40] * 12, 256, 260), ([64, 65], 1024, 256), ([33, 90], 8192, 132),     # 64-token tiles
    ([530, 600], 64, 640), ([515, 700], 256, 132), ([513, 600], 1024, 260),                         # 128-token tiles, up to 4 waves
])
@pytest.mark.parametrize("bits,zp", [(4, False), (4, True), (8, False)])
def test_wave_counts(oracle, sizes, k, n, bits, zp):
    run(oracle, sizes, k, n, bits=bits, groups=2 if bits == 4 else 1, zp=zp, seed=k + n)


def test_largest_group_bound(oracle):
    run(oracle, [70, 5, 90, 33], 128, 128, max_group=64)


@pytest.mark.parametrize("groups,n,k", [(16384, 4100, 16), (2048, 64, 32)])
def test_many_small_groups(groups, n, k):
    """Every token a group of its own: 16384 token tiles x 33 channel tiles are more than 2^16 per XCD.  Matrix g holds one
    code in every place and each channel a scale of its own, small enough that every result is exact."""
    import torch
    g = torch.arange(groups, device="cuda")
    ns = W.div_up(n, 4)
    desc = M.fc_int4_weights_desc(n, k, reference=True)
    assert M.packed_bytes(desc, n, groups, 1, k) == groups * W.div_up(k, 4) * ns * 8
    code = (g % 16).to(torch.uint8)
    weights = (code * 17).repeat_interleave(W.div_up(k, 4) * ns * 8)  # (one matrix after the other)
    channel_scale = (1 + torch.arange(ns * 4, device="cuda") % 7).half() / 64
    scale = channel_scale.repeat(groups)
    act = torch.randint(-2, 3, (groups, k), device="cuda").half()
    src = act.view(groups, k // 4, 4).transpose(0, 1).contiguous()
    params = torch.cat([torch.ones_like(g), g]).to(torch.int32)
    out = torch.full((ns, groups, 4), 7.0, dtype=torch.float16, device="cuda")
    op = M.fc_create(M.PRECISION_F32_F16, M.FLOAT16, M.FLOAT16, n, k, desc, scale_shape=(n, 1), max_tokens=groups, packed_groups=(0, groups, 1))
    op.bind([src, weights, scale, params], [out])
    op.set_shape(1, 1, groups)
    print("packed groups", groups, n, k, flush=True)
    op.launch(torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert op.kernel_name == "fc_w4_mfma_gemm_kernel"
    got = out.transpose(0, 1).reshape(groups, ns * 4)[:, :n].float()
    sums = act.float().sum(dim=1) * (code.float() - 8)
    assert torch.equal(got, sums[:, None] * channel_scale.float()[None, :n])


# every form of the launch (tokens of a tile x waves that share its K)
@pytest.mark.parametrize("sizes,k,n,form", [
    ([3] * 20, 64, 516, "32x1"), ([3] * 20, 256, 260, "32x2"), ([12, 20, 4] * 4, 512, 388, "32x4"), ([9, 0, 3], 4096, 128, "32x8"),
    ([30, 0, 31, 33, 64, 20, 32, 40, 30, 20], 64, 516, "64x1"), ([40] * 12, 256, 260, "64x2"), ([40, 100, 3], 1024, 132, "64x4"),
    ([40, 100, 3], 4096, 132, "64x8"), ([530, 600], 64, 640, "128x1"), ([515, 700], 256, 132, "128x2"), ([513, 600], 1024, 260, "128x4")])
@pytest.mark.parametrize("bits", [4, 8])
def test_forms(oracle, monkeypatch, sizes, k, n, form, bits):
    ops, create = [], M.fc_create
    monkeypatch.setattr(M, "fc_create", lambda *a, **kw: ops.append(create(*a, **kw)) or ops[-1])
    run(oracle, sizes, k, n, bits=bits, seed=k + n)
    assert ops[-1].kernel_variant == "packed " + form


# a 32-token tile for every CU and more
@pytest.mark.parametrize("sizes,k,n,form", [
    ([8] * 40, 256, 1000, "32x4"), ([5] * 90, 512, 388, "32x4"), ([6, 0] * 70, 128, 772, "32x1"), ([9, 1, 20] * 30, 64, 900, "32x1")])
@pytest.mark.parametrize("bits,zp", [(4, False), (4, True), (8, False)])
def test_forms_of_many_small_groups(oracle, monkeypatch, sizes, k, n, form, bits, zp):
    ops, create = [], M.fc_create
    monkeypatch.setattr(M, "fc_create", lambda *a, **kw: ops.append(create(*a, **kw)) or ops[-1])
    run(oracle, sizes, k, n, bits=bits, groups=2 if bits == 4 else 1, zp=zp, seed=k + n)
    assert ops[-1].kernel_variant == "packed " + form


# token tiles on the XCDs: as many as XCDs and one more, fewer, all in one group, more groups than tokens; channel tiles 1, 2, 9, 18
@pytest.mark.parametrize("sizes", [[1] * 9, [1] * 8, [0, 2, 0], [0] * 30 + [3] + [0] * 30, [40, 33, 0, 64, 1, 65, 70, 40, 2], [300]])
@pytest.mark.parametrize("n", [100, 256, 1152, 2244])
def test_tiles_over_the_xcds(oracle, sizes, n):
    run(oracle, sizes, 64, n, seed=n + len(sizes))
