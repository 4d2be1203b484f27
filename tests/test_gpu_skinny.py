"""The matrix-core kernel for few tokens over uint4 weights: channel tiles of 4, 8 and 16 slices, one and two blocks
of 16 tokens, several token tiles, K cut between work-groups, K tails, ragged channels, zero points, several matrices per launch;
against the float64 product of the dequantized weights."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

import mldhip as M
import workloads as W
from test_gpu_fc import textbook
from test_gpu_gemm import run_w4


def check(got, case):
    # as dequantized, a weight is rounded to fp16 (2^-11 relative, and the zero point's product with the scale once more),
    # the result once; random signs: the errors of a sum grow with the root of the sum of squares
    ref = textbook(case)
    act = case["act"].astype(np.float64)
    assert got.shape == ref.shape
    rms = np.sqrt(np.mean(ref ** 2)) + 1e-9
    assert np.all(np.isfinite(got)) and act.shape[0] == ref.shape[0]
    err = np.abs(got - ref)
    assert np.all(err <= 2.0 ** -10 * np.abs(ref) + 6 * 2.0 ** -10 * rms), float(err.max() / rms)


# channel tiles: 12800 channels = 200 strips (16 slices), 6400 and 6396 (8), fewer (4); K >= 8192: cut in 2, 4 and 8
@pytest.mark.parametrize("m", [5, 16, 17, 32])
@pytest.mark.parametrize("k,n,groups", [(64, 12800, 2), (96, 6400, 1), (250, 6396, 1), (2048, 264, 64), (1000, 4, 1),
                                        (8192, 2052, 64), (9001, 64, 1), (16384, 2048, 128), (2112, 128, 33)])
def test_shapes(m, k, n, groups):
    zp = (k + n) % 3 == 0
    case = W.make_fc_case(seed=m + k, m=m, k=k, n=n, weight_bits=4, tensor_dtype=np.float16, groups=groups, with_bias=m % 2 == 1,
                          with_zero_point=zp)
    print("skinny", m, k, n, groups, zp, flush=True)
    check(run_w4(case), case)


@pytest.mark.parametrize("m", [7, 20, 75])
@pytest.mark.parametrize("k,shapes", [(512, (260, 36, 1024)), (8192, (128, 2048)), (64, (12000, 800, 4))])
def test_several_matrices(m, k, shapes):
    """One launch of several matrices gives what single launches give within rounding, tile ends inside a strip among
    them."""
    cases = [W.make_fc_case(seed=i + m, m=m, k=k, n=n, weight_bits=4, tensor_dtype=np.float16, groups=k // 32) for i, n in enumerate(shapes)]
    for c in cases[1:]:
        c["act"] = cases[0]["act"]
    devs = [W.FcDevice(c) for c in cases]
    for d in devs[1:]:
        d.act = devs[0].act
        srcs = [d.act, d.weights, d.scale]
        d.op.bind(srcs, [d.out])
    import torch
    M.fc_launch_fused([d.op for d in devs], torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    for d, c in zip(devs, cases):
        assert d.op.kernel_name == "fc_w4_mfma_gemm_kernel"
        check(d.result(), c)


# several token tiles: 16, 32 and 64 channels where they make at most 256 work-groups, one more channel than that, the last
# token count, K cut in 4 and not cut far enough, ragged tokens, channels and K
@pytest.mark.parametrize("m,k,n,groups", [(33, 64, 2048, 2), (64, 96, 2052, 1), (97, 250, 1028, 1), (128, 512, 2048, 16), (256, 96, 2048, 3),
                                          (257, 64, 1792, 1), (384, 2112, 1300, 33), (384, 64, 4, 1), (385, 64, 260, 2), (300, 1000, 12, 1),
                                          (64, 8192, 2048, 64), (63, 8192, 2052, 64), (70, 9001, 100, 1)])
def test_token_tiles(m, k, n, groups):
    zp = n % 8 != 0
    case = W.make_fc_case(seed=m + k, m=m, k=k, n=n, weight_bits=4, tensor_dtype=np.float16, groups=groups, with_bias=m % 2 == 1,
                          with_zero_point=zp)
    print("token tiles", m, k, n, groups, zp, flush=True)
    check(run_w4(case), case)


# which kernel a launch takes, and both results: K cut in 1, 2, 4 and 8 and every tile of the kernel; against it two rounds of
# work-groups, a direct kernel cut more often, whole K of 6144 and more above 32 tokens, one batch of short K in whole strips
@pytest.mark.parametrize("m,k,n,zp,form", [
    (16, 64, 2048, True, "skinny 16x16 k1"), (33, 512, 1024, True, "skinny 16x32 k1"), (9, 64, 8192, False, "skinny 32x16 k1"),
    (17, 96, 8100, True, "skinny 32x32 k1"), (12, 544, 16384, False, "skinny 64x16 k1"), (20, 64, 12804, True, "skinny 64x32 k1"),
    (16, 2048, 17000, False, "skinny 64x16 k1"), (7, 8192, 9000, True, "skinny 64x16 k1"), (5, 8192, 5000, False, "skinny 64x16 k2"),
    (32, 8200, 4100, True, "skinny 64x32 k2"), (16, 8192, 4096, False, "skinny 64x16 k4"), (24, 8192, 2052, True, "skinny 64x32 k4"),
    (64, 8192, 2048, False, "skinny 64x32 k4"), (16, 16384, 1024, True, "skinny 64x16 k8"), (30, 16384, 2000, False, "skinny 64x32 k8"),
    (16, 512, 16384, True, "direct"), (20, 64, 16640, False, "direct"), (16, 1504, 17000, False, "direct"), (16, 8192, 17000, False, "direct"),
    (17, 8192, 9000, False, "direct"), (8, 12288, 5000, False, "direct"), (33, 8192, 4096, False, "direct"), (64, 6144, 5000, False, "direct"),
    (385, 64, 260, True, "direct")])
def test_kernel_choice(m, k, n, zp, form):
    case = W.make_fc_case(seed=m + k, m=m, k=k, n=n, weight_bits=4, tensor_dtype=np.float16, groups=k // 32 if k % 32 == 0 else 1,
                          with_bias=m % 2 == 1, with_zero_point=zp)
    print("kernel choice", m, k, n, zp, form, flush=True)
    dev = W.FcDevice(case)
    dev.run()
    got = dev.result()
    assert (dev.op.kernel_name, dev.op.kernel_variant) == ("fc_w4_mfma_gemm_kernel", form)
    check(got, case)


@pytest.mark.parametrize("m,k,shapes,form", [(7, 512, (260, 36, 1024), "skinny 16x16 k1"), (20, 8192, (128, 2048), "skinny 64x32 k4"),
                                             (75, 96, (1500, 800, 4), "skinny 32x32 k1"), (24, 8192, (9000, 4000), "direct")])
def test_several_matrices_with_zero_points(m, k, shapes, form):
    cases = [W.make_fc_case(seed=i + m, m=m, k=k, n=n, weight_bits=4, tensor_dtype=np.float16, groups=k // 32, with_zero_point=True)
             for i, n in enumerate(shapes)]
    for c in cases[1:]:
        c["act"] = cases[0]["act"]
    devs = [W.FcDevice(c) for c in cases]
    for d in devs[1:]:
        d.act = devs[0].act
        d.op.bind([d.act, d.weights, d.scale, d.zero_point], [d.out])
    import torch
    M.fc_launch_fused([d.op for d in devs], torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    for d, c in zip(devs, cases):
        assert d.op.kernel_variant == form
        check(d.result(), c)


@pytest.mark.parametrize("k,n,form", [(1600, 2600000, "direct"), (2048, 1000000, "skinny 64x16 k1")])
def test_offsets_below_two_gib(k, n, form):
    """A batch of loads that would reach past 2 GiB of one matrix's offsets (1600 input channels of 2048 in a batch, 2.08 GB of
    weights) goes to the direct kernel; channels at both ends and between against float64."""
    import torch
    m, ks, ns = 8, k // 4, n // 4
    gen = torch.Generator(device="cuda").manual_seed(1)
    desc = M.fc_int4_weights_desc(n, k, reference=True)
    weights = torch.randint(-2 ** 31, 2 ** 31, (ks * ns * 2,), dtype=torch.int32, device="cuda", generator=gen)
    act = torch.randn((ks, m, 4), device="cuda", generator=gen).half()
    scale = (torch.rand((k // 32, ns * 4), device="cuda", generator=gen) * 0.01).half()  # (groups of 32: few-token per-channel layers have a kernel of their own)
    out = torch.zeros((ns, m, 4), dtype=torch.float16, device="cuda")
    op = M.fc_create(M.PRECISION_F32_F16, M.FLOAT16, M.FLOAT16, n, k, desc, scale_shape=(n, k // 32), max_tokens=m)
    op.bind([act, weights, scale], [out])
    op.set_shape(1, 1, m)
    print("offsets", k, n, flush=True)
    op.launch(torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert op.kernel_variant == form
    words = weights.view(ks, ns, 2)
    for s in (0, 1, ns // 3, ns - 1):
        w = words[:, s].cpu().numpy().view(np.uint32)  # [ks][2]: bits 16 (i % 2) + 4 c of word i / 2
        u = np.stack([[(w[:, i // 2] >> (16 * (i % 2) + 4 * c)) & 15 for c in range(4)] for i in range(4)])  # [i][c][ks]
        wf = (u.transpose(2, 0, 1).reshape(k, 4).astype(np.float64) - 8) * scale[:, 4 * s:4 * s + 4].double().cpu().numpy().repeat(32, axis=0)
        ref = act.double().cpu().numpy().transpose(1, 0, 2).reshape(m, k) @ wf
        err = np.abs(out[s].double().cpu().numpy() - ref)
        assert np.all(err <= 2.0 ** -10 * np.abs(ref) + 6 * 2.0 ** -10 * np.sqrt(np.mean(ref ** 2)))


# 64-channel tiles up to 16 tokens: K tails, the last slices of a matrix, K cut in 8, activations with a mean, one token with an
# infinite value
@pytest.mark.parametrize("m,k,n,groups", [(5, 544, 12804, 17), (16, 2048, 16384, 64), (8, 1056, 12800, 33), (11, 8192, 2052, 64), (16, 9001, 100, 1)])
def test_whole_strips(m, k, n, groups):
    case = W.make_fc_case(seed=m + k, m=m, k=k, n=n, weight_bits=4, tensor_dtype=np.float16, groups=groups, with_bias=True)
    case["act"] = (case["act"].astype(np.float32) + 2.0).astype(np.float16)
    print("whole strips", m, k, n, groups, flush=True)
    dev = W.FcDevice(case)
    dev.run()
    got = dev.result()
    assert dev.op.kernel_variant.startswith("skinny 64x16 k"), dev.op.kernel_variant
    check(got, case)
    inf = dict(case, act=np.array(case["act"]))
    inf["act"][m - 1, k - 1] = np.inf
    dev = W.FcDevice(inf)
    dev.run()
    got_inf = dev.result()
    assert np.array_equal(got_inf[:m - 1], got[:m - 1])
    sign = np.sign(case["w"][:, k - 1].astype(np.float64) * case["scale"][:, -1].astype(np.float16).astype(np.float64))
    assert np.array_equal(got_inf[m - 1], np.where(sign == 0, np.nan, np.copysign(np.inf, sign)), equal_nan=True)


# An activation far above the others, where a channel's weight is zero: 0 * a adds nothing to that channel, whose error stays that of
# the other products.  (Codes multiplied before 8 is taken from them are off by 1e-3 .. 1e-1 of such a channel's size.)
@pytest.mark.parametrize("large", [1e4, 6e4])
@pytest.mark.parametrize("m,k,n,groups,form", [(8, 2048, 16384, 64, "skinny 64x16 k1"), (16, 8192, 4096, 256, "skinny 64x16 k4"), (8, 512, 1024, 16, "skinny 16x16 k1"),
                                               (24, 8192, 2052, 1, "skinny 64x32 k4"), (12, 64, 16640, 2, "direct")])
def test_large_activation_meets_zero_weights(m, k, n, groups, form, large):
    case = W.make_fc_case(seed=m + k, m=m, k=k, n=n, weight_bits=4, tensor_dtype=np.float16, groups=groups)
    case["act"] = np.array(case["act"])
    case["act"][:, k // 3] = large
    case["w"][::2, k // 3] = 0
    print("large activation", m, k, n, groups, large, flush=True)
    dev = W.FcDevice(case)
    dev.run()
    got = dev.result()
    assert dev.op.kernel_variant == form, dev.op.kernel_variant
    ref = textbook(case)[:, ::2]
    assert np.all(np.abs(got[:, ::2] - ref) <= 2.0 ** -10 * np.abs(ref) + 6 * 2.0 ** -10 * np.sqrt(np.mean(ref ** 2)))
