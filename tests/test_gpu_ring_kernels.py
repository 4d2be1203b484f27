"""GPU parity of the two kernels that serve ringed uint8 weights at decode sizes (fc_w8_ring_i_column_kernel:
ring over the input channels, any window that one work-group walks; fc_w8_ring_o_kernel: ring over the output
channels from 64 KB of weights on), against the float64 product over the rolled weights: more tokens than the
partial-sum kernel takes, window lengths around a pass of the work-group, slices that the end of the ring cuts,
widths that fill no group of 8 slices, batched weights, bounds, fp16 activations below the normal range."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

import mldhip as M
import workloads as W
from test_oracle_ring import make, rolled_product


def run(axis, src_c, dst_c, ring, tokens, offsets, f16, batch=1, seed=1, src_end=None, dst_end=None, tiny=False, kernel=None, form=None):
    import torch
    td, mt = (np.float16, M.FLOAT16) if f16 else (np.float32, M.FLOAT32)
    q, _, scale, zp, bias = make(seed, src_c, dst_c, ring, axis, batch)
    rng = np.random.default_rng(seed)
    act = rng.uniform(-1, 1, size=(batch * tokens, src_c))
    if tiny:  # probabilities of a long softmax: most of them are fp16 subnormals
        act = np.exp(rng.normal(-12.0, 3.0, size=act.shape))
        bias = bias * 0.0
    act, scale, bias = (v.astype(td).astype(np.float32) for v in (act, scale, bias))
    w_o, w_i = q.shape[0], q.shape[3]
    desc = M.make_desc(M.UINT8, M.LAYOUT_I4O4 if axis == "i" else M.LAYOUT_O4I4, (w_o + 3) // 4)
    packed = M.rearrange_int8_as_uint8(q, desc)
    ns = (dst_c + 3) // 4
    pad = lambda v: np.tile(np.pad(v, (0, ns * 4 - dst_c)).astype(td), batch)
    kw = {"ring_%s_offset_index" % axis: 1, "ring_size": ring, ("src" if axis == "i" else "dst") + "_channels": src_c if axis == "i" else dst_c}
    if batch > 1:
        kw["weights_batch"] = batch
    if src_end is not None:
        kw["src_end_ch_index"] = 2
    if dst_end is not None:
        kw["dst_end_ch_index"] = 3
    op = M.fc_create(M.PRECISION_F32_F16 if f16 else M.PRECISION_F32, mt, mt, w_o, w_i, desc, has_bias=True, has_zero_point_tensor=True,
                     scale_shape=(dst_c, 1), max_tokens=batch * tokens, **kw)
    params = np.array([-1, 0, src_end or 0, dst_end or 0], np.int32)
    d_params = torch.from_numpy(params).cuda()
    cuda = lambda v: torch.from_numpy(np.ascontiguousarray(v)).cuda()
    srcs = [cuda(W.to_slices(act).astype(td))]
    if batch > 1:
        srcs.append(torch.arange(batch, dtype=torch.int32, device="cuda"))
    bias_t = np.pad(bias, (0, ns * 4 - dst_c)).astype(td)
    srcs += [cuda(packed), cuda(pad(scale)), cuda(pad(zp)), cuda(bias_t), d_params]
    out = torch.zeros((ns, batch * tokens, 4), dtype=torch.float16 if f16 else torch.float32, device="cuda")
    op.bind(srcs, [out])
    op.set_shape(1, batch, tokens) if batch > 1 else op.set_shape(1, 1, tokens)
    for off in offsets:
        params[1] = off
        d_params.copy_(torch.from_numpy(params))
        out.fill_(7.0)
        print("ring kernel", axis, src_c, dst_c, ring, "tokens", tokens, "batch", batch, "offset", off, "f16", f16, src_end, dst_end, flush=True)
        op.launch(torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        assert op.kernel_name == (kernel or "fc_w8_ring_%s_kernel" % axis), op.kernel_name
        assert form is None or op.kernel_variant == form, op.kernel_variant
        got = W.from_slices(out.cpu().numpy().astype(np.float64), dst_c)
        n_written = dst_c if dst_end is None else min((dst_end + 31) // 32 * 32, ns * 4)
        if n_written < dst_c:
            assert np.all(got[:, n_written:] == 7.0)
        active = None if src_end is None else (min(src_end, src_c) + 3) // 4 * 4
        for b in range(batch):
            for t in range(tokens):
                a = act[b * tokens + t]
                exact = rolled_product(q, a, scale, zp, bias, axis, ring, off, b, src_c, dst_c, active=active)[:n_written]
                # fp32 sums: the products of a thread one after the other (some 100 at most), then a tree; every partial sum is of
                # the size of the root of the sum of squares (weights of random sign) or, in the zero point's half, of the
                # sum of magnitudes; a lost slice of 4 channels is sqrt(4 / src_c) of the former, over 0.01 at 33000 channels.
                # fp16 results are rounded twice (result, bias)
                s_abs = scale[:n_written].astype(np.float64)
                size = np.sqrt((a.astype(np.float64) ** 2).sum()) * 74.0  # (rms of a weight: 127 / sqrt(3))
                tol = 2.0 ** -24 * s_abs * (128 * size + 64 * np.abs(a).sum()) + (
                    2.0 ** -10 * (np.abs(exact) + np.abs(bias[:n_written])) + 2.0 ** -24 if f16 else 2.0 ** -22 * (np.abs(exact) + np.abs(bias[:n_written])))
                assert np.all(np.abs(got[b * tokens + t][:n_written] - exact) <= tol), (b, t, off)


@pytest.mark.parametrize("f16", [True, False])
@pytest.mark.parametrize("tokens", [1, 2, 3, 5, 8, 16])
def test_ring_i_token_counts(f16, tokens):
    run("i", 300, 72, 1024, tokens, [0, 1, 722, 1023, -6], f16, seed=tokens)


@pytest.mark.parametrize("src_c,ring", [(1021, 1024), (2044, 2052), (2048, 2048), (4096, 4104), (4097, 8192), (8190, 8192), (12, 16)])
def test_ring_i_windows(src_c, ring):
    """Windows around one and two rows per thread at both work-group sizes, full turns of the ring, a short one."""
    run("i", src_c, 40, ring, 6, [0, 3, ring - 2], True, seed=src_c)


@pytest.mark.parametrize("f16", [True, False])
@pytest.mark.parametrize("tokens", [1, 2, 4, 7, 9])
def test_ring_o_token_counts(f16, tokens):
    run("o", 68, 1000, 1024, tokens, [0, 1, 722, 1023, -6], f16, seed=tokens)


@pytest.mark.parametrize("src_c,dst_c,ring", [(256, 2048, 2048), (64, 4093, 4096), (30, 8192, 8192), (260, 515, 1000)])
def test_ring_o_shapes(src_c, dst_c, ring):
    run("o", src_c, dst_c, ring, 8, [0, 5, ring - 1], True, seed=dst_c)


def test_ring_batches_and_bounds():
    run("i", 512, 320, 512, 5, [0, 258], True, batch=3, src_end=301, dst_end=70)
    run("o", 128, 600, 1024, 6, [3, 900], True, batch=2, src_end=61, dst_end=200)
    run("o", 128, 600, 1024, 3, [3, 900], False, batch=2)


def test_ring_i_subnormal_probabilities():
    run("i", 8192, 64, 8192, 8, [0, 4099], True, tiny=True)


@pytest.mark.parametrize("src_c,tokens,f16", [(16384, 1, True), (16389, 1, True), (20000, 1, False), (32769, 3, True), (33000, 2, True),
                                              (33000, 5, True)])
def test_ring_i_windows_around_the_split(src_c, tokens, f16):
    """Window lengths where the launcher passes from one work-group per slice to the split window (up to 4 tokens)."""
    run("i", src_c, 24, (src_c + 7) // 4 * 4, tokens, [0, 2, src_c // 2 + 1], f16, seed=src_c)


@pytest.mark.parametrize("src_c,dst_c,ring", [(16, 40, 32), (256, 2052, 1024), (64, 8192, 8188)])
def test_ring_o_refuses_more_channels_than_the_ring(src_c, dst_c, ring):
    """dst channels that would wrap the ring: an error at any size, and nothing is launched."""
    import torch
    desc = M.make_desc(M.UINT8, M.LAYOUT_O4I4, ring // 4)
    op = M.fc_create(M.PRECISION_F32_F16, M.FLOAT16, M.FLOAT16, ring, src_c, desc, scale_shape=(dst_c, 1), max_tokens=2,
                     ring_o_offset_index=0, ring_size=ring, dst_channels=dst_c)
    half = lambda *shape: torch.zeros(shape, dtype=torch.float16, device="cuda")
    out = torch.full((dst_c // 4, 2, 4), 7.0, dtype=torch.float16, device="cuda")
    op.bind([half(src_c // 4, 2, 4), torch.zeros(ring * src_c, dtype=torch.uint8, device="cuda"), half(dst_c),
             torch.zeros(1, dtype=torch.int32, device="cuda")], [out])
    op.set_shape(1, 1, 2)
    with pytest.raises(M.MldhipError):
        op.launch(torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert torch.all(out == 7.0)


# column walk, split window (one token over more than 16384 positions), ring over the output channels
@pytest.mark.parametrize("axis,src_c,dst_c,ring,tokens", [("i", 300, 72, 1024, 5), ("i", 20000, 24, 20004, 1), ("o", 68, 1000, 1024, 3)])
@pytest.mark.parametrize("f16", [True, False])
@pytest.mark.parametrize("zero_point", [True, False])
def test_ring_infinite_activations(axis, src_c, dst_c, ring, tokens, f16, zero_point):
    """An infinite activation gives the infinities and NaNs of the unspecialised kernel, which multiplies every product by
    itself: infinite where no weight of the channel is exactly its zero point, with the product's sign."""
    import torch
    td, mt = (torch.float16, M.FLOAT16) if f16 else (torch.float32, M.FLOAT32)
    rng = np.random.default_rng(src_c)
    o, i = (dst_c, ring) if axis == "i" else (ring, src_c)
    desc = M.make_desc(M.UINT8, M.LAYOUT_I4O4 if axis == "i" else M.LAYOUT_O4I4, (o + 3) // 4)
    packed = M.rearrange_int8_as_uint8(rng.integers(-2, 3, size=(o, 1, 1, i), dtype=np.int8), desc)
    act = rng.uniform(-1, 1, size=(tokens, src_c))
    act[0, src_c // 2] = np.inf
    if tokens > 1:
        act[1, 3], act[1, src_c - 1] = -np.inf, -np.inf
    ns = (dst_c + 3) // 4
    kw = {"ring_%s_offset_index" % axis: 0, "ring_size": ring, ("src" if axis == "i" else "dst") + "_channels": src_c if axis == "i" else dst_c}
    op = M.fc_create(M.PRECISION_F32_F16 if f16 else M.PRECISION_F32, mt, mt, o, i, desc, scale_shape=(dst_c, 1), max_tokens=tokens,
                     has_zero_point_tensor=zero_point, **kw)
    srcs = [torch.from_numpy(W.to_slices(act)).to(td).cuda(), torch.from_numpy(packed).cuda(), torch.full((ns * 4,), 0.01, dtype=td, device="cuda")]
    if zero_point:
        srcs.append(torch.from_numpy(rng.integers(-2, 3, size=ns * 4)).to(td).cuda())
    srcs.append(torch.tensor([ring // 3], dtype=torch.int32, device="cuda"))
    results = []
    for generic in (0, 1):
        out = torch.full((ns, tokens, 4), 7.0, dtype=td, device="cuda")
        op.bind(srcs, [out])
        op.set_shape(1, 1, tokens)
        with M.tuning(force_generic=generic):
            op.launch(torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        assert op.kernel_name == ("fc_generic_kernel" if generic else "fc_w8_ring_%s_kernel" % axis)
        results.append(W.from_slices(out.cpu().numpy().astype(np.float64), dst_c))
    got, ref = results
    assert np.isinf(ref[0]).any() and np.isnan(ref[0]).any()
    assert np.array_equal(np.isnan(got), np.isnan(ref)) and np.array_equal(np.isinf(got), np.isinf(ref))
    assert np.array_equal(got[np.isinf(got)], ref[np.isinf(ref)])


# the kernel by window, width, tokens and rows: column walk, split window (up to 4 tokens per row and 16 in all), unspecialised
@pytest.mark.parametrize("src_c,dst_c,tokens,batch,f16,form", [
    (1024, 64, 1, 1, True, "column"), (2100, 256, 4, 1, True, "column"), (16380, 24, 1, 1, True, "column"), (16388, 24, 1, 1, True, "split"),
    (32760, 16, 3, 1, False, "column"), (32772, 16, 3, 1, False, "split"), (2048, 1200, 1, 4, True, "split"), (2560, 4096, 2, 1, False, "split"),
    (640, 72, 5, 4, True, "column"), (4096, 20, 17, 1, True, "column"), (300, 40, 4, 5, False, "column"), (2100, 520, 9, 4, False, "unspecialised"),
    (2100, 1400, 33, 1, True, "unspecialised"), (64, 12, 64, 1, True, "column")])
def test_ring_i_kernel_choice(src_c, dst_c, tokens, batch, f16, form):
    ring = (src_c + 3) // 4 * 4
    run("i", src_c, dst_c, ring, tokens, [0, src_c // 2 + 1], f16, batch=batch, seed=src_c,
        **(dict(kernel="fc_generic_kernel", form="") if form == "unspecialised" else dict(form=form)))


# A single activation of 1, scales of 1, no zero point: the result is that input channel's weights, exactly.  The first and last
# channel, both sides of the seams of a slice, a wave, a pass of 256 and of 1024 threads, and where the window meets the ring's end
@pytest.mark.parametrize("axis,src_c,dst_c,ring,tokens,form", [
    ("i", 1021, 40, 1024, 8, "column"), ("i", 8190, 12, 8192, 6, "column"), ("i", 16384, 24, 16384, 1, "column"), ("i", 32757, 8, 32760, 4, "column"),
    ("i", 16390, 20, 16392, 1, "split"), ("i", 33000, 24, 33004, 3, "split"), ("i", 2560, 6400, 2560, 2, "split"),
    ("o", 68, 1000, 1024, 7, ""), ("o", 260, 515, 1000, 4, ""), ("o", 1030, 64, 64, 2, "")])
@pytest.mark.parametrize("f16", [True, False])
def test_ring_one_channel(axis, src_c, dst_c, ring, tokens, form, f16):
    import torch
    td, mt = (torch.float16, M.FLOAT16) if f16 else (torch.float32, M.FLOAT32)
    rng = np.random.default_rng(src_c + dst_c)
    o, i = (dst_c, ring) if axis == "i" else (ring, src_c)
    q = rng.integers(-127, 128, size=(o, 1, 1, i), dtype=np.int8)
    desc = M.make_desc(M.UINT8, M.LAYOUT_I4O4 if axis == "i" else M.LAYOUT_O4I4, (o + 3) // 4)
    packed = torch.from_numpy(M.rearrange_int8_as_uint8(q, desc)).cuda()
    ns, ks = (dst_c + 3) // 4, (src_c + 3) // 4
    kw = {"ring_%s_offset_index" % axis: 0, "ring_size": ring, ("src" if axis == "i" else "dst") + "_channels": src_c if axis == "i" else dst_c}
    op = M.fc_create(M.PRECISION_F32_F16 if f16 else M.PRECISION_F32, mt, mt, o, i, desc, scale_shape=(dst_c, 1), max_tokens=tokens, **kw)
    act = torch.zeros((ks, tokens, 4), dtype=td, device="cuda")
    out = torch.zeros((ns, tokens, 4), dtype=td, device="cuda")
    params = torch.zeros(1, dtype=torch.int32, device="cuda")
    op.bind([act, packed, torch.ones(ns * 4, dtype=td, device="cuda"), params], [out])
    op.set_shape(1, 1, tokens)
    for off in (0, 1, 2, 3, ring - 1, ring - 6):
        seams = [0, 3, 4, 255, 256, 1023, 1024, 2047, 2048, 4095, 4096, 8191, 8192, ring - off - 1, ring - off, src_c - 5, src_c - 4, src_c - 1]
        places = sorted({c for c in seams if 0 <= c < src_c})
        params.fill_(off)
        for first in range(0, len(places), tokens):
            some = [places[min(first + t, len(places) - 1)] for t in range(tokens)]
            act.zero_()
            for t, c in enumerate(some):
                act[c // 4, t, c % 4] = 1.0
            out.fill_(7.0)
            print("one channel", axis, src_c, dst_c, ring, off, some, f16, flush=True)
            op.launch(torch.cuda.current_stream().cuda_stream)
            torch.cuda.synchronize()
            assert (op.kernel_name, op.kernel_variant) == ("fc_w8_ring_%s_kernel" % axis, form)
            got = W.from_slices(out.cpu().numpy().astype(np.float64), dst_c)
            for t, c in enumerate(some):
                want = q[:, 0, 0, (c + off) % ring] if axis == "i" else q[(np.arange(dst_c) + off) % ring, 0, 0, c]
                assert np.array_equal(got[t], want.astype(np.float64)), (off, c)
