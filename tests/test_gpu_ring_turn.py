"""GPU parity of the ring kernels where the window is the whole ring (fc_w8_ring_i_turn_kernel, fc_w8_ring_o_turn_kernel): every shift of
the ring's start against a slice, the last rows of a wave, of a pass of 256 and of 1024 threads and of a second pass, one to several token
slots with a remainder, matrices of a batch, with and without zero points, where the sums of the activations leave some launches to the kernel for any window; one
work-group of 1024 threads per CU and two.  Small whole numbers make every product and sum exact, so
the results are those of the rolled weights whatever the order of the sums, and those of the unspecialised kernel with an infinite
activation."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

import mldhip as M
import workloads as W

SHAPES = [  # axis, ring, other channels, tokens, batch
    ("i", 4, 8, 1, 1), ("i", 252, 20, 3, 2), ("i", 260, 72, 8, 1), ("i", 2052, 12, 5, 1), ("i", 4104, 260, 6, 1), ("i", 8200, 24, 1, 1),
    ("i", 16384, 8, 7, 1), ("i", 1024, 1032, 5, 1), ("i", 4104, 260, 10, 1), ("i", 4096, 516, 6, 1), ("i", 2052, 16, 64, 4), ("i", 2052, 256, 12, 1), ("o", 1024, 256, 1, 1), ("o", 1000, 70, 3, 2), ("o", 8200, 64, 9, 1), ("o", 68, 1030, 6, 1)]


def turns(axis, ring, other, tokens, rows, f16, zero_point):
    """Whether a window that is the whole ring runs on a turn kernel."""
    if axis == "o" or not zero_point:
        return True
    ns, small = (other + 3) // 4, ring // 4 + 1 <= 512  # (256 threads instead of 1024)
    slots = 4 if ns * rows * ((tokens + 3) // 4) >= 256 else 2
    while slots > tokens:
        slots //= 2
    if f16:  # two rows per thread cover the ring
        return (small or slots <= 2) and ring // 4 <= (512 if small else 2048)
    # fp32, two slots, 1024 threads: at most 1.25 work-groups for every CU of the busiest XCD
    runs = min(8, (ns + 7) // 8)
    planes, copies = (tokens + 1) // 2 * rows, {1: 8, 2: 4, 3: 2, 4: 2}.get(runs, 1)
    shared = planes if planes <= 8 else max(8, -(-planes // copies))
    return slots != 2 or small or (ns // 64 * 8 + min(8, ns % 64)) * shared / 32 <= 1.25


@pytest.mark.parametrize("axis,ring,other,tokens,batch", SHAPES)
@pytest.mark.parametrize("f16", [True, False])
@pytest.mark.parametrize("zero_point", [True, False])
def test_ring_turn(axis, ring, other, tokens, batch, f16, zero_point):
    import torch
    td, mt = (torch.float16, M.FLOAT16) if f16 else (torch.float32, M.FLOAT32)
    rng = np.random.default_rng(ring + other)
    src_c, dst_c = (ring, other) if axis == "i" else (other, ring)
    shape = (dst_c, batch, 1, ring) if axis == "i" else (ring, batch, 1, src_c)
    q = rng.integers(-3, 4, size=shape, dtype=np.int8)
    q[0, 0, 0, 0], q[-1, -1, 0, -1] = 127, -127
    desc = M.make_desc(M.UINT8, M.LAYOUT_I4O4 if axis == "i" else M.LAYOUT_O4I4, (shape[0] + 3) // 4)
    packed = torch.from_numpy(M.rearrange_int8_as_uint8(q, desc)).cuda()
    # activations of -1, 0 and 1 in 60 channels: sums of at most 60 * 6 + 2 * 131, whole numbers that fp16 holds
    act = np.zeros((batch * tokens, src_c))
    for a in act:
        a[rng.integers(0, src_c, size=60)] = rng.integers(-1, 2, size=60)
        a[0], a[-1] = 1, 1
    ns = (dst_c + 3) // 4
    zp = rng.integers(-3, 4, size=dst_c) if zero_point else np.zeros(dst_c, np.int64)
    kw = {"ring_%s_offset_index" % axis: 0, "ring_size": ring, ("src" if axis == "i" else "dst") + "_channels": ring}
    if batch > 1:
        kw["weights_batch"] = batch
    op = M.fc_create(M.PRECISION_F32_F16 if f16 else M.PRECISION_F32, mt, mt, shape[0], shape[3], desc, scale_shape=(dst_c, 1),
                     max_tokens=batch * tokens, has_zero_point_tensor=zero_point, **kw)
    d_act = torch.from_numpy(W.to_slices(act)).to(td).cuda()
    params = torch.zeros(1, dtype=torch.int32, device="cuda")
    srcs = [d_act] + ([torch.arange(batch, dtype=torch.int32, device="cuda")] if batch > 1 else []) + [packed]
    srcs.append(torch.ones(batch * ns * 4, dtype=td, device="cuda"))
    if zero_point:
        srcs.append(torch.from_numpy(np.tile(np.pad(zp, (0, ns * 4 - dst_c)), batch)).to(td).cuda())
    srcs.append(params)

    def launch(off, generic=0):
        out = torch.full((ns, batch * tokens, 4), 7.0, dtype=td, device="cuda")
        op.bind(srcs, [out])
        op.set_shape(1, batch, tokens)
        params.fill_(off)
        print("ring turn", axis, ring, other, "tokens", tokens, "batch", batch, "offset", off, f16, zero_point, flush=True)
        with M.tuning(force_generic=generic):
            op.launch(torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        assert (op.kernel_name, op.kernel_whole) == (
            ("fc_generic_kernel", False) if generic else ("fc_w8_ring_%s_kernel" % axis, turns(axis, ring, other, tokens, batch, f16, zero_point)))
        return W.from_slices(out.cpu().numpy().astype(np.float64), dst_c)

    for off in (0, 1, 2, 3, ring - 1, ring - 3, ring // 2 + 1, -6):
        got = launch(off)
        for b in range(batch):
            w = q[:, b, 0].astype(np.int64)
            w = np.roll(w, -off, axis=1 if axis == "i" else 0) - zp[:, None]
            want = act[b * tokens:(b + 1) * tokens] @ w.T
            assert np.array_equal(got[b * tokens:(b + 1) * tokens], want), (off, b)
    d_act[0, 0, 1] = float("inf")
    d_act[-1, -1, (src_c - 1) % 4] = -float("inf")
    got, ref = launch(ring // 3), launch(ring // 3, generic=1)
    assert np.isinf(ref).any() and np.array_equal(got, ref, equal_nan=True)


# Scales, zero points and biases of their own for every channel and matrix (powers of two and whole numbers: sums, products and results
# stay exact), the ring's start at all four places against a slice: an index that is off by a channel, a slice or a matrix shows.
# other channels that fill no slice, batches, several token slots with a remainder; a window one slice shorter than the ring and a bound
# that cuts nothing stay on the kernels for any window.
@pytest.mark.parametrize("axis,ring,other,tokens,batch", [("i", 1028, 30, 1, 2), ("i", 2064, 22, 3, 1), ("i", 516, 260, 5, 2), ("o", 1028, 260, 1, 2),
                                                          ("o", 520, 132, 3, 2), ("o", 1036, 68, 6, 1)])
@pytest.mark.parametrize("f16", [True, False])
@pytest.mark.parametrize("zero_point", [True, False])
@pytest.mark.parametrize("bias", [True, False])
@pytest.mark.parametrize("form", ["whole", "short", "bound"])
def test_ring_turn_channel_parameters(axis, ring, other, tokens, batch, f16, zero_point, bias, form):
    import torch
    td, mt = (torch.float16, M.FLOAT16) if f16 else (torch.float32, M.FLOAT32)
    rng = np.random.default_rng(ring + other + tokens)
    window = ring - 4 if form == "short" else ring
    src_c, dst_c = (window, other) if axis == "i" else (other, window)
    w_o, w_i = (other, ring) if axis == "i" else (ring, other)
    q = rng.integers(-3, 4, size=(w_o, batch, 1, w_i), dtype=np.int8)
    desc = M.make_desc(M.UINT8, M.LAYOUT_I4O4 if axis == "i" else M.LAYOUT_O4I4, (w_o + 3) // 4)
    # 12 activations of -1 and 1: |sum| at most 12 * 6 (weights less zero points), times a scale of 1/4 .. 4 plus a bias of at most 15
    act = np.zeros((batch * tokens, src_c))
    for a in act:
        a[rng.choice(src_c, 12, replace=False)] = rng.choice([-1, 1], 12)
    ns = (dst_c + 3) // 4
    scale = 2.0 ** rng.integers(-2, 3, size=(batch, dst_c))
    zp = rng.integers(-3, 4, size=(batch, dst_c)) if zero_point else np.zeros((batch, dst_c), np.int64)
    b = rng.integers(-15, 16, size=dst_c) if bias else np.zeros(dst_c, np.int64)
    kw = {"ring_%s_offset_index" % axis: 0, "ring_size": ring, ("src" if axis == "i" else "dst") + "_channels": window}
    if batch > 1:
        kw["weights_batch"] = batch
    if form == "bound":
        kw["dst_end_ch_index"] = 1
    op = M.fc_create(M.PRECISION_F32_F16 if f16 else M.PRECISION_F32, mt, mt, w_o, w_i, desc, scale_shape=(dst_c, 1), max_tokens=batch * tokens,
                     has_zero_point_tensor=zero_point, has_bias=bias, **kw)
    pad = lambda v: torch.from_numpy(np.pad(v, [(0, 0)] * (v.ndim - 1) + [(0, ns * 4 - dst_c)]).astype(np.float32)).to(td).cuda()
    ids = np.arange(batch)[::-1].astype(np.int32).copy()
    srcs = [torch.from_numpy(W.to_slices(act)).to(td).cuda()] + ([torch.from_numpy(ids).cuda()] if batch > 1 else [])
    srcs += [torch.from_numpy(M.rearrange_int8_as_uint8(q, desc)).cuda(), pad(scale)] + ([pad(zp)] if zero_point else []) + ([pad(b)] if bias else [])
    params = torch.tensor([0, ring + 64], dtype=torch.int32, device="cuda")
    out = torch.zeros((ns, batch * tokens, 4), dtype=td, device="cuda")
    op.bind(srcs + [params], [out])
    op.set_shape(1, batch, tokens)
    for off in (0, 1, 2, 3, ring - 2):
        params[0] = off
        out.fill_(7.0)
        print("channel parameters", axis, ring, other, "tokens", tokens, "batch", batch, "offset", off, f16, zero_point, bias, form, flush=True)
        op.launch(torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        assert (op.kernel_name, op.kernel_whole) == ("fc_w8_ring_%s_kernel" % axis, form == "whole" and turns(axis, ring, other, tokens, batch, f16, zero_point))
        got = W.from_slices(out.cpu().numpy().astype(np.float64), dst_c)
        for r in range(batch):
            w = np.roll(q[:, ids[r] if batch > 1 else 0, 0].astype(np.int64), -off, axis=1 if axis == "i" else 0)
            w = w[:, :window] if axis == "i" else w[:window]
            m = ids[r] if batch > 1 else 0
            want = (act[r * tokens:(r + 1) * tokens] @ (w - zp[m][:, None]).T) * scale[m] + b
            assert np.array_equal(got[r * tokens:(r + 1) * tokens], want), (off, r)


# Both sides of the lines: rows of a thread's first two, token slots, work-groups per CU
@pytest.mark.parametrize("ring,channels,tokens,f16,expected", [
    (2044, 24, 2, True, True), (2048, 24, 2, True, True), (8192, 24, 2, True, True), (8196, 24, 2, True, False), (1024, 1032, 5, True, True),
    (4096, 1032, 5, True, False), (16384, 24, 1, False, True), (4096, 64, 2, False, True), (4096, 256, 10, False, True),
    (4096, 256, 12, False, False), (4096, 1032, 5, False, True)])
def test_ring_turn_lines(ring, channels, tokens, f16, expected):
    assert turns("i", ring, channels, tokens, 1, f16, True) == expected
    test_ring_turn("i", ring, channels, tokens, 1, f16, True)


# Token slots of the keys' kernels: a turn takes four where two give 512 work-groups, a window that is not the whole ring where four do
@pytest.mark.parametrize("ring,window,tokens,slots", [
    (8192, 8192, 8, 4), (8188, 8188, 7, 4), (8128, 8128, 8, 2), (10880, 10880, 6, 2), (10944, 10944, 6, 4), (16384, 16384, 4, 4), (16384, 16384, 2, 2),
    (16320, 16320, 4, 2), (4096, 4096, 1, 1), (16388, 16384, 8, 4), (16324, 16320, 8, 2)])
def test_ring_o_slots(ring, window, tokens, slots):
    import torch
    k, ns, wns = 16, window // 4, ring // 4
    rng = np.random.default_rng(ring + tokens)
    q = rng.integers(-3, 4, size=(ring, 1, 1, k), dtype=np.int8)
    desc = M.make_desc(M.UINT8, M.LAYOUT_O4I4, wns)
    act = rng.integers(-2, 3, size=(tokens, k)).astype(np.float64)
    op = M.fc_create(M.PRECISION_F32_F16, M.FLOAT16, M.FLOAT16, ring, k, desc, scale_shape=(window, 1), max_tokens=tokens, ring_o_offset_index=0,
                     ring_size=ring, dst_channels=window)
    out = torch.zeros((ns, tokens, 4), dtype=torch.float16, device="cuda")
    off = ring // 3 + 1
    op.bind([torch.from_numpy(W.to_slices(act)).half().cuda(), torch.from_numpy(M.rearrange_int8_as_uint8(q, desc)).cuda(),
             torch.ones(ns * 4, dtype=torch.float16, device="cuda"), torch.tensor([off], dtype=torch.int32, device="cuda")], [out])
    op.set_shape(1, 1, tokens)
    print("slots", ring, window, tokens, flush=True)
    op.launch(torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert (op.kernel_name, op.kernel_whole, op.kernel_tiles) == ("fc_w8_ring_o_kernel", ring == window, (slots, 4, 1))
    got = W.from_slices(out.cpu().numpy().astype(np.float64), window)
    assert np.array_equal(got, act @ np.roll(q[:, 0, 0].astype(np.int64), -off, axis=0)[:window].T)
