"""The work that programs built on this library have it do, as cases that can be timed.

Every case goes through the public binding (ml-drift_amd/python/mldhip.py): ops are created, bound and
shaped once, as a graph builder does at load time, and a pass launches them.  Decode steps (a handful of
tokens, tens of launches of a few microseconds each) are captured into a HIP graph once and replayed, as
decoder_stack.DecoderStack.capture and bench.py do; prefill passes and single ops are launched directly.

Weights are random codes over the full range of their type in the packed layout that the library asks
for, scales |N(0, 0.02)| / (largest code), activations N(0, 1): the distributions of
workloads.make_fc_case, generated on the device.  The packed bytes are drawn directly: the packers only
move codes, so a buffer of random bytes is a packed random matrix.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "ml-drift_amd", "python"))  # (the working folder is the repository's root)
import mldhip as M

# ---------------------------------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------------------------------


def listed():
    return [
        # The smallest call: one uint8 FullyConnected over one token with fp32 tensors (the fp32 precision of the
        # builder), launched directly.  Range: 1..16 tokens, 256..4096 channels each way, odd ones too.
        dict(name="f32_u8_1tok", kind="f32_u8", tokens=1, k=2048, n=2048, bias=False, zero_point=False),
        # One decode step of a decoder stack (hidden 2048, one key/value head of 256, gated MLP of 16384), every
        # FullyConnected of every layer with weights of its own: q/k/v in one launch, o, gate/up in one, down.
        # Range: 2..18 layers, hidden 1024..3072, MLP 4096..16384, groups of 32, 64 or 128 input channels.
        dict(name="decode_stack", kind="stack", tokens=1, layers=18, hidden=2048, kv=256, mlp=16384, group=32),
        # The MLPs of a larger model at one token, per-channel scales: gate, up and their activation in one launch,
        # then down.  Range: 2..6 layers, hidden 2048..5120, MLP 4096..16384, 1 or 2 tokens.
        dict(name="decode_mlp_per_channel", kind="mlp", tokens=1, layers=6, hidden=4096, mlp=14336),
        # The same stack for a small batch of sequences or a few speculated tokens.  Range: 2..16 tokens.
        dict(name="decode_stack_8tok", kind="stack", tokens=8, layers=18, hidden=2048, kv=256, mlp=16384, group=32),
        # A prompt chunk of 128 tokens through the same stack.  Range: 17..384 tokens, odd counts too.
        dict(name="prefill_stack_128tok", kind="stack", tokens=128, layers=18, hidden=2048, kv=256, mlp=16384, group=32),
        # One projection of a longer prompt, groups of 32.  Range: 129..8192 tokens, 512..14336 channels, per-channel
        # scales and groups of 32..128, with and without bias and zero points, uint4 and uint8.
        dict(name="prefill_fc_512tok", kind="fc", tokens=512, k=4096, n=4096, group=32, bits=4, bias=False, zero_point=False),
        # The largest: a long prompt through the up projection of a larger model.
        dict(name="prefill_fc_8192tok", kind="fc", tokens=8192, k=4096, n=14336, group=32, bits=4, bias=False,
             zero_point=False),
        # uint8 weights, a prompt of any length and channel counts that fill no tile, bias and zero points.
        dict(name="prefill_u8_ragged", kind="fc", tokens=333, k=1656, n=2900, group=0, bits=8, bias=True, zero_point=True),
        # Dynamic quantization of the activations and the int8 x int8 product with its rescale.
        # Range: 64..4096 tokens, 512..8192 channels, symmetric and asymmetric.
        dict(name="int8_dynamic", kind="int8", tokens=2048, k=2048, n=8192, symmetric=True),
        # The expert projections of mixture-of-experts layers at one token: 8 of 128 experts by runtime ids, gate and
        # up over the token, down over their rows.  Range: 2..8 chosen of 8..128 experts, 512..4096 channels.
        dict(name="moe_decode", kind="moe_decode", layers=6, experts=128, top=8, hidden=2048, mlp=768, group=32),
        # The same layer's experts over a prompt of 512 tokens: 4096 rows sorted by expert, group sizes known on the
        # device only (an expert may get up to all 512 tokens).  Range: 64..1024 tokens.
        dict(name="moe_prefill", kind="moe_prefill", tokens=512, experts=128, top=8, hidden=2048, mlp=768, group=32),
        # Attention of one decode step over quantized caches bound as ringed weights: the query heads that share a
        # cache against its keys (ring over the output channels), their probabilities against its values (ring
        # over the input channels).  Range: 1..8 heads per cache, caches of 1024..16384 positions, heads of 64..256.
        dict(name="kv_ring_decode", kind="kv_ring", layers=18, heads=8, positions=8192, head_dim=256),
    ]


def _log(rng, lo, hi, multiple=1):
    """A whole number of [lo, hi], spread over its logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi + 0.999)))
    return max(lo, min(hi, int(v) // multiple * multiple))


def draw(rng):
    kind = rng.choice(["f32_u8", "stack", "stack", "stack", "mlp", "fc", "fc", "fc", "int8", "moe_decode", "moe_prefill", "kv_ring"])
    if kind == "f32_u8":
        return dict(kind=kind, tokens=_log(rng, 1, 16), k=_log(rng, 256, 4096), n=_log(rng, 256, 4096), bias=rng.random() < 0.5,
                    zero_point=rng.random() < 0.3)
    if kind == "stack":
        tokens = rng.choice([1, _log(rng, 2, 16), _log(rng, 17, 384)])
        # (more tokens, fewer layers: the step stays within the listed ones' cost)
        return dict(kind=kind, tokens=tokens, layers=rng.randint(2, 18 if tokens <= 128 else 6), hidden=_log(rng, 1024, 3072, 128),
                    kv=rng.choice([128, 256, 512]), mlp=_log(rng, 4096, 16384, 128), group=rng.choice([32, 32, 64, 128]))
    if kind == "mlp":
        return dict(kind=kind, tokens=rng.choice([1, 1, 2]), layers=rng.randint(2, 6), hidden=_log(rng, 2048, 5120, 64),
                    mlp=_log(rng, 4096, 16384, 64))
    if kind == "fc":
        tokens, n, group = _log(rng, 129, 8192), _log(rng, 512, 14336), rng.choice([0, 32, 32, 64, 128])
        k = _log(rng, 512, 4096, group if group else 1)
        return dict(kind=kind, tokens=tokens, k=k, n=n, group=group, bits=rng.choice([4, 4, 8]), bias=rng.random() < 0.3,
                    zero_point=rng.random() < 0.3)
    if kind == "int8":
        tokens, k, n = _log(rng, 64, 4096), _log(rng, 512, 4096), _log(rng, 512, 8192)
        return dict(kind=kind, tokens=tokens, k=k, n=n, symmetric=rng.random() < 0.5)
    if kind == "moe_decode":
        experts = rng.choice([8, 16, 32, 64, 128])
        mlp = _log(rng, 512, 1536 if experts > 16 else 4096, 64)
        return dict(kind=kind, layers=rng.randint(1, 6), experts=experts, top=rng.choice([2, 4, 8]), hidden=_log(rng, 1024, 3072, 64),
                    mlp=mlp, group=rng.choice([32, 64]))
    if kind == "moe_prefill":
        experts = rng.choice([8, 16, 32, 64, 128])
        return dict(kind=kind, tokens=_log(rng, 64, 1024), experts=experts, top=rng.choice([2, 4, 8]), hidden=_log(rng, 1024, 3072, 64),
                    mlp=_log(rng, 512, 1536, 64), group=rng.choice([32, 64]))
    return dict(kind=kind, layers=rng.randint(2, 18), heads=rng.choice([1, 2, 4, 8]), positions=_log(rng, 1024, 16384, 4),
                head_dim=rng.choice([64, 128, 256]))


# ---------------------------------------------------------------------------------------------------
# Inputs, ops
# ---------------------------------------------------------------------------------------------------


def _slices(c):
    return (c + 3) // 4


class _Program:
    """Device data from one seed, and the ops of a case in launch order."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda").manual_seed(seed)
        self.steps = []  # callables of one argument, the stream
        self.outputs = []
        self.keep = []  # whatever the ops read (an op holds raw pointers)

    def normal(self, shape, dtype=torch.float16):
        t = torch.randn(shape, device="cuda", generator=self.gen).to(dtype)
        self.keep.append(t)
        return t

    def act(self, channels, tokens, dtype=torch.float16):
        """[slices][tokens][4], channels beyond the last one zero."""
        t = self.normal((_slices(channels), tokens, 4), dtype)
        if channels % 4:
            t[-1, :, channels % 4:] = 0
        return t

    def codes(self, desc, o, batch, i):
        """Packed random weights of `batch` matrices."""
        size = M.packed_bytes(desc, o, batch, 1, i)
        if desc.type == M.UINT8:  # -127..127, held as 1..255
            t = torch.randint(1, 256, (size,), dtype=torch.uint8, device="cuda", generator=self.gen)
        else:  # whole words: every nibble -8..7
            t = torch.randint(-2 ** 31, 2 ** 31, ((size + 3) // 4,), dtype=torch.int32, device="cuda",
                              generator=self.gen).view(torch.uint8)[:size]
        if desc.type == M.UINT8 and i % 4 and desc.layout == M.LAYOUT_I4O4:
            # rows that pad the input channels hold the code of zero, as the packers write them
            t.view(-1, batch, _slices(i), desc.output_group_size, 4, 4)[:, :, -1, :, i % 4:, :] = 128
        self.keep.append(t)
        return t

    def scale(self, shape, channels, qmax, dtype=torch.float16):
        """|N(0, 0.02)| / qmax, zero in the channels that pad the last slice."""
        t = ((torch.randn(shape, device="cuda", generator=self.gen) * 0.02).abs() / qmax).to(dtype)
        return self._padded(t, channels)

    def _padded(self, t, channels):
        if channels % 4:
            t.view(-1, _slices(channels) * 4)[:, channels:] = 0
        self.keep.append(t)
        return t

    def out(self, channels, tokens, dtype=torch.float16):
        t = torch.zeros((_slices(channels), tokens, 4), dtype=dtype, device="cuda")
        self.outputs.append(t)
        return t

    def fc(self, src, o, i, tokens, desc, group=0, dtype=torch.float16, bias=False, zero_point=False, batch=1, rows=None,
           shared_src=False, ids=None, packed=None, params=None, dst=None):
        """One FullyConnected op with its weights; `dst`: where its result goes (else an output of the case)."""
        ns, groups = _slices(o), (i // group if group else 1)
        mt = M.FLOAT16 if dtype == torch.float16 else M.FLOAT32
        srcs = [src]
        if ids is not None:
            srcs.append(ids)
        srcs.append(self.codes(desc, o, batch, i))
        srcs.append(self.scale((groups, batch, ns, 4), o, 7.0 if desc.type == M.UINT4 else 127.0, dtype))
        if zero_point:
            srcs.append(self._padded(torch.randint(-3, 4, (groups, batch, ns, 4), device="cuda", generator=self.gen).to(dtype), o))
        if bias:
            srcs.append(self._padded(torch.randn((ns * 4,), device="cuda", generator=self.gen).to(dtype), o))
        if params is not None:
            srcs.append(params)
        total = tokens * (rows or 1)
        if dst is None:
            dst = self.out(o, total, dtype)
        kw = {}
        if ids is not None:
            kw = dict(weights_batch=batch, shared_src=shared_src)
        if packed is not None:
            kw = dict(packed_groups=packed)
        op = M.fc_create(M.PRECISION_F32_F16 if mt == M.FLOAT16 else M.PRECISION_F32, mt, mt, o, i, desc, scale_shape=(o, groups),
                         has_zero_point_tensor=zero_point, has_bias=bias, max_tokens=total, **kw)
        op.bind(srcs, [dst])
        op.set_shape(1, rows or 1, tokens)
        self.keep.append(op)
        return op

    def launch(self, stream):
        for step in self.steps:
            step(stream)

    def capture(self):
        """One pass as a HIP graph (after a first pass outside of it)."""
        self.launch(torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            self.launch(torch.cuda.current_stream().cuda_stream)
        self.graph = graph


def _stack(p, c):
    tokens, hidden, kv, mlp, group = c["tokens"], c["hidden"], c["kv"], c["mlp"], c["group"]
    x, y = p.act(hidden, tokens), p.act(mlp, tokens)
    desc = lambda n, k: M.fc_int4_weights_desc(n, k, decode=tokens == 1)  # (the layout for ops that run one token)
    shapes = [(x, hidden, hidden), (x, kv, hidden), (x, kv, hidden), (x, hidden, hidden), (x, mlp, hidden), (x, mlp, hidden),
              (y, hidden, mlp)]  # q, k, v, o, gate, up, down
    # the results of one projection over the layers, in one tensor
    outs = [torch.zeros((c["layers"], _slices(n), tokens, 4), dtype=torch.float16, device="cuda") for _, n, _k in shapes]
    p.outputs += outs
    for layer in range(c["layers"]):
        ops = [p.fc(src, n, k, tokens, desc(n, k), group, dst=outs[i][layer]) for i, (src, n, k) in enumerate(shapes)]
        for first, last in ((0, 3), (3, 4), (4, 6), (6, 7)):
            p.steps.append(lambda s, together=ops[first:last]: _launch_group(together, s))


def _launch_group(ops, stream):
    """The ops of a layer that read one tensor: one launch where the library can serve them together."""
    if len(ops) > 1:
        try:
            M.fc_launch_fused(ops, stream)
            return
        except M.MldhipError as e:
            if e.code != M.FAILED_PRECONDITION:
                raise
    for op in ops:
        op.launch(stream)


def _mlp(p, c):
    tokens, hidden, mlp = c["tokens"], c["hidden"], c["mlp"]
    x = p.act(hidden, tokens)
    unused = torch.zeros((_slices(mlp), tokens, 4), dtype=torch.float16, device="cuda")  # (a gated launch writes its own dst)
    p.keep.append(unused)
    desc = lambda n, k: M.fc_int4_weights_desc(n, k, decode=tokens == 1)
    for _ in range(c["layers"]):
        gate = p.fc(x, mlp, hidden, tokens, desc(mlp, hidden), dst=unused)
        up = p.fc(x, mlp, hidden, tokens, desc(mlp, hidden), dst=unused)
        h = p.out(mlp, tokens)
        down = p.fc(h, hidden, mlp, tokens, desc(hidden, mlp))
        p.steps.append(lambda s, g=gate, u=up, d=h: M.fc_launch_gated(g, u, M.GATE_SILU, d, s))
        p.steps.append(down.launch)


def _int8(p, c):
    m, k, n = c["tokens"], c["k"], c["n"]
    k16, ns = (k + 15) // 16, _slices(n)
    src = p.act(k, m)
    codes = torch.zeros((k16, m, 16), dtype=torch.int8, device="cuda")
    params = torch.zeros((m, 4), dtype=torch.float32, device="cuda")
    quant = M.quantization_create(M.FLOAT16, M.PACKED_INT8C16, k, calculate_sum=False, symmetric=c["symmetric"], max_tokens=m)
    quant.bind([src], [codes, params])
    quant.set_shape(1, 1, m)
    w = torch.randint(-127, 128, (k16, n, 16), dtype=torch.int8, device="cuda", generator=p.gen)
    if k % 16:
        w[-1, :, k % 16:] = 0
    wsum = torch.zeros((ns * 4,), dtype=torch.int32, device="cuda")
    wsum[:n] = w.sum(dim=(0, 2), dtype=torch.int32)
    conv = M.conv_int8_create(M.FLOAT16, n, k, M.conv_int8_weights_desc(n, k), max_tokens=m)
    dst = p.out(n, m)
    conv.bind([codes, w, params, wsum, p.scale((ns * 4,), n, 127.0, torch.float32)], [dst])
    conv.set_shape(1, 1, m)
    p.outputs += [codes, params]
    p.keep += [quant, conv, w, wsum]
    p.steps += [quant.launch, conv.launch]


def _moe_decode(p, c):
    experts, top, hidden, mlp, group = c["experts"], c["top"], c["hidden"], c["mlp"], c["group"]
    x, h = p.act(hidden, 1), p.act(mlp, top)
    for _ in range(c["layers"]):
        ids = torch.randperm(experts, generator=p.gen, device="cuda")[:top].to(torch.int32)
        p.keep.append(ids)
        kw = dict(group=group, batch=experts, rows=top, ids=ids)
        gate = p.fc(x, mlp, hidden, 1, M.fc_int4_weights_desc(mlp, hidden), shared_src=True, **kw)
        up = p.fc(x, mlp, hidden, 1, M.fc_int4_weights_desc(mlp, hidden), shared_src=True, **kw)
        down = p.fc(h, hidden, mlp, 1, M.fc_int4_weights_desc(hidden, mlp), **kw)
        p.steps += [gate.launch, up.launch, down.launch]


def _moe_prefill(p, c):
    tokens, experts, top, hidden, mlp, group = c["tokens"], c["experts"], c["top"], c["hidden"], c["mlp"], c["group"]
    rows = tokens * top
    # every token picks `top` different experts, some of them more popular than others
    odds = torch.rand((experts,), device="cuda", generator=p.gen) + 0.25
    keys = torch.rand((tokens, experts), device="cuda", generator=p.gen) ** (1.0 / odds)
    picks = keys.topk(top, dim=1).indices
    sizes = torch.bincount(picks.reshape(-1), minlength=experts)
    params = torch.cat([sizes, sizes.cumsum(0) - sizes]).to(torch.int32)
    p.keep.append(params)
    kw = dict(group=group, batch=experts, packed=(0, experts, tokens), params=params)
    x, h = p.act(hidden, rows), p.act(mlp, rows)
    gate = p.fc(x, mlp, hidden, rows, M.fc_int4_weights_desc(mlp, hidden), **kw)
    up = p.fc(x, mlp, hidden, rows, M.fc_int4_weights_desc(mlp, hidden), **kw)
    down = p.fc(h, hidden, mlp, rows, M.fc_int4_weights_desc(hidden, mlp), **kw)
    p.steps += [gate.launch, up.launch, down.launch]


def _kv_ring(p, c):
    heads, positions, dim = c["heads"], c["positions"], c["head_dim"]
    query = p.act(dim, heads)
    probs = torch.softmax(torch.randn((positions, heads), device="cuda", generator=p.gen) * 2.0, dim=0)
    probs = probs.to(torch.float16).view(positions // 4, 4, heads).transpose(1, 2).contiguous()
    params = torch.randint(0, positions, (1,), device="cuda", generator=p.gen).to(torch.int32)  # where the ring starts
    p.keep += [probs, params]
    for _ in range(c["layers"]):
        for axis in "oi":
            # keys: [positions] output channels of [dim] inputs; values: [dim] output channels of [positions] inputs
            o, i = (positions, dim) if axis == "o" else (dim, positions)
            desc = M.make_desc(M.UINT8, M.LAYOUT_O4I4 if axis == "o" else M.LAYOUT_I4O4, _slices(o))
            kw = {"ring_%s_offset_index" % axis: 0, "ring_size": positions}
            kw.update(dict(dst_channels=o) if axis == "o" else dict(src_channels=i))
            op = M.fc_create(M.PRECISION_F32_F16, M.FLOAT16, M.FLOAT16, o, i, desc, scale_shape=(o, 1), max_tokens=heads, **kw)
            dst = p.out(o, heads)
            op.bind([query if axis == "o" else probs, p.codes(desc, o, 1, i), p.scale((_slices(o) * 4,), o, 127.0), params], [dst])
            op.set_shape(1, 1, heads)
            p.keep.append(op)
            p.steps.append(op.launch)


def prepare(case, seed):
    p = _Program(seed)
    kind = case["kind"]
    graph = False
    if kind == "f32_u8":
        m, k, n = case["tokens"], case["k"], case["n"]
        op = p.fc(p.act(k, m, torch.float32), n, k, m, M.fc_int8_weights_desc(n, k, decode=m == 1), dtype=torch.float32,
                      bias=case["bias"], zero_point=case["zero_point"])
        p.steps.append(op.launch)
    elif kind == "fc":
        m, k, n = case["tokens"], case["k"], case["n"]
        desc = M.fc_int8_weights_desc(n, k) if case["bits"] == 8 else M.fc_int4_weights_desc(n, k)
        op = p.fc(p.act(k, m), n, k, m, desc, case["group"], bias=case["bias"], zero_point=case["zero_point"])
        p.steps.append(op.launch)
    elif kind == "stack":
        _stack(p, case)
        graph = case["tokens"] <= 16
    elif kind == "mlp":
        _mlp(p, case)
        graph = True
    elif kind == "int8":
        _int8(p, case)
    elif kind == "moe_decode":
        _moe_decode(p, case)
        graph = True
    elif kind == "moe_prefill":
        _moe_prefill(p, case)
    else:
        _kv_ring(p, case)
        graph = True
    p.graph = None
    if graph:
        p.capture()
    return p


def run(state):
    if state.graph is not None:
        state.graph.replay()
    else:
        state.launch(torch.cuda.current_stream().cuda_stream)
    return state.outputs


# ---------------------------------------------------------------------------------------------------
# What a pass cannot do without, and what may differ
# ---------------------------------------------------------------------------------------------------


def _fc_work(tokens, k, n, bits, group=0, size=2, zero_point=False, bias=False, act=True):
    """One FullyConnected: packed weights, scales (zero points, bias), activations in, results out."""
    groups = k // group if group else 1
    b = n * k * bits // 8 + n * groups * size * (2 if zero_point else 1) + (n * size if bias else 0)
    b += (tokens * k * size if act else 0) + tokens * n * size
    return b, 2.0 * tokens * k * n


def work(case):
    kind = case["kind"]
    if kind in ("f32_u8", "fc"):
        parts = [_fc_work(case["tokens"], case["k"], case["n"], case.get("bits", 8), case.get("group", 0), 4 if kind == "f32_u8" else 2,
                          case["zero_point"], case["bias"])]
    elif kind == "stack":
        m, h, kv, f, g = case["tokens"], case["hidden"], case["kv"], case["mlp"], case["group"]
        # (q, k, v, o, gate and up read one activation tensor, down another; they stay the same over the layers)
        shapes = [(h, h), (h, kv), (h, kv), (h, h), (h, f), (h, f), (f, h)]
        parts = [_fc_work(m, k, n, 4, g, act=False) for k, n in shapes] * case["layers"] + [(2 * m * (h + f), 0.0)]
    elif kind == "mlp":
        m, h, f = case["tokens"], case["hidden"], case["mlp"]
        pair = _fc_work(m, h, f, 4, act=False)
        gated = (2 * pair[0] - 2 * m * f, 2 * pair[1])  # one output for the two matrices
        parts = [gated, _fc_work(m, f, h, 4)] * case["layers"] + [(2 * m * h, 0.0)]
    elif kind == "int8":
        m, k, n = case["tokens"], case["k"], case["n"]
        # activations in, codes out and in, parameters out and in, weights, sums and scales, results
        parts = [(2 * m * k + 2 * m * k + 2 * 16 * m + n * k + 8 * n + 2 * m * n, 2.0 * m * k * n)]
    elif kind == "moe_decode":
        h, f, g, t = case["hidden"], case["mlp"], case["group"], case["top"]
        one = [_fc_work(1, h, f, 4, g, act=False)] * (2 * t) + [_fc_work(1, f, h, 4, g, act=False)] * t
        parts = one * case["layers"] + [(2 * h + 2 * t * f, 0.0)]
    elif kind == "moe_prefill":
        h, f, g, rows = case["hidden"], case["mlp"], case["group"], case["tokens"] * case["top"]
        weights = min(case["experts"], rows) * (h * f // 2 + 2 * h * f // g)  # (of one projection)
        # three projections; gate and up read one tensor
        parts = [(3 * weights + 2 * rows * (h + f + 2 * f + h), 6.0 * rows * h * f)]
    else:
        m, pos, d = case["heads"], case["positions"], case["head_dim"]
        parts = [_fc_work(m, d, pos, 8, act=False), _fc_work(m, pos, d, 8, act=False)] * case["layers"] + [(2 * m * (pos + d), 0.0)]
    return {"bytes": float(sum(b for b, _ in parts)), "flops": float(sum(f for _, f in parts))}


def tolerance(case):
    kind = case["kind"]
    if kind == "int8":
        return "exact"  # codes, sums and the rescale's order of operations are fixed bit for bit
    # about four times the error against the product in float64: 2.0e-7 (largest 1.0e-6 of the output's root mean
    # square) with fp32 tensors, 2.1e-4 .. 2.8e-4 (5e-4 .. 1.5e-3) with fp16 ones, most of it the rounding of the
    # fp16 results and, in the products over many tokens, of the dequantized weights
    if kind == "f32_u8":
        return {"rel": 1e-6, "max": 5e-6}
    return {"rel": 1.2e-3, "max": 6e-3}
