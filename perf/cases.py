"""The work a user of this library has it do, as cases to time.

A case is a dict of plain values; "op" names its kind.  prepare() puts the operands of one case into HBM (torch tensors,
handed to the library by address) and run() makes the operator calls of one pass on the stream torch works on, without
waiting for them, as an inference program or a conformance run does.  One library context serves the whole process.
"""
import math

import torch

from reference_model_amd import Context, capi

TYPES = {  # name: (element type of the library, torch type, bytes)
    "int8": (capi.INT8, torch.int8, 1), "int16": (capi.INT16, torch.int16, 2), "fp16": (capi.FP16, torch.float16, 2),
    "bf16": (capi.BF16, torch.bfloat16, 2), "fp32": (capi.FP32, torch.float32, 4)}
DEVICE = "cuda:0"

_context = None


def context():
    """The process's library context, on the stream torch works on."""
    global _context
    if _context is None:
        _context = Context(0)
        _context.set_stream(torch.cuda.current_stream().cuda_stream)
    return _context


# ---- the cases --------------------------------------------------------------------------------------------------------

def listed():
    return [
        # The smallest call: the int8 1x1 layer of the reference's example graph.  A conformance run makes thousands of
        # calls of this size; launch and host time are all there is.
        dict(name="conv1x1_int8_example", op="conv", n=1, h=32, w=32, ic=8, oc=16, k=1, stride=1, in_zp=-3, out_zp=5, clamp=False,
             shift_lo=36, shift_hi=40),
        # The headline layer: an int8 3x3 of a residual stage with its RESCALE and a fused ReLU.
        dict(name="conv3x3_int8", op="conv", n=8, h=56, w=56, ic=64, oc=64, k=3, stride=1, in_zp=-7, out_zp=0, clamp=True,
             shift_lo=38, shift_hi=38),
        # A depthwise layer at serving batch: bandwidth.
        dict(name="depthwise_int8", op="depthwise", n=64, h=112, w=112, ic=96, k=3, stride=2, in_zp=4, out_zp=0, clamp=False,
             shift_lo=34, shift_hi=40),
        # A whole mobile network on one image: latency over some fifty small layers.
        dict(name="mobilenetv2_int8_n1", op="network", net="mobilenetv2", n=1, size=224, width=1.0),
        # A whole residual classification network on a small batch (poolings and classifier included).
        dict(name="resnet50_int8_n8", op="network", net="resnet50", n=8, size=224, width=1.0),
        # An fp16 3x3 layer with a long reduction.
        dict(name="conv3x3_fp16", op="conv_fp", type="fp16", n=16, h=28, w=28, ic=256, oc=256, k=3, stride=1),
        # Batched int8 product with zero points, int32 results.
        dict(name="matmul_int8", op="matmul", type="int8", n=8, h=1024, c=1024, w=1024, a_zp=-5, b_zp=3),
        # The largest: a bf16 product bound by the matrix cores.
        dict(name="matmul_bf16", op="matmul", type="bf16", n=4, h=2048, c=4096, w=2048, a_zp=0, b_zp=0),
        # Ragged products: scores and values of an attention layer over 197 tokens (8 sequences, 12 heads of 64).
        dict(name="attention_fp16_197", op="attention", type="fp16", n=96, tokens=197, dim=64),
        # Upsampling in a decoder: TRANSPOSE_CONV2D, then RESCALE and CLAMP as calls of their own (it has no fused form).
        dict(name="upsample_int8", op="upsample", n=8, h=28, w=28, ic=128, oc=64, k=3, stride=2, in_zp=-7, out_zp=-5),
        # A layer of a network with 16-bit activations and 8-bit weights: INT48 sums, then RESCALE to INT16.
        dict(name="conv3x3_int16", op="conv_int16", n=8, h=56, w=56, ic=64, oc=64, k=3, stride=1),
        # The conformance flow of a floating-point layer: the result, its fp64 pass, its bounds pass, and the check.
        dict(name="compliance_conv3x3_fp32", op="compliance", layer="conv", type="fp32", n=16, h=28, w=28, ic=256, oc=256, k=3,
             stride=1),
    ]


def _log(rng, lo, hi):
    """an integer spread over the logarithm of [lo, hi]"""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _channels(rng, lo, hi):
    """a channel count: most networks have multiples of 8 or 16, some do not"""
    c = _log(rng, lo, hi)
    step = rng.choice((1, 8, 8, 16))
    return max(lo, (c + step - 1) // step * step)


def _drawn(rng):
    op = rng.choice(("conv", "conv", "depthwise", "network", "conv_fp", "matmul", "matmul", "attention", "upsample", "conv_int16",
                     "compliance"))
    zp = rng.randint(-20, 20)
    if op in ("conv", "depthwise"):
        h = _log(rng, 7, 160)
        lo = rng.randint(34, 38)
        case = dict(op=op, n=_log(rng, 1, 64), h=h, w=max(7, h + rng.choice((0, 0, 0, -3, 5))), ic=_channels(rng, 3, 640), k=rng.choice((1, 3, 3, 5)),
                    stride=rng.choice((1, 1, 2)), in_zp=zp, out_zp=rng.randint(-128, 20), clamp=rng.random() < 0.5, shift_lo=lo,
                    shift_hi=rng.randint(lo, 40))
        if op == "conv":
            case["oc"] = _channels(rng, 8, 640)
            if case["k"] == 1:
                case["stride"] = 1
        else:
            case["k"] = max(3, case["k"])
        return case
    if op == "network":
        return dict(op=op, net=rng.choice(("mobilenetv2", "resnet50")), n=_log(rng, 1, 16), size=rng.randint(96, 288),
                    width=rng.choice((0.5, 0.75, 1.0, 1.25)))
    if op == "matmul":
        t = rng.choice(("int8", "fp16", "bf16"))
        z = (rng.randint(-10, 10), rng.randint(-10, 10)) if t == "int8" else (0, 0)
        r = lambda v: (v + 15) // 16 * 16 if rng.random() < 0.5 else v  # noqa: E731
        return dict(op=op, type=t, n=_log(rng, 1, 64), h=r(_log(rng, 1, 2048)), c=r(_log(rng, 16, 4096)), w=r(_log(rng, 16, 4096)),
                    a_zp=z[0], b_zp=z[1])
    if op == "attention":
        return dict(op=op, type=rng.choice(("fp16", "bf16")), n=_log(rng, 4, 192), tokens=_log(rng, 17, 600),
                    dim=rng.choice((32, 40, 64, 80, 96, 128)))
    if op == "upsample":
        return dict(op=op, n=_log(rng, 1, 8), h=_log(rng, 7, 64), w=_log(rng, 7, 64), ic=_channels(rng, 16, 256), oc=_channels(rng, 8, 256),
                    k=rng.choice((2, 3, 3, 4)), stride=2, in_zp=zp, out_zp=rng.randint(-20, 20))
    case = dict(op=op, n=_log(rng, 1, 16), h=_log(rng, 7, 112), w=_log(rng, 7, 112), ic=_channels(rng, 8, 512), oc=_channels(rng, 8, 512),
                k=rng.choice((1, 3, 3)), stride=rng.choice((1, 1, 2)))
    if case["k"] == 1:
        case["stride"] = 1
    if op == "conv_fp":
        case["type"] = rng.choice(("fp16", "fp16", "bf16", "fp32"))
    if op == "compliance":
        case["type"] = rng.choice(("fp16", "bf16", "fp32"))
        case["layer"] = rng.choice(("conv", "conv", "depthwise", "matmul"))
        if case["layer"] == "depthwise":
            case["oc"], case["k"] = case["ic"], 3
        if case["layer"] == "matmul":    # n products of h x ic and ic x oc
            case.update(w=1, k=1, stride=1)
    return case


# the most operations and bytes of a drawn case of each kind: about the listed one's
_MOST = {"conv": (2e10, 1e8), "depthwise": (1e10, 1e8), "network": (1e11, 2e8), "conv_fp": (1.5e10, 1e8), "matmul": (1.3e11, 2e8),
         "attention": (1e11, 2e8), "upsample": (4e9, 5e7), "conv_int16": (2e9, 5e7), "compliance": (4.5e10, 1e8)}


def draw(rng):
    while True:
        case = _drawn(rng)
        w = work(case)
        if w["flops"] <= _MOST[case["op"]][0] and w["bytes"] <= _MOST[case["op"]][1]:
            return case


# ---- geometry ---------------------------------------------------------------------------------------------------------

def _same(size, k, stride):
    """output size and the two pads of a window that covers the image (SAME)"""
    out = -(-size // stride)
    pad = max(0, (out - 1) * stride + k - size)
    return out, pad // 2, pad - pad // 2


def _conv_shape(case):
    oh, top, bottom = _same(case["h"], case["k"], case["stride"])
    ow, left, right = _same(case["w"], case["k"], case["stride"])
    return oh, ow, (top, bottom, left, right)


def _layers(case):
    """(kind, h, ic, oc, k, stride, relu) of the layers of a classification network in the order they run; the shortcuts
    around its blocks are not operators of this library."""
    ch = lambda c: max(8, int(c * case["width"] + 4) // 8 * 8)  # noqa: E731
    hw, out = case["size"], []

    def add(kind, ic, oc, k, stride, relu=True):
        nonlocal hw
        out.append((kind, hw, ic, oc, k, stride, relu))
        hw = -(-hw // stride)
        return oc

    if case["net"] == "resnet50":
        c = add("conv", 3, ch(64), 7, 2)
        add("max_pool", c, c, 3, 2)
        for mid, blocks, stride in ((64, 3, 1), (128, 4, 2), (256, 6, 2), (512, 3, 2)):
            for b in range(blocks):
                c = add("conv", c, ch(mid), 1, 1)
                c = add("conv", c, ch(mid), 3, stride if b == 0 else 1)
                c = add("conv", c, ch(4 * mid), 1, 1)
    else:
        c = add("conv", 3, ch(32), 3, 2)
        add("depthwise", c, c, 3, 1)
        c = add("conv", c, ch(16), 1, 1, False)
        for oc, blocks, stride in ((24, 2, 2), (32, 3, 2), (64, 4, 2), (96, 3, 1), (160, 3, 2), (320, 1, 1)):
            for b in range(blocks):
                e = add("conv", c, 6 * c, 1, 1)
                add("depthwise", e, e, 3, stride if b == 0 else 1)
                c = add("conv", e, ch(oc), 1, 1, False)
        c = add("conv", c, max(1280, ch(1280)), 1, 1)
    out.append(("avg_pool", hw, c, c, hw, hw, False))
    out.append(("conv", 1, c, 1000, 1, 1, False))
    return out


# ---- operands ---------------------------------------------------------------------------------------------------------

class _Operands:
    """Seeded operands on the GPU."""

    def __init__(self, seed):
        self.gen = torch.Generator(device=DEVICE)
        self.gen.manual_seed(seed)

    def ints(self, lo, hi, shape, dtype):
        return torch.randint(lo, hi + 1, shape, generator=self.gen, device=DEVICE, dtype=torch.int32).to(dtype)

    def normal(self, std, shape, dtype):
        return (torch.randn(shape, generator=self.gen, device=DEVICE) * std).to(dtype)

    def weights(self, shape):
        """int8 weights as quantisation leaves them"""
        return self.normal(30, shape, torch.float32).round_().clamp_(-127, 127).to(torch.int8)

    def scales(self, channels, scale):
        """multiplier and shift of per-channel RESCALE factors spread around `scale`"""
        s = scale * (0.7 + 0.7 * torch.rand(channels, generator=self.gen, device=DEVICE, dtype=torch.float64))
        mantissa, exponent = torch.frexp(s)
        return (mantissa * 2.0 ** 31).to(torch.int64).clamp_(1 << 30, (1 << 31) - 1).to(torch.int32), (31 - exponent).to(torch.int8)


def _empty(shape, dtype):
    return torch.empty(shape, dtype=dtype, device=DEVICE)


def _conv_call(ctx, ops, depthwise, x, n, h, w, ic, oc, k, stride, in_zp, out_zp, clamp, mult, shift):
    """the fused int8 CONV2D / DEPTHWISE_CONV2D + RESCALE (+ CLAMP) call on x, and its result"""
    oh, ow, pad = _conv_shape(dict(h=h, w=w, k=k, stride=stride))
    wt = ops.weights((k, k, ic, 1) if depthwise else (oc, k, k, ic))
    bias = ops.normal(2 ** 10, (oc,), torch.float32).round_().to(torch.int32)
    out = _empty((n, oh, ow, oc), torch.int8)
    d = ctx.conv_desc(capi.INT8, capi.INT32, (n, h, w, ic), oc, k, k, (oh, ow), pad, (stride, stride), (1, 1), oc)
    r = ctx.rescale_desc(capi.INT32, capi.INT8, oc, oc, 0, out_zp)
    fn = ctx.depthwise_conv2d_rescale_clamp if depthwise else ctx.conv2d_rescale_clamp
    return (fn, (d, x, wt, bias, in_zp, 0, r, mult, shift, out, clamp)), out


def _pool_call(ctx, kind, x, n, h, c, k, stride):
    o, before, after = _same(h, k, stride)
    d = capi.PoolDesc()
    d.dtype, d.acc_dtype, d.nan_mode = capi.INT8, capi.INT32, 1
    d.N, d.IH, d.IW, d.C, d.OH, d.OW = n, h, h, c, o, o
    d.kernel[:], d.stride[:], d.pad[:] = [k, k], [stride, stride], [before, after, before, after]
    out = _empty((n, o, o, c), torch.int8)
    if kind == "max_pool":
        return (ctx.max_pool2d, (d, x, out)), out
    return (ctx.avg_pool2d, (d, x, -128, -128, out)), out


def _network(ctx, ops, case):
    n, zp, rms = case["n"], -3, 74.0    # the image: uniform bytes
    x = ops.ints(-128, 127, (n, case["size"], case["size"], 3), torch.int8)
    calls, outs = [], []
    for kind, h, ic, oc, k, stride, relu in _layers(case):
        if kind.endswith("pool"):
            call, x = _pool_call(ctx, kind, x, n, h, oc, k, stride)
        else:
            depthwise = kind == "depthwise"
            reach = k * k * (1 if depthwise else ic)
            mult, shift = ops.scales(oc, 50.0 / (30.0 * rms * math.sqrt(reach)))
            out_zp = -128 if relu else 3
            call, x = _conv_call(ctx, ops, depthwise, x, n, h, h, ic, oc, k, stride, zp, out_zp, (-128, 127) if relu else None, mult, shift)
            zp, rms = out_zp, 35.0 if relu else 50.0
        calls.append(call)
        outs.append(x)
    return calls, outs


def _float_layer(ctx, ops, case, dtype):
    """CONV2D / DEPTHWISE_CONV2D / MATMUL on floating-point operands: its call and what the fp64 passes need"""
    code, tt, _ = TYPES[dtype]
    n, h, w, ic, oc, k, stride = (case[q] for q in ("n", "h", "w", "ic", "oc", "k", "stride"))
    if case.get("layer") == "matmul":
        a, b = ops.normal(1.0, (n, h, ic), tt), ops.normal(1 / math.sqrt(ic), (n, ic, oc), tt)
        out = _empty((n, h, oc), torch.float32)
        return (ctx.matmul, (code, n, h, ic, oc, a, b, 0, 0, out)), out, capi.FP32, ic
    depthwise = case.get("layer") == "depthwise"
    oh, ow, pad = _conv_shape(case)
    reach = k * k * (1 if depthwise else ic)
    x = ops.normal(1.0, (n, h, w, ic), tt)
    wt = ops.normal(1 / math.sqrt(reach), (k, k, ic, 1) if depthwise else (oc, k, k, ic), tt)
    bias = ops.normal(0.1, (oc,), tt)
    out = _empty((n, oh, ow, oc), tt)
    d = ctx.conv_desc(code, code, (n, h, w, ic), oc, k, k, (oh, ow), pad, (stride, stride), (1, 1), oc)
    return (ctx.depthwise_conv2d if depthwise else ctx.conv2d, (d, x, wt, bias, 0, 0, out)), out, code, reach + 1


def prepare(case, seed):
    ctx, ops, op = context(), _Operands(seed), case["op"]
    if op in ("conv", "depthwise"):
        oc = case.get("oc", case["ic"])
        x = ops.ints(-128, 127, (case["n"], case["h"], case["w"], case["ic"]), torch.int8)
        mult = ops.ints(1 << 30, (1 << 31) - 2, (oc,), torch.int32)
        shift = ops.ints(case["shift_lo"], case["shift_hi"], (oc,), torch.int8)
        call, out = _conv_call(ctx, ops, op == "depthwise", x, case["n"], case["h"], case["w"], case["ic"], oc, case["k"], case["stride"],
                               case["in_zp"], case["out_zp"], (max(0, case["out_zp"]), 127) if case["clamp"] else None, mult, shift)
        return dict(calls=[call], out=out)
    if op == "network":
        calls, outs = _network(ctx, ops, case)
        return dict(calls=calls, out=outs)
    if op == "conv_fp":
        call, out, _, _ = _float_layer(ctx, ops, case, case["type"])
        return dict(calls=[call], out=out)
    if op == "matmul":
        code, tt, _ = TYPES[case["type"]]
        n, h, c, w = (case[q] for q in "nhcw")
        if tt == torch.int8:
            a, b = ops.ints(-128, 127, (n, h, c), tt), ops.ints(-128, 127, (n, c, w), tt)
        else:
            a, b = ops.normal(1 / 64, (n, h, c), tt), ops.normal(1 / 64, (n, c, w), tt)
        out = _empty((n, h, w), torch.int32 if tt == torch.int8 else torch.float32)
        return dict(calls=[(ctx.matmul, (code, n, h, c, w, a, b, case["a_zp"], case["b_zp"], out))], out=out)
    if op == "attention":
        code, tt, _ = TYPES[case["type"]]
        n, t, dim = case["n"], case["tokens"], case["dim"]
        q, k, v = ops.normal(1.0, (n, t, dim), tt), ops.normal(1.0, (n, dim, t), tt), ops.normal(1.0, (n, t, dim), tt)
        p = torch.softmax(ops.normal(1.0, (n, t, t), torch.float32), -1).to(tt)
        scores, values = _empty((n, t, t), torch.float32), _empty((n, t, dim), torch.float32)
        return dict(calls=[(ctx.matmul, (code, n, t, dim, t, q, k, 0, 0, scores)), (ctx.matmul, (code, n, t, t, dim, p, v, 0, 0, values))],
                    out=[scores, values])
    if op == "upsample":
        return _upsample(ctx, ops, case)
    if op == "conv_int16":
        n, h, w, ic, oc, k, stride = (case[q] for q in ("n", "h", "w", "ic", "oc", "k", "stride"))
        oh, ow, pad = _conv_shape(case)
        x = ops.normal(8000, (n, h, w, ic), torch.float32).round_().clamp_(-32768, 32767).to(torch.int16)
        wt = ops.weights((oc, k, k, ic))
        bias = ops.normal(2 ** 20, (oc,), torch.float32).round_().to(torch.int64)
        acc, out = _empty((n, oh, ow, oc), torch.int64), _empty((n, oh, ow, oc), torch.int16)
        d = ctx.conv_desc(capi.INT16, capi.INT48, (n, h, w, ic), oc, k, k, (oh, ow), pad, (stride, stride), (1, 1), oc)
        # 16-bit scales (INT48 input takes no others); results spread over the 16 bits
        mult, shift = ops.scales(oc, 1 / (30.0 * math.sqrt(k * k * ic)))
        mult, shift = (mult >> 16).to(torch.int16), shift - 16
        r = ctx.rescale_desc(capi.INT48, capi.INT16, oc, oc, 0, 0, scale32=False, rounding_mode=capi.ROUND_SINGLE)
        return dict(calls=[(ctx.conv2d, (d, x, wt, bias, 0, 0, acc)), (ctx.rescale, (r, 4, n * oh * ow, oc, acc, mult, shift, out))],
                    out=[acc, out])
    call, out, code, terms = _float_layer(ctx, ops, case, case["type"])
    ref, bound = (_empty(out.shape, torch.float64) for _ in range(2))
    args = call[1]
    if case["layer"] == "matmul":
        passes = [(ctx.matmul_precise, args[:7] + (bounds, to)) for bounds, to in ((False, ref), (True, bound))]
    else:
        passes = [(ctx.conv2d_precise, args[:4] + (bounds, to, case["layer"] == "depthwise")) for bounds, to in ((False, ref), (True, bound))]
    return dict(calls=[call] + passes, out=[out, ref, bound], check=(ctx.dot_product_check, (code, out.numel(), out, ref, bound, terms)))


def _upsample(ctx, ops, case):
    n, h, w, ic, oc, k, s = (case[q] for q in ("n", "h", "w", "ic", "oc", "k", "stride"))
    crop = s - k    # so that the result has s times the input's height and width
    lo, hi = -(-crop // 2), crop // 2
    x = ops.ints(-128, 127, (n, h, w, ic), torch.int8)
    wt = ops.weights((oc, k, k, ic))
    bias = ops.normal(2 ** 14, (oc,), torch.float32).round_().to(torch.int32)
    acc = _empty((n, h * s, w * s, oc), torch.int32)
    scaled, out = (_empty(acc.shape, torch.int8) for _ in range(2))
    d = capi.TconvDesc()
    d.in_dtype, d.out_dtype = capi.INT8, capi.INT32
    d.N, d.IH, d.IW, d.IC, d.OC, d.KH, d.KW, d.OH, d.OW = n, h, w, ic, oc, k, k, h * s, w * s
    d.out_pad[:], d.stride[:], d.bias_len = [lo, hi, lo, hi], [s, s], oc
    mult, shift = ops.scales(oc, 50.0 / (30.0 * 74.0 * math.sqrt(max(1, k * k // (s * s)) * ic)))
    r = ctx.rescale_desc(capi.INT32, capi.INT8, oc, oc, 0, case["out_zp"])
    return dict(calls=[(ctx.transpose_conv2d, (d, x, wt, bias, case["in_zp"], 0, acc)),
                       (ctx.rescale, (r, 4, n * h * w * s * s, oc, acc, mult, shift, scaled)),
                       (ctx.clamp, (capi.INT8, scaled.numel(), scaled, case["out_zp"], 127, out))], out=[acc, scaled, out])


def run(state):
    for fn, args in state["calls"]:
        fn(*args)
    if "check" not in state:
        return state["out"]
    fn, args = state["check"]
    verdict = fn(*args)
    return state["out"] + [int(verdict.failed_elements), int(verdict.compliant)]


# ---- what a pass cannot do without ------------------------------------------------------------------------------------

def work(case):
    """Multiply-adds count as two operations; every call reads its operands and writes its result once."""
    op = case["op"]
    if op == "network":
        size, flops = 0, 0
        for kind, h, ic, oc, k, stride, _ in _layers(case):
            o = -(-h // stride)
            size += case["n"] * (h * h * ic + o * o * oc)
            if not kind.endswith("pool"):
                per = k * k * (1 if kind == "depthwise" else ic)
                size += oc * (per + 9)
                flops += 2 * case["n"] * o * o * oc * per
        return dict(bytes=size, flops=flops)
    if op == "matmul":
        n, h, c, w = (case[q] for q in "nhcw")
        return dict(bytes=n * (TYPES[case["type"]][2] * (h * c + c * w) + 4 * h * w), flops=2 * n * h * c * w)
    if op == "attention":
        n, t, dim = case["n"], case["tokens"], case["dim"]
        return dict(bytes=n * (2 * (3 * t * dim + t * t) + 4 * (t * t + t * dim)), flops=4 * n * t * t * dim)
    n, h, w, ic, k, s = (case[q] for q in ("n", "h", "w", "ic", "k", "stride"))
    oc = case.get("oc", ic)
    if op == "upsample":
        results = n * h * w * s * s * oc
        return dict(bytes=n * h * w * ic + oc * (k * k * ic + 9) + results * (4 + 5 + 2), flops=2 * n * h * w * ic * oc * k * k)
    oh, ow, _ = _conv_shape(case)
    depthwise = op == "depthwise" or case.get("layer") == "depthwise"
    reach = k * k * (1 if depthwise else ic)
    results, macs = n * oh * ow * oc, n * oh * ow * oc * reach
    if op in ("conv", "depthwise"):
        return dict(bytes=n * h * w * ic + oc * (reach + 9) + results, flops=2 * macs)
    if op == "conv_int16":
        return dict(bytes=2 * n * h * w * ic + oc * (reach + 11) + results * (8 + 8 + 2), flops=2 * macs)
    size = TYPES[case["type"]][2]
    matmul = case.get("layer") == "matmul"
    operands = size * (n * h * w * ic + (n * ic * oc if matmul else oc * (reach + 1)))
    result = results * (4 if matmul else size)
    if op == "conv_fp":
        return dict(bytes=operands + result, flops=2 * macs)
    return dict(bytes=3 * operands + 2 * result + 4 * 8 * results, flops=6 * macs)


def tolerance(case):
    """Whole numbers are the reference's bit for bit.  Floating-point sums are fp32 whatever the operands are; a 16-bit
    result may fall either side of a rounding."""
    kind = case.get("type", "int8")
    if kind == "int8" or case["op"] == "conv_int16":
        return "exact"
    if case.get("layer") == "matmul" or case["op"] in ("matmul", "attention"):
        return {"rel": 1e-5}    # fp32 results
    return {"rel": {"fp16": 5e-4, "bf16": 4e-3, "fp32": 1e-5}[kind]}
