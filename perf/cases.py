"""Workloads that stand for how this framework is used, for timing it.

Each case is one pass through the public entry points of `poplibs_amd`, on
tensors that live in HBM: an inference layer, a layer's share of a training
step (forward, input gradient, weight deltas, bias update), or a matrix
product.  Hidden layers keep their activations channels-last from one layer to
the next, the way `createInput` hands them out; only a network's first layer
takes the `[B][C][H][W]` tensor a data loader delivers.

`listed()` holds the fixed cases, `draw()` makes more of the same kinds,
`prepare()` builds what a program holds before the call, `run()` makes the
call.
"""
import math

import torch

import poplibs_amd as pa
from poplibs_amd import capi

TYPES = {"quarter": pa.QUARTER, "half": pa.HALF, "float": pa.FLOAT}

# No drawn case costs more than the largest listed ones, nor moves less than
# the smallest.
MAX_FLOPS = 2 * 4096 ** 3
MAX_BYTES = 350e6
MIN_BYTES = 140e3


def _conv(kind, name, batch, field, kernel, ci, co, groups=1, stride=1,
          type="half", bias=True, nchw=False):
    """A convolution case; `field` square, padded by (kernel - 1) // 2.
    Channel counts are per conv group."""
    case = {"kind": kind, "type": type, "batch": batch, "field": field,
            "kernel": kernel, "in_chans": ci, "out_chans": co,
            "groups": groups, "stride": stride, "bias": bias, "nchw": nchw}
    return dict(case, name=name) if name else case


def _matmul(name, m, k, n, type="half"):
    case = {"kind": "matmul", "type": type, "m": m, "k": k, "n": n}
    return dict(case, name=name) if name else case


def listed():
    return [
        # The smallest call: one small image through a small float layer, where
        # the cost of issuing the call and of the launch is all there is.
        _conv("forward", "one_image_3x3_fp32", 1, 32, 3, 16, 16,
              type="float", bias=False),
        # The three layers a residual network is made of: 3x3, 1x1 ...
        _conv("forward", "resnet_3x3_fp16", 32, 28, 3, 128, 128),
        _conv("forward", "resnet_1x1_fp16", 32, 56, 1, 256, 64),
        # ... and a deep 3x3 layer in fp8 with per-tensor scales.
        _conv("forward", "resnet_3x3_fp8", 64, 14, 3, 256, 256,
              type="quarter"),
        # A depthwise layer of a mobile network.
        _conv("forward", "mobilenet_depthwise_fp16", 32, 112, 3, 1, 1,
              groups=96, stride=2),
        # A layer that fills the chip several times over: throughput serving
        # or a large training batch.
        _conv("forward", "large_batch_3x3_fp16", 128, 28, 3, 256, 256),
        # A network's first layer on images as the data loader delivers them.
        _conv("forward", "first_layer_nchw_fp16", 32, 224, 7, 3, 64, stride=2,
              nchw=True),
        # One layer's share of a training step.
        _conv("train", "train_3x3_fp16", 32, 28, 3, 128, 128),
        # The same for a downsampling layer, on an odd field, an odd batch and
        # channel counts that fill no tile.
        _conv("train", "train_downsample_odd_fp16", 25, 57, 3, 72, 200,
              stride=2),
        # ... and for a depthwise layer.
        _conv("train", "train_depthwise_fp16", 32, 56, 3, 1, 1, groups=144),
        # matMul with weights that stay: a few rows (decoding tokens) ...
        _matmul("matmul_few_rows_fp16", 16, 4096, 4096),
        # ... and many (a training batch, a prompt).
        _matmul("matmul_many_rows_fp16", 4096, 4096, 4096),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _chans(rng, lo, hi):
    """Mostly whole vectors of 8 channels, one time in eight whatever comes."""
    c = _log_int(rng, lo, hi)
    return c if rng.random() < 0.125 else max(8, (c + 4) // 8 * 8)


def _draw_any(rng):
    family = rng.choice(("fp32", "dense", "dense", "fp8", "depthwise", "first",
                         "train", "train", "train_depthwise", "matmul",
                         "matmul"))
    bias = rng.random() < 0.75
    if family == "fp32":
        return _conv("forward", "", _log_int(rng, 1, 16), _log_int(rng, 8, 64),
                     rng.choice((1, 3, 3, 5)), _chans(rng, 16, 256),
                     _chans(rng, 16, 256), type="float", bias=bias,
                     stride=rng.choice((1, 1, 2)))
    if family == "dense":
        return _conv("forward", "", _log_int(rng, 1, 128),
                     _log_int(rng, 7, 64), rng.choice((1, 1, 3, 3, 5)),
                     _chans(rng, 32, 768), _chans(rng, 32, 768), bias=bias,
                     stride=rng.choice((1, 1, 1, 2)))
    if family == "fp8":
        return _conv("forward", "", _log_int(rng, 1, 128),
                     _log_int(rng, 7, 64), rng.choice((1, 3)),
                     16 * _log_int(rng, 4, 32), 16 * _log_int(rng, 4, 32),
                     type="quarter", bias=bias,
                     stride=rng.choice((1, 1, 2)))
    if family == "depthwise":
        return _conv("forward", "", _log_int(rng, 1, 64),
                     _log_int(rng, 7, 112), rng.choice((3, 3, 5, 7)), 1, 1,
                     groups=8 * _log_int(rng, 4, 120), bias=bias,
                     stride=rng.choice((1, 2)))
    if family == "first":
        return _conv("forward", "", _log_int(rng, 1, 64),
                     _log_int(rng, 64, 256), rng.choice((3, 5, 7)), 3,
                     rng.choice((16, 32, 48, 64)), bias=bias, nchw=True,
                     stride=rng.choice((1, 2, 2)))
    if family == "train":
        groups = rng.choice((1, 1, 1, 1, 32))
        if groups == 32:
            ci = co = rng.choice((4, 8, 16))
        else:
            ci, co = _chans(rng, 32, 512), _chans(rng, 32, 512)
        return _conv("train", "", _log_int(rng, 4, 64), _log_int(rng, 7, 64),
                     rng.choice((1, 3, 3)), ci, co, groups=groups, bias=bias,
                     stride=rng.choice((1, 1, 2)),
                     type=rng.choice(("half", "half", "half", "half",
                                      "float")))
    if family == "train_depthwise":
        return _conv("train", "", _log_int(rng, 4, 64),
                     _log_int(rng, 7, 112), rng.choice((3, 3, 5)), 1, 1,
                     groups=8 * _log_int(rng, 4, 120), bias=bias,
                     stride=rng.choice((1, 2)))
    return _matmul("", _log_int(rng, 1, 4096), _chans(rng, 128, 8192),
                   _chans(rng, 128, 8192))


def draw(rng):
    while True:
        case = _draw_any(rng)
        w = work(case)
        # Float runs at a sixteenth of half's rate on the matrix cores; a
        # training step's passes are the costlier ones per operation and byte.
        passes = 3 if case["kind"] == "train" else 1
        rate = 16 if case["type"] == "float" else 1
        if (w["flops"] * passes * rate <= MAX_FLOPS
                and w["bytes"] * passes <= MAX_BYTES
                and w["bytes"] >= MIN_BYTES):
            return case


def _params(case):
    if case["kind"] == "matmul":
        t = TYPES[case["type"]]
        return pa.matMulParams(t, t, 1, case["m"], case["k"], case["n"])
    in_type = TYPES[case["type"]]
    out_type = pa.HALF if in_type == pa.QUARTER else in_type
    p = pa.ConvParams(in_type, out_type, case["batch"], [case["field"]] * 2,
                      [case["kernel"]] * 2, case["in_chans"],
                      case["out_chans"], case["groups"])
    p.inputTransform.paddingLower = [(case["kernel"] - 1) // 2] * 2
    p.inputTransform.paddingUpper = [(case["kernel"] - 1) // 2] * 2
    p.outputTransform.stride = [case["stride"]] * 2
    return p


def _sizes(p):
    """Elements of a layer's input, weights and output."""
    taps = pixels = out_pixels = 1
    for k, f, o in zip(p.kernelShape, p.inputFieldShape,
                       p.getOutputFieldShape()):
        taps, pixels, out_pixels = taps * k, pixels * f, out_pixels * o
    return (p.batchSize * pixels * p.getNumInputChans(),
            p.getNumOutputChans() * p.inputChannelsPerConvGroup * taps,
            p.batchSize * out_pixels * p.getNumOutputChans())


def work(case):
    p = _params(case)
    n_in, n_w, n_out = _sizes(p)
    in_bytes = capi.TYPE_BYTES[p.inputType]
    out_bytes = capi.TYPE_BYTES[p.outputType]
    moved = (n_in + n_w) * in_bytes + n_out * out_bytes
    flops = p.getFwdFlops()
    if case["kind"] == "train":
        # the input, the weights and the output's gradient come in; the output
        # and the gradients of input and weights go out
        return {"bytes": 2 * moved, "flops": 3 * flops}
    return {"bytes": moved, "flops": flops}


def tolerance(case):
    # fp32 sums either way: float results differ by the order of summation,
    # half results by the rounding of the sum.
    return {"rel": 1e-5} if case["type"] == "float" else {"rel": 1e-3}


_TORCH = {pa.QUARTER: torch.uint8, pa.HALF: torch.float16,
          pa.FLOAT: torch.float32}


class _Layer:
    """What every program holds: device tensors, made from a seed."""

    def __init__(self, case, seed):
        self.dev = torch.device("cuda:0")
        self.gen = torch.Generator(device=self.dev).manual_seed(seed)
        self.stream = torch.cuda.current_stream().cuda_stream
        self.p = _params(case)
        self.in_dtype = _TORCH[self.p.inputType]
        self.out_dtype = _TORCH[self.p.outputType]

    def normal(self, n, dtype, std=1.0, relu=False):
        x = torch.randn(n, generator=self.gen, device=self.dev)
        if relu:
            x.clamp_min_(0)
        return x.mul_(std).to(dtype)

    def quarter(self, n, std=1.0, relu=False):
        """E4M3 bytes and their metadata: a power-of-two scale that puts six
        standard deviations at the top of the format's range."""
        scale = math.ceil(math.log2(6 * std / 448.0))
        x = self.normal(n, torch.float32, std / 2.0 ** scale, relu)
        x = x.clamp_(-448, 448).to(torch.float8_e4m3fn).view(torch.uint8)
        return x, pa.quarter_metadata(1, scale)

    def empty(self, n, dtype):
        return torch.empty(max(n, 16), dtype=dtype, device=self.dev)[:n]

    def workspace(self, nbytes):
        return torch.empty(max(nbytes, 16), dtype=torch.uint8,
                           device=self.dev)


class _Forward(_Layer):
    """A layer of an inference program: the weights are packed once."""

    def __init__(self, case, seed):
        super().__init__(case, seed)
        p, self.nchw = self.p, case["nchw"]
        n_in, n_w, n_out = _sizes(p)
        self.plan = pa.Plan(p)
        std = math.sqrt(2.0 / (n_w // p.getNumOutputChans()))
        self.is_quarter = p.inputType == pa.QUARTER
        relu = not self.nchw  # (a hidden layer's input has been through one)
        if self.is_quarter:
            self.x, self.x_meta = self.quarter(n_in, relu=relu)
            weights, self.w_meta = self.quarter(n_w, std)
        else:
            self.x = self.normal(n_in, self.in_dtype, relu=relu)
            weights = self.normal(n_w, self.in_dtype, std)
        self.bias = (self.normal(p.getNumOutputChans(), self.out_dtype, 0.1)
                     if case["bias"] else None)
        self.packed = self.workspace(
            self.plan.buffer_bytes(capi.BUF_WEIGHTS_PACKED))
        self.plan.pack_weights(weights.data_ptr(), self.packed.data_ptr(),
                               self.stream)
        self.x_internal = (self.empty(n_in, self.in_dtype) if self.nchw
                           else self.x)
        self.y = self.empty(n_out, self.out_dtype)
        self.ws_bytes = self.plan.buffer_bytes(capi.BUF_WORKSPACE)
        self.ws = self.workspace(self.ws_bytes)

    def step(self):
        bias = self.bias.data_ptr() if self.bias is not None else None
        if self.nchw:
            self.plan.acts_to_internal(
                self.x.data_ptr(), self.x_internal.data_ptr(), self.stream)
        if self.is_quarter:
            self.plan.fwd_quarter(
                self.x_internal.data_ptr(), self.x_meta,
                self.packed.data_ptr(), self.w_meta, self.y.data_ptr(), bias,
                self.ws.data_ptr(), self.ws_bytes, self.stream)
        else:
            self.plan.fwd(
                self.x_internal.data_ptr(), self.packed.data_ptr(),
                self.y.data_ptr(), bias, self.ws.data_ptr(), self.ws_bytes,
                self.stream)
        return self.y


class _Train(_Layer):
    """A layer's share of a training step.  The weights have changed since the
    step before, so they are packed again for both directions."""

    def __init__(self, case, seed):
        super().__init__(case, seed)
        p = self.p
        n_in, n_w, n_out = _sizes(p)
        self.fwd_plan = pa.Plan(p, {"pass": "TRAINING_FWD"})
        self.bwd_plan = pa.Plan(pa.getGradientParams(p),
                                {"pass": "TRAINING_BWD"})
        self.wu_plan = pa.WeightUpdatePlan(p)
        std = math.sqrt(2.0 / (n_w // p.getNumOutputChans()))
        self.x = self.normal(n_in, self.in_dtype, relu=True)
        self.w = self.normal(n_w, self.in_dtype, std)
        self.dy = self.normal(n_out, self.out_dtype, 0.1)
        self.y = self.empty(n_out, self.out_dtype)
        self.dx = self.empty(n_in, self.out_dtype)
        self.w_turned = self.empty(n_w, self.in_dtype)
        self.dw = self.empty(n_w, self.out_dtype)

        def packed(plan):
            return self.workspace(plan.buffer_bytes(capi.BUF_WEIGHTS_PACKED))

        self.fwd_packed = packed(self.fwd_plan)
        self.bwd_packed = packed(self.bwd_plan)
        self.fwd_ws_bytes = self.fwd_plan.buffer_bytes(capi.BUF_WORKSPACE)
        self.bwd_ws_bytes = self.bwd_plan.buffer_bytes(capi.BUF_WORKSPACE)
        self.wu_ws_bytes = self.wu_plan.workspace_bytes()
        self.chans = p.getNumOutputChans()
        self.outer = n_out // self.chans
        self.bias_ws_bytes = pa.bias_update_workspace_bytes(self.outer,
                                                            self.chans)
        self.ws_bytes = max(self.fwd_ws_bytes, self.bwd_ws_bytes,
                            self.wu_ws_bytes, self.bias_ws_bytes)
        self.ws = self.workspace(self.ws_bytes)
        self.bias = (self.normal(self.chans, self.out_dtype, 0.1)
                     if case["bias"] else None)
        # The step updates the biases in place; at this rate they stay small
        # numbers over any number of steps on the same data.
        self.rate = -1e-3

    def step(self):
        s, ws, n = self.stream, self.ws.data_ptr(), self.ws_bytes
        x, w, dy = self.x.data_ptr(), self.w.data_ptr(), self.dy.data_ptr()
        turned = self.w_turned.data_ptr()
        fwd_packed = self.fwd_packed.data_ptr()
        bwd_packed = self.bwd_packed.data_ptr()
        bias = self.bias.data_ptr() if self.bias is not None else None
        self.fwd_plan.pack_weights(w, fwd_packed, s)
        self.fwd_plan.fwd(x, fwd_packed, self.y.data_ptr(), bias, ws, n, s)
        pa.weightsTransposeChansFlipXY(self.p, w, turned, s)
        self.bwd_plan.pack_weights(turned, bwd_packed, s)
        self.bwd_plan.fwd(dy, bwd_packed, self.dx.data_ptr(), None, ws, n, s)
        self.wu_plan.calculate_weight_deltas(dy, x, self.dw.data_ptr(), ws, n,
                                             s)
        if bias is None:
            return self.y, self.dx, self.dw
        pa.convolutionBiasUpdate(self.p.outputType, dy, self.outer,
                                 self.chans, self.p.outputType, bias,
                                 self.rate, ws, n, s)
        return self.y, self.dx, self.dw, self.bias


class _MatMul(_Layer):
    """C = A B with B, the weights, packed once."""

    def __init__(self, case, seed):
        super().__init__(case, seed)
        t = TYPES[case["type"]]
        m, k, n = case["m"], case["k"], case["n"]
        self.plan = pa.MatMulPlan(t, t, 1, m, k, n)
        self.a = self.normal(m * k, self.in_dtype)
        b = self.normal(k * n, self.in_dtype, 1 / math.sqrt(k))
        self.packed = self.workspace(
            self.plan.buffer_bytes(capi.BUF_WEIGHTS_PACKED))
        self.plan.pack_rhs(b.data_ptr(), self.packed.data_ptr(), self.stream)
        self.c = self.empty(m * n, self.out_dtype)
        self.ws_bytes = self.plan.buffer_bytes(capi.BUF_WORKSPACE)
        self.ws = self.workspace(self.ws_bytes)

    def step(self):
        self.plan.fwd(self.a.data_ptr(), self.packed.data_ptr(),
                      self.c.data_ptr(), None, self.ws.data_ptr(),
                      self.ws_bytes, self.stream)
        return self.c


def prepare(case, seed):
    return {"forward": _Forward, "train": _Train,
            "matmul": _MatMul}[case["kind"]](case, seed)


def run(state):
    return state.step()
