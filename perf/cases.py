"""The work a program of this framework has it do, as cases that can be timed one by one.

A case is one step of a network's forward / backward pass: a handful of calls through the public entry
points (`mshadow_amd.load_cases()`: the C ABI's fixed-function operations, and the C++ expression API where a
step is an expression or a half_t tensor), on tensors that are already in HBM. Six kinds of step:

  map          dst = A*B + 0.5f*F<sigmoid>(C) - D on float tensors, dst = A*B + C on half_t ones: any
               elementwise layer or update
  head         the classifier of a network: Softmax, SoftmaxGrad against the labels, and the gradient of the
               classifier's bias, sum_rows of that gradient
  channel_sum  sumall_except_dim<1> over an NCHW tensor: a convolution's bias gradient, batch statistics
  column_sum   sum_rows over a matrix: a dense layer's bias gradient
  pool         max pooling, and for float tensors its gradient (half_t: the forward pass of inference)
  patches      the two ends of a convolution as a matrix product: unpack_patch2col(pad(image)) of the forward
               pass and crop(pack_col2patch(matrix)) of the backward pass

The listed cases are the shapes of the repository's own benchmark and tests; `draw` gives others of the same
ranges, from one small minibatch to those.
"""
import math

import numpy as np
import torch

import mshadow_amd

LIB = mshadow_amd.load_cases()
HALF_ONE = 0x3C00   # 1.0 as binary16: the scale argument of a half_t reduction

# the longest any case runs is the classifier over a vocabulary of 32000; every other kind is bounded by the
# benchmark's shape of that kind
MOST_LOGITS = 8192 * 32000
MOST_MAP = 4096 * 4096
MOST_CHANNEL = 64 * 256 * 56 * 56
MOST_COLUMN = 16384 * 4096
MOST_PIXELS = 128 * 64 * 112 * 112
MOST_MATRIX = 2304 * 32 * 56 * 56
# (window, step, padding) of pooling layers and of convolutions
POOLS = ((3, 2), (2, 2), (3, 1), (3, 2), (2, 2), (5, 1))
CONVOLUTIONS = ((3, 1, 1), (3, 2, 1), (1, 1, 0), (3, 1, 0), (5, 1, 2), (7, 2, 3), (3, 1, 1))


class Tensor:
    """A torch tensor's memory under the attributes that the entry points read of a device buffer:
    the last dimension is the row, everything before it the rows."""

    def __init__(self, t):
        self.tensor = t
        self.ptr = t.data_ptr()
        self.shape = tuple(t.shape)
        self.cols = self.shape[-1]
        self.rows = t.numel() // self.cols
        self.stride = self.cols
        # half_t tensors travel as their 16-bit patterns
        self.dtype = np.dtype(np.uint16 if t.dtype == torch.float16 else np.float32)


def listed():
    return [
        # the elementwise map of the benchmark; HBM only
        {"name": "map_4096", "kind": "map", "dtype": "f32", "rows": 4096, "cols": 4096},
        # the smallest call: one minibatch against ten classes, three launches of next to no work
        {"name": "head_128x10", "kind": "head", "dtype": "f32", "rows": 128, "cols": 10},
        # an image classifier's thousand classes over many rows
        {"name": "head_65536x1000", "kind": "head", "dtype": "f32", "rows": 65536, "cols": 1000},
        # a vocabulary whose rows are of odd length: nothing is aligned
        {"name": "head_2048x50257", "kind": "head", "dtype": "f32", "rows": 2048, "cols": 50257},
        # the benchmark's vocabulary: the largest case
        {"name": "head_8192x32000", "kind": "head", "dtype": "f32", "rows": 8192, "cols": 32000},
        # the same classifier kept in half_t
        {"name": "head_half_8192x32000", "kind": "head", "dtype": "f16", "rows": 8192, "cols": 32000},
        # bias gradient of a convolution in the middle of a network
        {"name": "channel_sum_256x56", "kind": "channel_sum", "dtype": "f32", "n": 64, "c": 256, "h": 56, "w": 56},
        # bias gradient of a dense layer over a long minibatch
        {"name": "column_sum_16384x4096", "kind": "column_sum", "dtype": "f32", "rows": 16384, "cols": 4096},
        # pooling forward and backward early in a network
        {"name": "pool_112_k3s2", "kind": "pool", "dtype": "f32", "n": 128, "c": 64, "h": 112, "w": 112, "k": 3, "s": 2},
        # the same on planes of odd size
        {"name": "pool_55_k3s2", "kind": "pool", "dtype": "f32", "n": 64, "c": 96, "h": 55, "w": 55, "k": 3, "s": 2},
        # a 3x3 convolution in half_t, both directions
        {"name": "patches_half_56_k3", "kind": "patches", "dtype": "f16", "n": 32, "c": 256, "h": 56, "w": 56, "k": 3, "s": 1, "p": 1},
        # the first convolution of a network, on float images
        {"name": "patches_224_k7s2", "kind": "patches", "dtype": "f32", "n": 32, "c": 3, "h": 224, "w": 224, "k": 7, "s": 2, "p": 3},
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _size(rng, low, high):
    """a size spread over the range's logarithm, half of the time rounded to a multiple of 8"""
    v = _log(rng, low, high)
    return min(max(8, v // 8 * 8), high) if v >= 16 and rng.random() < 0.5 else v


def _pooled(size, k, s):
    return (size - k) // s + 1


def _patches(size, k, s, p):
    return (size + 2 * p - k) // s + 1


def draw(rng):
    kind = rng.choice(("map", "head", "head", "head", "channel_sum", "column_sum", "pool", "pool", "patches", "patches"))
    case = {"kind": kind, "dtype": rng.choice(("f32", "f32", "f16"))}
    if kind in ("map", "column_sum"):
        most = MOST_MAP if kind == "map" else MOST_COLUMN
        rows = _size(rng, 64, 16384)
        case.update(rows=rows, cols=_size(rng, 64, max(64, min(32000, most // rows))))
    elif kind == "head":
        # minibatches of 32 rows and more; ten classes to a vocabulary of 128000 (few rows of those)
        cols = _size(rng, 10, 128000)
        most = MOST_LOGITS // cols // (4 if cols > 32768 else 1)
        case.update(rows=_size(rng, 32, max(32, min(131072, most))), cols=cols)
    elif kind == "channel_sum":
        h, w = _size(rng, 7, 112), _size(rng, 7, 112)
        c = _size(rng, 16, 2048)
        case.update(n=_size(rng, 1, max(1, min(256, MOST_CHANNEL // (c * h * w)))), c=c, h=h, w=w)
    elif kind == "pool":
        k, s = rng.choice(POOLS)
        h, w = _size(rng, 7, 224), _size(rng, 7, 224)
        c = _size(rng, 16, 512)
        case.update(n=_size(rng, 1, max(1, min(256, MOST_PIXELS // (c * h * w)))), c=c, h=h, w=w, k=k, s=s)
    else:
        k, s, p = rng.choice(CONVOLUTIONS)
        h, w = _size(rng, 7, 224), _size(rng, 7, 224)
        per_image = k * k * _patches(h, k, s, p) * _patches(w, k, s, p)
        c = _size(rng, 3, max(3, min(512, MOST_MATRIX // 2 // per_image)))
        case.update(n=_size(rng, 1, max(1, min(128, MOST_MATRIX // 2 // (per_image * c)))), c=c, h=h, w=w, k=k, s=s, p=p)
    return case


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    dtype = torch.float16 if case["dtype"] == "f16" else torch.float32

    def normal(*shape, sigma=1.0):
        t = torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32)
        return Tensor((t if sigma == 1.0 else t.mul_(sigma)).to(dtype))

    def uniform(*shape):
        return Tensor(torch.rand(shape, generator=gen, device="cuda", dtype=torch.float32).mul_(2).sub_(1).to(dtype))

    def empty(*shape):
        return Tensor(torch.empty(shape, device="cuda", dtype=dtype))

    kind = case["kind"]
    state = {"case": case}
    if kind == "map":
        shape = (case["rows"], case["cols"])
        state.update({name: uniform(*shape) for name in "abcd"}, dst=empty(*shape))
    elif kind == "head":
        rows, cols = case["rows"], case["cols"]
        # a half_t label is exact up to 2048
        top = cols if dtype == torch.float32 else min(cols, 2049)
        label = torch.randint(0, top, (rows,), generator=gen, device="cuda")
        state.update(logits=normal(rows, cols, sigma=3.0), label=Tensor(label.to(dtype)),
                     prob=empty(rows, cols), grad=empty(rows, cols), bias=empty(cols))
    elif kind == "channel_sum":
        state.update(src=normal(case["n"], case["c"], case["h"], case["w"]), dst=empty(case["c"]))
    elif kind == "column_sum":
        state.update(src=normal(case["rows"], case["cols"]), dst=empty(case["cols"]))
    elif kind == "pool":
        n, c, h, w, k, s = (case[x] for x in "nchwks")
        pooled = (n, c, _pooled(h, k, s), _pooled(w, k, s))
        state.update(src=uniform(n, c, h, w), pooled=empty(*pooled))
        if dtype == torch.float32:
            state.update(grad=normal(*pooled), dst=empty(n, c, h, w))
    else:
        n, c, h, w, k, s, p = (case[x] for x in "nchwksp")
        matrix = (c * k * k, n * _patches(h, k, s, p) * _patches(w, k, s, p))
        state.update(image=uniform(n, c, h, w), matrix=empty(*matrix), grad=normal(*matrix), dst=empty(n, c, h, w))
    return state


def run(state):
    case, kind = state["case"], state["case"]["kind"]
    half = case["dtype"] == "f16"
    if kind == "map":
        if half:
            LIB.case_map_muladd_f16(state["dst"], state["a"], state["b"], state["c"])
        else:
            LIB.case_map_fused(state["dst"], state["a"], state["b"], state["c"], state["d"])
        return state["dst"].tensor
    if kind == "head":
        prob, grad, bias = state["prob"], state["grad"], state["bias"]
        if half:
            LIB.case_softmax(prob, state["logits"])
            LIB.case_softmax_grad(grad, prob, state["label"])
            LIB.case_reduce_keep_lowest(bias, grad, scale=HALF_ONE)
        else:
            LIB.softmax(prob, state["logits"])
            LIB.softmax_grad(grad, prob, state["label"])
            LIB.reduce_keep_lowest(bias, grad)
        return prob.tensor, grad.tensor, bias.tensor
    if kind == "channel_sum":
        if half:
            LIB.case_reduce_keep_highdim(state["dst"], state["src"], scale=HALF_ONE)
        else:
            LIB.reduce_keep_highdim(state["dst"], state["src"])
        return state["dst"].tensor
    if kind == "column_sum":
        if half:
            LIB.case_reduce_keep_lowest(state["dst"], state["src"], scale=HALF_ONE)
        else:
            LIB.reduce_keep_lowest(state["dst"], state["src"])
        return state["dst"].tensor
    if kind == "pool":
        k, s = case["k"], case["s"]
        if half:
            LIB.case_pool(state["pooled"], state["src"], k, k, s, s)
            return state["pooled"].tensor
        LIB.pool(state["pooled"], state["src"], k, k, s, s)
        LIB.unpool(state["dst"], state["src"], state["pooled"], state["grad"], k, k, s, s)
        return state["pooled"].tensor, state["dst"].tensor
    k, s, p = case["k"], case["s"], case["p"]
    LIB.im2col(state["matrix"], state["image"], k, k, s, s, pad_y=p, pad_x=p)
    LIB.col2im(state["dst"], state["grad"], k, k, s, s, pad_y=p, pad_x=p)
    return state["matrix"].tensor, state["dst"].tensor


def work(case):
    """Each call's inputs read once and its outputs written once; the calls of a step are separate ones, so
    what one writes for the next is read again. Flops are the adds, products, comparisons and exponentials of
    the definitions."""
    e = 2 if case["dtype"] == "f16" else 4
    kind = case["kind"]
    if kind == "map":
        n = case["rows"] * case["cols"]
        return {"bytes": (4 if e == 2 else 5) * e * n, "flops": (2 if e == 2 else 7) * n}
    if kind == "head":
        rows, cols = case["rows"], case["cols"]
        return {"bytes": e * (5 * rows * cols + rows + cols), "flops": 6 * rows * cols}
    if kind == "channel_sum":
        n = case["n"] * case["c"] * case["h"] * case["w"]
        return {"bytes": e * (n + case["c"]), "flops": n}
    if kind == "column_sum":
        n = case["rows"] * case["cols"]
        return {"bytes": e * (n + case["cols"]), "flops": n}
    if kind == "pool":
        n, c, h, w, k, s = (case[x] for x in "nchwks")
        src, pooled = n * c * h * w, n * c * _pooled(h, k, s) * _pooled(w, k, s)
        if e == 2:
            return {"bytes": e * (src + pooled), "flops": pooled * k * k}
        return {"bytes": e * (3 * src + 3 * pooled), "flops": 4 * pooled * k * k}
    n, c, h, w, k, s, p = (case[x] for x in "nchwksp")
    image = n * c * h * w
    matrix = n * c * k * k * _patches(h, k, s, p) * _patches(w, k, s, p)
    return {"bytes": e * 2 * (image + matrix), "flops": matrix}


def tolerance(case):
    """Every result is the CPU path's bit for bit - its sums run in index order - except what goes through an
    exponential. Against correctly rounded exponentials summed in the same order, float results differ by up to
    1e-7 (the bias gradient of 128 x 10; the probabilities by 6e-8); half_t results did not differ, and where
    another exponential turns one binary16 rounding over, a row's sum may move by one unit, 5e-4 at most."""
    if case["kind"] != "head":
        return "exact"
    return {"rel": 5e-4} if case["dtype"] == "f16" else {"rel": 5e-7}
