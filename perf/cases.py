"""What a program of this framework spends its time on: one case per kind of call, over the
sizes it meets, each through ``ninetoothed_amd.make`` / ``jit`` and the Handle they return.

The arrangements and applications are the ones NineToothed programs write for these
operations.  Sizes are those of the repository's benchmark and tests (512^3 fp32 matmul,
4096^3 addmm, the 256-channel 3 x 3 convolution, attention at B=4, H=32, S=4096, D=128, softmax
8192 x 8192, max_pool2d on [32, 128, 112, 112]) or generic ones for the same calls: linear
layers with 4096 and 11008 features, a decode step against 4,000 cached keys, the late layers
of a convolutional network, logits of 50,257 classes, a 4096-wide norm.
"""

import functools
import math

import torch

import ninetoothed_amd as ninetoothed
import ninetoothed_amd.language as ntl
from ninetoothed_amd import Symbol, Tensor

DEVICE = "cuda"
DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
BYTES = {"f32": 4, "f16": 2, "bf16": 2}


# ---------------------------------------------------------------------------- the programs
BLOCK_SIZE_M = Symbol("BLOCK_SIZE_M", meta=True)
BLOCK_SIZE_N = Symbol("BLOCK_SIZE_N", meta=True)
BLOCK_SIZE_K = Symbol("BLOCK_SIZE_K", meta=True)


def matmul_arrangement(lhs, rhs, output, BLOCK_SIZE_M=BLOCK_SIZE_M, BLOCK_SIZE_N=BLOCK_SIZE_N,
                       BLOCK_SIZE_K=BLOCK_SIZE_K):
    output_tiled = output.tile((BLOCK_SIZE_M, BLOCK_SIZE_N))
    lhs_tiled = lhs.tile((BLOCK_SIZE_M, BLOCK_SIZE_K)).tile((1, -1)).expand((-1, output_tiled.shape[1]))
    lhs_tiled.dtype = lhs_tiled.dtype.squeeze(0)
    rhs_tiled = rhs.tile((BLOCK_SIZE_K, BLOCK_SIZE_N)).tile((-1, 1)).expand((output_tiled.shape[0], -1))
    rhs_tiled.dtype = rhs_tiled.dtype.squeeze(1)
    return lhs_tiled, rhs_tiled, output_tiled


def matmul_application(lhs, rhs, output):
    accumulator = ntl.zeros(output.shape, dtype=ntl.float32)
    for k in range(lhs.shape[0]):
        accumulator += ntl.dot(lhs[k], rhs[k])
    output = accumulator  # noqa: F841


def addmm_arrangement(input, mat1, mat2, beta, alpha, output):
    _, _, input_arranged = matmul_arrangement(mat1, mat2, input)
    mat1_arranged, mat2_arranged, output_arranged = matmul_arrangement(mat1, mat2, output)
    return input_arranged, mat1_arranged, mat2_arranged, beta, alpha, output_arranged


def addmm_application(input, mat1, mat2, beta, alpha, output):
    matmul_output = ntl.zeros(output.shape, dtype=ntl.float32)
    matmul_application(mat1, mat2, matmul_output)
    output = beta * input + alpha * matmul_output  # noqa: F841


def conv2d_arrangement(input, filter, output):
    padding_h = Symbol("padding_h", constexpr=True)
    padding_w = Symbol("padding_w", constexpr=True)
    input_padded = input.pad(((0, 0), (0, 0), (padding_h, padding_h), (padding_w, padding_w)))
    input_tiled = input_padded.tile((1, *filter.shape[1:]), strides=(-1, -1, 1, 1))
    input_squeezed = input_tiled.squeeze(1)
    input_squeezed.dtype = input_squeezed.dtype.squeeze(0)
    input_flattened = input_squeezed.ravel().flatten(end_dim=3).flatten(start_dim=1)
    filter_permuted = filter.flatten(start_dim=1).permute((1, 0))
    output_flattened = output.permute((0, 2, 3, 1)).flatten(end_dim=3)
    return matmul_arrangement(input_flattened, filter_permuted, output_flattened)


ATT_BLOCK_SIZE_M = ninetoothed.block_size(lower_bound=64, upper_bound=128)
ATT_BLOCK_SIZE_N = ninetoothed.block_size(lower_bound=32, upper_bound=64)


def attention_arrangement(q, k, v, is_causal, o, BLOCK_SIZE_M=ATT_BLOCK_SIZE_M, BLOCK_SIZE_N=ATT_BLOCK_SIZE_N):
    def arrange_q_or_o(input):
        arranged = input.tile((1, 1, BLOCK_SIZE_M, -1))
        arranged.dtype = arranged.dtype.squeeze((0, 1))
        return arranged

    def arrange_k_or_v(input):
        arranged = input.tile((1, 1, BLOCK_SIZE_N, -1)).tile((1, 1, -1, -1)).expand((-1, -1, q_arranged.shape[-2], -1))
        arranged.dtype = arranged.dtype.squeeze((0, 1, 3))
        arranged.dtype.dtype = arranged.dtype.dtype.squeeze((0, 1))
        return arranged

    q_arranged = arrange_q_or_o(q)
    return q_arranged, arrange_k_or_v(k), arrange_k_or_v(v), is_causal, arrange_q_or_o(o)


def attention_application(q, k, v, is_causal, o):
    q_loaded = (q * 1.44269504089).to(q.dtype)
    acc = ntl.zeros((q.shape[-2], q.shape[-1]), dtype=ntl.float32)
    l_i = ntl.full((q.shape[-2],), 1, dtype=ntl.float32)
    m_i = ntl.full((q.shape[-2],), float("-inf"), dtype=ntl.float32)
    for i in range(k.shape[0]):
        qk = ntl.dot(q_loaded, ntl.trans(k[i]))
        qk = ntl.where(k[i].offsets(-2) < k.source.shape[-2], qk, float("-inf"))
        if is_causal:
            mask = q.offsets(-2)[:, None] >= k[i].offsets(-2)[None, :]
            qk = ntl.where(mask, qk, float("-inf"))
        m_ij = ntl.maximum(m_i, ntl.max(qk, 1))
        p = ntl.exp2(qk - m_ij[:, None])
        l_ij = ntl.sum(p, 1)
        alpha = ntl.exp2(m_i - m_ij)
        acc = acc * alpha[:, None] + ntl.dot(p.to(v[i].dtype), v[i])
        m_i = m_ij
        l_i = l_i * alpha + l_ij
    acc /= l_i[:, None]
    o = acc  # noqa: F841


def max_pool2d_arrangement(input, output):
    BLOCK_SIZE = Symbol("BLOCK_SIZE", meta=True)
    WINDOW_HEIGHT = Symbol("WINDOW_HEIGHT", constexpr=True, upper_bound=16)
    WINDOW_WIDTH = Symbol("WINDOW_WIDTH", constexpr=True, upper_bound=16)
    input_arranged = input.tile((1, 1, WINDOW_HEIGHT, WINDOW_WIDTH), floor_mode=True).ravel()
    input_arranged = input_arranged.flatten(end_dim=4).flatten(start_dim=1).tile((BLOCK_SIZE, -1))
    output_arranged = output.tile((1, 1, 1, 1)).ravel().flatten(end_dim=4).flatten(start_dim=1)
    output_arranged = output_arranged.tile((BLOCK_SIZE, -1))
    output_arranged.dtype = output_arranged.dtype.squeeze(1)
    return input_arranged, output_arranged


def max_pool2d_application(input, output):
    output = ntl.max(input, axis=1)  # noqa: F841


WIDTH = Symbol("WIDTH", constexpr=True)


def rms_norm_arrangement(x, weight, eps, output, WIDTH=WIDTH):
    return x.tile((1, WIDTH)), weight.tile((1, WIDTH)), eps, output.tile((1, WIDTH))


def rms_norm_application(x, weight, eps, output):
    x32 = ntl.cast(x, ntl.float32)
    mean_square = ntl.sum(x32 * x32, axis=1) / x.shape[1]
    output = x32 * ntl.rsqrt(mean_square[:, None] + eps) * ntl.cast(weight, ntl.float32)  # noqa: F841


@functools.lru_cache(maxsize=None)
def _handle(kind):
    """The Handle a program makes once, at start-up, and calls with tensors of any size."""
    if kind == "matmul":
        return ninetoothed.make(matmul_arrangement, matmul_application, (Tensor(2), Tensor(2), Tensor(2)))
    if kind == "addmm":
        return ninetoothed.make(addmm_arrangement, addmm_application,
                                (Tensor(2), Tensor(2), Tensor(2), Tensor(0), Tensor(0), Tensor(2)))
    if kind == "conv2d":
        return ninetoothed.make(conv2d_arrangement, matmul_application,
                                (Tensor(4), Tensor(4, shape_options={"constexpr": True}), Tensor(4)))
    if kind == "attention":
        q, k, v, o = (
            Tensor(4, shape_options=(None, None, {"constexpr": True}, {"constexpr": True, "upper_bound": 128}))
            for _ in range(4)
        )
        return ninetoothed.make(attention_arrangement, attention_application, (q, k, v, Tensor(0, constexpr=True), o))
    if kind == "softmax":
        BLOCK_SIZE = Symbol("BLOCK_SIZE", constexpr=True)

        @ninetoothed.jit
        def softmax_kernel(
            input_row: Tensor(2, other=float("-inf")).tile((1, BLOCK_SIZE)),
            output_row: Tensor(2).tile((1, BLOCK_SIZE)),
        ):
            row_minus_max = input_row - ntl.max(input_row)
            numerator = ntl.exp(row_minus_max)
            denominator = ntl.sum(numerator)
            output_row = numerator / denominator  # noqa: F841

        return softmax_kernel
    if kind == "max_pool2d":
        return ninetoothed.make(max_pool2d_arrangement, max_pool2d_application,
                                (Tensor(4, other=float("-inf")), Tensor(4)))
    if kind == "rms_norm":
        return ninetoothed.make(rms_norm_arrangement, rms_norm_application,
                                (Tensor(2), Tensor(2), Tensor(0, dtype="float32"), Tensor(2)))
    raise ValueError(kind)


# ------------------------------------------------------------------------------- the cases
def listed():
    return [
        # the README's matmul: one small product, where the launch and its latency count
        dict(name="matmul_f32_512", kind="matmul", dtype="f32", m=512, n=512, k=512),
        # the headline product of the benchmark
        dict(name="addmm_f16_4096", kind="addmm", dtype="f16", m=4096, n=4096, k=4096),
        # a linear layer of a decode step: a few tokens against the whole weight
        dict(name="linear_bf16_decode", kind="linear", dtype="bf16", m=16, n=11008, k=4096),
        # the same layer type on one short prompt, whose length is what the user typed
        dict(name="linear_f16_prompt", kind="linear", dtype="f16", m=200, n=4096, k=4096),
        # the benchmark's convolution: a wide 3 x 3 layer on a large image
        dict(name="conv2d_f16_56", kind="conv2d", dtype="f16", n=16, c=256, h=56, w=56, k=256, r=3),
        # the last stage of a convolutional network: many channels, a 7 x 7 image
        dict(name="conv2d_bf16_7", kind="conv2d", dtype="bf16", n=8, c=512, h=7, w=7, k=512, r=3),
        # attention over a long prompt (the benchmark's causal configuration)
        dict(name="attention_f16_prompt", kind="attention", dtype="f16", b=4, heads=32, sq=4096, sk=4096, d=128,
             causal=True),
        # attention of a decode step: one new token a sequence against its cached keys
        dict(name="attention_bf16_decode", kind="attention", dtype="bf16", b=8, heads=32, sq=1, sk=4000, d=128,
             causal=False),
        # the benchmark's softmax: many rows of a power of two
        dict(name="softmax_f16_8192", kind="softmax", dtype="f16", rows=8192, cols=8192),
        # probabilities from the logits of one decode batch: few rows, long and odd
        dict(name="softmax_f32_logits", kind="softmax", dtype="f32", rows=32, cols=50257),
        # the benchmark's pooling layer
        dict(name="max_pool2d_f16", kind="max_pool2d", dtype="f16", n=32, c=128, h=112, w=112, window=2),
        # a norm between two layers: a program of the user's own, outside the named families
        dict(name="rms_norm_bf16", kind="rms_norm", dtype="bf16", rows=2048, cols=4096),
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, spread over their logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi):
    """A size between lo and hi: a multiple of 64, of 8, or any number."""
    step = rng.choice((64, 8, 1))
    return min(hi, max(lo, _log(rng, lo, hi) // step * step))


def _draw(rng):
    half = rng.choice(("f16", "bf16"))
    kind = rng.choice(("matmul", "addmm", "linear", "linear", "conv2d", "conv2d", "prompt", "decode", "softmax",
                       "softmax", "max_pool2d", "rms_norm"))
    if kind == "matmul":
        return dict(kind=kind, dtype="f32", m=_size(rng, 64, 2048), n=_size(rng, 64, 2048), k=_size(rng, 64, 2048))
    if kind == "addmm":
        return dict(kind=kind, dtype=half, m=_size(rng, 256, 4096), n=_size(rng, 256, 4096), k=_size(rng, 256, 4096))
    if kind == "linear":
        return dict(kind=kind, dtype=half, m=_log(rng, 1, 1024), n=_size(rng, 1024, 11008), k=_size(rng, 1024, 11008))
    if kind == "conv2d":
        side = rng.choice((7, 14, 28, 56, _log(rng, 7, 56)))
        return dict(kind=kind, dtype=half, n=_log(rng, 1, 32), c=8 * _log(rng, 4, 64), h=side, w=side,
                    k=8 * _log(rng, 4, 64), r=rng.choice((1, 3, 3)))
    if kind == "prompt":
        s = _size(rng, 128, 4096)
        return dict(kind="attention", dtype=half, b=_log(rng, 1, 4), heads=rng.choice((8, 12, 16, 32)), sq=s, sk=s,
                    d=rng.choice((64, 128)), causal=rng.choice((False, True)))
    if kind == "decode":
        return dict(kind="attention", dtype=half, b=_log(rng, 1, 16), heads=rng.choice((8, 12, 16, 32)),
                    sq=rng.choice((1, 1, 4)), sk=_size(rng, 256, 8192), d=rng.choice((64, 128)), causal=False)
    if kind == "softmax":
        return dict(kind=kind, dtype=rng.choice(("f32", "f16", "bf16")), rows=_log(rng, 8, 8192),
                    cols=_size(rng, 256, 131072))
    if kind == "max_pool2d":
        side = _size(rng, 28, 112)
        return dict(kind=kind, dtype=rng.choice(("f32", "f16")), n=_log(rng, 1, 32), c=8 * _log(rng, 4, 32), h=side,
                    w=side, window=rng.choice((2, 3)))
    return dict(kind=kind, dtype=half, rows=_log(rng, 1, 8192), cols=_size(rng, 512, 8192))


def _cost(case):
    """Seconds the case's work takes at the card's nominal rates."""
    need = work(case)
    return max(need["bytes"] / 8e12, need["flops"] / (157e12 if case["dtype"] == "f32" else 2.5e15))


def draw(rng):
    limits = {}
    for case in listed():
        limits[case["kind"]] = max(limits.get(case["kind"], 0.0), _cost(case))
    while True:
        case = _draw(rng)
        # a case costs no more than the largest listed one of its kind; the small fp32
        # matmul stands for fp32 products up to the size of the ordinary 16-bit one
        limit = limits["addmm"] if case["kind"] in ("matmul", "linear") else limits[case["kind"]]
        if _cost(case) <= limit:
            return case


def work(case):
    kind, size = case["kind"], BYTES[case["dtype"]]
    if kind in ("matmul", "linear", "addmm"):
        m, n, k = case["m"], case["n"], case["k"]
        elements = m * k + k * n + m * n * (2 if kind == "addmm" else 1)
        return {"bytes": elements * size, "flops": 2 * m * n * k}
    if kind == "conv2d":
        n, c, h, w, k, r = (case[x] for x in ("n", "c", "h", "w", "k", "r"))
        return {"bytes": (n * c * h * w + k * c * r * r + n * k * h * w) * size, "flops": 2 * n * h * w * k * c * r * r}
    if kind == "attention":
        bh, sq, sk, d = case["b"] * case["heads"], case["sq"], case["sk"], case["d"]
        pairs = sq * (sq + 1) // 2 if case["causal"] else sq * sk
        return {"bytes": bh * (2 * sq + 2 * sk) * d * size, "flops": 4 * bh * pairs * d}
    if kind == "max_pool2d":
        n, c, h, w, win = (case[x] for x in ("n", "c", "h", "w", "window"))
        outputs = n * c * (h // win) * (w // win)
        return {"bytes": (n * c * h * w + outputs) * size, "flops": outputs * win * win}
    elements = case["rows"] * case["cols"]
    if kind == "softmax":
        return {"bytes": 2 * elements * size, "flops": 4 * elements}
    return {"bytes": (2 * elements + case["cols"]) * size, "flops": 4 * elements}  # rms_norm


# The largest relative errors another order of the fp32 sums and the rounding to 16 bits give:
# about four times what the path shows against 64 bits (products, convolutions and norms
# 2.1e-4 in fp16 and 1.7e-3 in bf16, the rounding of the result; attention, which also rounds
# its weights, 4.7e-4 and 3.9e-3; fp32 sums up to 2.5e-7, more where summed in sequence).
def tolerance(case):
    if case["kind"] == "max_pool2d":
        return "exact"
    if case["dtype"] == "f32":
        return {"rel": 2e-6}
    if case["kind"] == "attention":
        return {"rel": 1.6e-2 if case["dtype"] == "bf16" else 2e-3}
    return {"rel": 8e-3 if case["dtype"] == "bf16" else 1e-3}


# -------------------------------------------------------------------------------- one pass
def _inputs(case, seed):
    g = torch.Generator(device=DEVICE).manual_seed(seed)
    dtype = DTYPES[case["dtype"]]

    def normal(*shape, scale=1.0):
        return (torch.randn(shape, generator=g, device=DEVICE) * scale).to(dtype)

    kind = case["kind"]
    if kind == "matmul":
        return normal(case["m"], case["k"]), normal(case["k"], case["n"])
    if kind == "addmm":
        scale = case["k"] ** -0.5
        return (normal(case["m"], case["n"]), normal(case["m"], case["k"]), normal(case["k"], case["n"], scale=scale))
    if kind == "linear":  # activations and a weight of [out features, in features]
        return normal(case["m"], case["k"]), normal(case["n"], case["k"], scale=case["k"] ** -0.5)
    if kind == "conv2d":
        c, k, r = case["c"], case["k"], case["r"]
        return normal(case["n"], c, case["h"], case["w"]), normal(k, c, r, r, scale=(c * r * r) ** -0.5)
    if kind == "attention":
        b, heads, d = case["b"], case["heads"], case["d"]
        # the usual 1 / sqrt(d) is in q
        return (normal(b, heads, case["sq"], d, scale=d**-0.5), normal(b, heads, case["sk"], d),
                normal(b, heads, case["sk"], d))
    if kind == "softmax":
        return (normal(case["rows"], case["cols"], scale=2.0),)
    if kind == "max_pool2d":
        return (normal(case["n"], case["c"], case["h"], case["w"]),)
    return normal(case["rows"], case["cols"]), 1 + normal(case["cols"], scale=0.1)  # rms_norm


def prepare(case, seed):
    inputs = _inputs(case, seed)
    kind, dtype = case["kind"], DTYPES[case["dtype"]]
    if kind in ("matmul", "addmm", "linear"):
        shape = (case["m"], case["n"])
    elif kind == "conv2d":
        shape = (case["n"], case["k"], case["h"], case["w"])
    elif kind == "max_pool2d":
        shape = (case["n"], case["c"], case["h"] // case["window"], case["w"] // case["window"])
    else:
        shape = inputs[0].shape
    return {"kind": kind, "case": case, "kernel": _handle("matmul" if kind == "linear" else kind), "inputs": inputs,
            "out": torch.empty(shape, dtype=dtype, device=DEVICE)}


def run(state):
    kernel, inputs, out, case = state["kernel"], state["inputs"], state["out"], state["case"]
    kind = state["kind"]
    if kind == "matmul":
        kernel(inputs[0], inputs[1], out)
    elif kind == "addmm":
        kernel(inputs[0], inputs[1], inputs[2], 0.5, 1.0, out)
    elif kind == "linear":
        kernel(inputs[0], inputs[1].t(), out)
    elif kind == "conv2d":
        kernel(inputs[0], inputs[1], out, padding_h=case["r"] // 2, padding_w=case["r"] // 2)
    elif kind == "attention":
        kernel(inputs[0], inputs[1], inputs[2], case["causal"], out)
    elif kind == "softmax":
        kernel(inputs[0], out, BLOCK_SIZE=case["cols"])
    elif kind == "max_pool2d":
        kernel(inputs[0], out, WINDOW_HEIGHT=case["window"], WINDOW_WIDTH=case["window"])
    else:
        kernel(inputs[0], inputs[1].expand(inputs[0].shape), 1e-6, out, WIDTH=case["cols"])
    return out


def exact(case, seed):
    x = [t.double() for t in _inputs(case, seed)]
    kind = case["kind"]
    if kind == "matmul":
        return x[0] @ x[1]
    if kind == "addmm":
        return 0.5 * x[0] + x[1] @ x[2]
    if kind == "linear":
        return x[0] @ x[1].t().contiguous()
    if kind == "conv2d":
        n, k, h, w = case["n"], case["k"], case["h"], case["w"]
        filters = x[1].reshape(k, -1)
        out = torch.empty(n, k, h, w, dtype=torch.float64, device=DEVICE)
        for i in range(n):
            columns = torch.nn.functional.unfold(x[0][i : i + 1], case["r"], padding=case["r"] // 2)[0]
            out[i] = (filters @ columns).reshape(k, h, w)
        return out
    if kind == "attention":
        q, keys, values = x
        out = torch.empty_like(q)
        mask = None
        if case["causal"]:
            mask = torch.ones(case["sq"], case["sk"], dtype=torch.bool, device=DEVICE).tril().logical_not()
        for b in range(case["b"]):
            for h in range(case["heads"]):
                scores = q[b, h] @ keys[b, h].t().contiguous()
                if mask is not None:
                    scores.masked_fill_(mask, -math.inf)
                out[b, h] = torch.softmax(scores, -1) @ values[b, h]
        return out
    if kind == "softmax":
        return torch.softmax(x[0], -1)
    if kind == "max_pool2d":
        return torch.nn.functional.max_pool2d(x[0], case["window"])
    return x[0] * torch.rsqrt((x[0] * x[0]).mean(-1, keepdim=True) + 1e-6) * x[1]
