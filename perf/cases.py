"""The products that programs ask this library for, as cases to time: what goes in, one pass, and what it has to cost.

Every case goes through the package's public entry points.  `listed()` holds one case per kind of use, `draw()` gives
further ones of the same kinds with other sizes, types and options.  Sizes of the listed cases are those of the tests,
the benchmark and the reference scripts' own runs.
"""
import math
import os
import sys

import torch

_PACKAGE = os.path.join(os.getcwd(), "stream-k.tvm_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)
import streamk  # noqa: E402

# Cases are dicts of: kind, dtype, M (rows of A), N, K, and by kind bias / activation / alpha / layers.
#   "linear": StreamKLinear, the layer of a model; dtype is its weight format; bias and activation in the epilogue
#   "mlp":    one decode step through `layers` pairs of layers (K -> N with the activation, N -> K), captured in a HIP
#             graph the way a serving loop does, M rows in flight
#   "gemm":   the reference-named functions on plain tensors: streamk_fp16 / _bf16 / _fp32 / _fp8 / _int8 / _q4


def listed():
    return [
        # one token of one sequence through a small quantised layer, called eagerly: launch and host latency
        dict(name="linear_q4_1row", kind="linear", dtype="q4", M=1, N=4096, K=4096, bias=False, activation="none"),
        # a decode step of four sequences through four MLP blocks with asymmetric 4-bit weights, one captured graph
        dict(name="mlp_graph_q4zp_4rows", kind="mlp", dtype="q4_zp", M=4, N=11008, K=4096, layers=4, activation="silu"),
        # the shape of the reference's fp16 and fp32 scripts: a batch of 16 tokens against a wide weight matrix
        dict(name="f16_16x16384x8192", kind="gemm", dtype="float16", layout="nt", M=16, N=16384, K=8192),
        dict(name="f32_16x16384x8192", kind="gemm", dtype="float32", layout="nn", M=16, N=16384, K=8192),
        # the shape of the reference's Q4 script
        dict(name="q4_16x16384x16384", kind="gemm", dtype="q4", layout="nt", M=16, N=16384, K=16384),
        # 64 sequences decoding against fp8 weights, per-tensor scales, bias and activation fused
        dict(name="f8_64x28672x8192", kind="gemm", dtype="float8_e4m3", layout="nt", M=64, N=28672, K=8192, alpha=0.01,
             bias=True, activation="silu"),
        # a short prompt (ragged number of tokens) through a bfloat16 layer
        dict(name="linear_bf16_100rows", kind="linear", dtype="bfloat16", M=100, N=11008, K=4096, bias=True,
             activation="gelu_tanh"),
        # integer inference, a ragged batch
        dict(name="i8_300x11008x4096", kind="gemm", dtype="int8", layout="nt", M=300, N=11008, K=4096),
        # a prompt of 512 tokens through a 4-bit layer
        dict(name="linear_q4_512rows", kind="linear", dtype="q4", M=512, N=8192, K=8192, bias=True, activation="none"),
        # few output tiles and a long K: what the Stream-K split is for
        dict(name="f16_1024x1024x8192", kind="gemm", dtype="float16", layout="nt", M=1024, N=1024, K=8192),
        # large, irregular, weights as [K, N]
        dict(name="f16nn_3000x5120x12288", kind="gemm", dtype="float16", layout="nn", M=3000, N=5120, K=12288),
        # the dense headline
        dict(name="f16_8192x8192x8192", kind="gemm", dtype="float16", layout="nt", M=8192, N=8192, K=8192),
    ]


def _log_int(rng, lo, hi, step=1):
    """An integer from lo to hi, spread evenly over its logarithm, a multiple of `step`."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(step, min(hi // step * step, int(round(v / step)) * step))


# largest product of each type a drawn case asks for, in multiply-adds: the time of the largest listed case or less
_MOST = {"float16": 8192 ** 3 // 2, "bfloat16": 8192 ** 3 // 2, "float8_e4m3": 8192 ** 3, "float8_e5m2": 8192 ** 3,
         "int8": 8192 ** 3, "q4": 8192 ** 3 // 3, "q4_zp": 8192 ** 3 // 3, "float32": 8192 ** 3 // 16}
_K_STEP = {"float16": 8, "bfloat16": 8, "float8_e4m3": 16, "float8_e5m2": 16, "int8": 16, "q4": 128, "q4_zp": 128,
           "float32": 4}


def draw(rng):
    kind = rng.choice(["linear", "linear", "gemm", "gemm", "gemm", "mlp"])
    if kind == "mlp":
        dtype = rng.choice(["float16", "bfloat16", "q4", "q4_zp"])
        step = 64 if dtype in ("float16", "bfloat16") else 128
        return dict(kind="mlp", dtype=dtype, M=_log_int(rng, 1, 64), N=_log_int(rng, 2048, 14336, step),
                    K=_log_int(rng, 1024, 8192, step), layers=rng.randint(1, 4),
                    activation=rng.choice(["relu", "gelu_tanh", "silu"]))
    if kind == "linear":
        dtype = rng.choice(["float16", "bfloat16", "q4", "q4_zp"])
    else:
        dtype = rng.choice(["float16", "float16", "bfloat16", "float32", "float8_e4m3", "float8_e5m2", "int8", "q4"])
    step = _K_STEP[dtype]
    # sizes of layers: half of them multiples of 256, the others anything the type takes
    if rng.random() < 0.5:
        N, K = _log_int(rng, 1024, 28672, 256), _log_int(rng, 1024, 16384, 256)
    else:
        N, K = _log_int(rng, 513, 28672, 8), _log_int(rng, 512, 16384, step)
        if kind == "linear" and rng.random() < 0.3:
            N += rng.randint(1, 7)
    most = max(1, min(8192, _MOST[dtype] // (N * K)))
    M = _log_int(rng, 1, most) if most > 1 else 1
    c = dict(kind=kind, dtype=dtype, M=M, N=N, K=K)
    if kind == "linear":
        c.update(bias=rng.random() < 0.5, activation=rng.choice(["none", "none", "relu", "gelu_tanh", "silu"]))
        return c
    c["layout"] = rng.choice(["nt", "nn"]) if dtype in ("float16", "bfloat16", "float32") else "nt"
    if dtype.startswith("float8"):
        c.update(alpha=0.01, bias=rng.random() < 0.5, activation=rng.choice(["none", "silu"]))
    return c


_TORCH = {"float16": torch.float16, "bfloat16": torch.bfloat16, "float32": torch.float32}


def _normal(gen, shape, std, dtype):
    return torch.randn(*shape, generator=gen, device="cuda", dtype=torch.float32).mul_(std).to(dtype)


def _q4_weights(gen, N, K, zero_points):
    """Nibbles 1..15 bell-shaped around 8 as a quantiser leaves them, scales and (asymmetric) zero points around it."""
    half = lambda: torch.randint(0, 256, (N, K // 2), generator=gen, device="cuda", dtype=torch.uint8) & 0x77  # noqa: E731
    q = half() + half() + 0x11   # each nibble 0..7 + 0..7 + 1
    scales = torch.empty(N, K // 128, device="cuda").uniform_(0.005, 0.02, generator=gen).to(torch.float16)
    zeros = torch.randint(6, 11, (N, K // 128), generator=gen, device="cuda").to(torch.float16) if zero_points else None
    return q, scales, zeros


def _layer(gen, K, N, fmt, bias, activation):
    layer = streamk.StreamKLinear(K, N, bias, weight_format=fmt, device="cuda",
                                  activation=None if activation == "none" else activation)
    if fmt in ("q4", "q4_zp"):
        q, scales, zeros = _q4_weights(gen, N, K, fmt == "q4_zp")
        layer.qweight.copy_(q)
        layer.scales.copy_(scales.mul_(24 / math.sqrt(K)))   # keeps the outputs near one, as trained weights do
        if zeros is not None:
            layer.zeros.copy_(zeros)
    else:
        layer.weight.copy_(_normal(gen, (N, K), 1 / math.sqrt(K), layer.dtype))
    if bias:
        layer.bias.copy_(_normal(gen, (N,), 0.5, layer.dtype))
    return layer


class _DecodeStep:
    """What a serving loop keeps: the layers, the input's buffer and the captured graph that reads both."""

    def __init__(self, gen, case):
        M, N, K, dtype = case["M"], case["N"], case["K"], case["dtype"]
        self.blocks = [(_layer(gen, K, N, dtype, False, case["activation"]), _layer(gen, N, K, dtype, False, "none"))
                       for _ in range(case["layers"])]
        self.x = _normal(gen, (M, K), 1.0, self.blocks[0][0].dtype)
        # warm up on the stream that is captured, then capture
        stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            self.step()
        torch.cuda.current_stream().wait_stream(stream)
        torch.cuda.synchronize()
        self.graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(self.graph, stream=stream):
            self.out = self.step()

    def step(self):
        h = self.x
        for up, down in self.blocks:
            h = down(up(h))
        return h

    def __call__(self):
        self.graph.replay()
        return self.out


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    M, N, K, dtype = case["M"], case["N"], case["K"], case["dtype"]
    if case["kind"] == "linear":
        layer = _layer(gen, K, N, dtype, case["bias"], case["activation"])
        x = _normal(gen, (M, K), 1.0, layer.dtype)
        return lambda: layer(x)
    if case["kind"] == "mlp":
        return _DecodeStep(gen, case)
    if dtype == "q4":
        A = _normal(gen, (M, K), 1.0, torch.float16)
        q, scales, _ = _q4_weights(gen, N, K, False)
        return lambda: streamk.streamk_q4(A, q, scales)
    if dtype == "int8":
        A = torch.randint(-127, 128, (M, K), generator=gen, device="cuda", dtype=torch.int8)
        B = torch.randint(-127, 128, (N, K), generator=gen, device="cuda", dtype=torch.int8)
        return lambda: streamk.streamk_int8(A, B)
    if dtype.startswith("float8"):
        kind = torch.float8_e4m3fn if dtype == "float8_e4m3" else torch.float8_e5m2
        A, B = _normal(gen, (M, K), 1.0, torch.float32).to(kind), _normal(gen, (N, K), 1.0, torch.float32).to(kind)
        bias = _normal(gen, (N,), 0.5, torch.float16) if case["bias"] else None
        activation = None if case["activation"] == "none" else case["activation"]
        return lambda: streamk.streamk_fp8(A, B, alpha=case["alpha"], bias=bias, activation=activation)
    A = _normal(gen, (M, K), 1.0, _TORCH[dtype])
    B = _normal(gen, (N, K) if case["layout"] == "nt" else (K, N), 1 / math.sqrt(K), _TORCH[dtype])
    f = {"float16": streamk.streamk_fp16, "bfloat16": streamk.streamk_bf16, "float32": streamk.streamk_fp32}[dtype]
    return lambda: f(A, B, layout=case["layout"])


def run(state):
    return state()


_IN = {"float16": 2, "bfloat16": 2, "float32": 4, "float8_e4m3": 1, "float8_e5m2": 1, "int8": 1}
_OUT = {"float16": 2, "bfloat16": 2, "float32": 4, "float8_e4m3": 2, "float8_e5m2": 2, "int8": 4, "q4": 2, "q4_zp": 2}


def work(case):
    """The operands once, C once; 2 M N K operations."""
    M, N, K, dtype = case["M"], case["N"], case["K"], case["dtype"]
    if dtype in ("q4", "q4_zp"):
        weights, a = N * K // 2 + (2 if dtype == "q4" else 4) * N * (K // 128), 2 * M * K
    else:
        weights, a = _IN[dtype] * N * K, _IN[dtype] * M * K
    n = 2 * case["layers"] if case["kind"] == "mlp" else 1
    # between the layers of an MLP the activations may stay on the chip: x and the last output are what must move
    bytes_ = n * weights + a + _OUT[dtype] * M * (K if case["kind"] == "mlp" else N)
    if case.get("bias"):
        bytes_ += _OUT[dtype] * N
    return {"bytes": bytes_, "flops": n * 2.0 * M * N * K}


def tolerance(case):
    """About four times what the present results show against the same product in 64 bits (in parentheses)."""
    dtype = case["dtype"]
    if dtype == "int8":
        return "exact"
    if dtype == "float32":
        return {"rel": 4e-6, "max": 2.5e-5}                     # (8e-7, 6e-6)
    # one 16-bit result, and where a kernel rounds its weights or partial sums to 16 bits, those; they add up over the
    # layers of an MLP as independent errors do
    rel, most = (6.5e-3, 2e-2) if dtype == "bfloat16" else (1.1e-3, 4.4e-3)   # (1.7e-3, 3.9e-3), (2.7e-4, 1.1e-3)
    grow = math.sqrt(2 * case["layers"]) if case["kind"] == "mlp" else 1.0    # (four blocks: 4.9e-3, 1.9e-2; 6.4e-4, 2.5e-3)
    return {"rel": rel * grow, "max": most * grow}
