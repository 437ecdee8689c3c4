"""Timed cases of the HIP backend: what programs that use it run, over the sizes they run it at.

Two public entry points carry the work, both on device memory and on the caller's stream: a compiled .mcg graph
(`Compiled`, inputs and outputs bound once, `enqueue` per pass) and the GEMM operator (`launch_matmul` on fp32
operands, `launch_matmul_lowp` on 16-bit ones, with the split count and workspace the library asks for). Sizes are
those of the shipped graphs, the benchmark and the tests, and ragged ones between them."""

from __future__ import annotations

import math

import torch

import minicompiler_amd as mc

DEVICE = "cuda"

# Normalisation applied to rows, its statistics given per row: the broadcast of [M, 1] inputs and of [N] constants.
ROW_NORM = """graph row_norm
dim M = 4096
dim N = 4096
input x : f32[M, N]
input mean : f32[M, 1]
input rstd : f32[M, 1]
const gamma : f32[N] = uniform(seed=4, lo=0.5, hi=1.5)
const beta : f32[N] = uniform(seed=5, lo=-0.1, hi=0.1)
centered = sub x, mean
normed = mul centered, rstd
scaled = mul normed, gamma
y = add scaled, beta
output y
"""

# The distribution of each graph's inputs: ("uniform", lo, hi) or ("normal", mean, std).
INPUTS = {
    "gelu_chain": [("uniform", -3.0, 3.0)],
    "batchnorm_relu": [("normal", 0.0, 1.0)],
    "row_norm": [("normal", 0.0, 1.0), ("normal", 0.0, 0.1), ("uniform", 0.5, 2.0)],
    "mlp_gelu": [("uniform", -1.0, 1.0)],
    "mlp_block_bn": [("uniform", -1.0, 1.0)],
    "matmul_bias_relu": [("uniform", -1.0, 1.0)],
    "matmul_bias_gelu": [("uniform", -1.0, 1.0)],
}
DIMS = {"gelu_chain": "MN", "batchnorm_relu": "RC", "row_norm": "MN", "mlp_gelu": "BDH", "mlp_block_bn": "BDH",
        "matmul_bias_relu": "MKN", "matmul_bias_gelu": "MKN"}
ELEMENTWISE = ("gelu_chain", "batchnorm_relu", "row_norm")
LOW_PRECISION = {"tensor_core_bf16": (mc.DTYPE_BF16, torch.bfloat16), "tensor_core_f16": (mc.DTYPE_F16, torch.float16)}


def listed():
    return [
        # One request through the MLP block: launches and the weights' bytes are all there is.
        {"name": "mlp_one_row", "graph": "mlp_gelu", "B": 1, "D": 512, "H": 2048},
        # A batch that fills no tile, with BatchNorm between the layers.
        {"name": "mlp_bn_100_rows", "graph": "mlp_block_bn", "B": 100, "D": 512, "H": 2048},
        # The benchmark's headline: the MLP block at its full batch.
        {"name": "mlp_8192_rows", "graph": "mlp_gelu", "B": 8192, "D": 512, "H": 2048},
        # A classifier-like layer whose sizes divide by nothing.
        {"name": "linear_ragged", "graph": "matmul_bias_relu", "M": 2000, "K": 1023, "N": 1001},
        # The FP32 operator on few rows: bound by the weights' bytes.
        {"name": "gemm_f32_16_rows", "gemm": "auto", "M": 16, "K": 4096, "N": 4096},
        # Activations of a transformer block through GELU.
        {"name": "gelu_4096x4096", "graph": "gelu_chain", "M": 4096, "N": 4096},
        # Inference BatchNorm over an odd number of channels and rows.
        {"name": "batchnorm_odd", "graph": "batchnorm_relu", "R": 50177, "C": 129},
        # A row-wise normalisation applied with per-row statistics.
        {"name": "row_norm", "graph": "row_norm", "M": 8192, "N": 2048},
        # The FFN shape of the benchmark on the bf16 matrix cores, bias and GELU in the same graph.
        {"name": "ffn_bf16", "graph": "matmul_bias_gelu", "M": 4096, "K": 4096, "N": 14336,
         "matmul": "tensor_core_bf16"},
        # The same kind of layer on a serving batch, fp16.
        {"name": "ffn_f16_32_rows", "graph": "matmul_bias_gelu", "M": 32, "K": 4096, "N": 4096,
         "matmul": "tensor_core_f16"},
        # The operator on fp32 operands that the matrix cores take as bf16 (rounded inside the call).
        {"name": "gemm_bf16_from_f32", "gemm": "tensor_core_bf16", "M": 2048, "K": 2048, "N": 2048, "operands": 32},
        # The operator on 16-bit operands, at sizes that are no multiple of a tile.
        {"name": "gemm_bf16_ragged", "gemm": "tensor_core_bf16", "M": 1000, "K": 1000, "N": 1000, "operands": 16},
    ]


def _size(rng, lo, hi):
    """A size between lo and hi, even over its logarithm: as it falls, or a multiple of 8 or of 64."""
    n = round(math.exp(rng.uniform(math.log(lo), math.log(hi))))
    step = rng.choice((1, 1, 8, 64))
    return max(lo, min(hi, (n + step - 1) // step * step))


def draw(rng):
    kind = rng.choice(("elementwise", "mlp", "linear", "lowp graph", "gemm f32", "gemm 16"))
    if kind == "elementwise":
        graph = rng.choice(ELEMENTWISE)
        cols = _size(rng, 64, 4096)
        rows = _size(rng, (1 << 20) // cols, (1 << 24) // cols)
        a, b = DIMS[graph]
        return {"graph": graph, a: rows, b: cols}
    if kind == "mlp":
        d = _size(rng, 128, 512)
        return {"graph": rng.choice(("mlp_gelu", "mlp_block_bn")), "B": _size(rng, 1, 8192), "D": d,
                "H": rng.choice((2, 4)) * d}
    case = {"graph": "matmul_bias_relu"} if kind == "linear" else {"graph": "matmul_bias_gelu"}
    most = 1 << 33  # multiply-adds of an fp32 product
    kernel = rng.choice(sorted(LOW_PRECISION))
    if kind == "lowp graph":
        case["matmul"] = kernel
        most = 1 << 36
    elif kind == "gemm f32":
        case = {"gemm": "auto"}
    elif kind == "gemm 16":
        case = {"gemm": kernel, "operands": rng.choice((16, 32))}
        most = 1 << 34
    case["M"] = _size(rng, 1, 4096)
    case["K"] = _size(rng, 256, 4096)
    case["N"] = _size(rng, 256, max(256, min(4096, most // (case["M"] * case["K"]))))
    return case


# ---------------------------------------------------------------- inputs and passes

_stream = None


def _ready():
    """PyTorch's GPU context before the library loads (one HIP runtime serves both); the stream of all passes."""
    global _stream
    if _stream is None:
        torch.zeros(1, device=DEVICE)
        _stream = torch.cuda.Stream()
        mc.library()
    return _stream


def _values(shape, dist, gen):
    kind, a, b = dist
    t = torch.empty(shape, dtype=torch.float32, device=DEVICE)
    return t.uniform_(a, b, generator=gen) if kind == "uniform" else t.normal_(a, b, generator=gen)


def _compile(case, **kw):
    dims = {d: case[d] for d in DIMS[case["graph"]]}
    if case["graph"] == "row_norm":
        return mc.Compiled(ROW_NORM, dims=dims, **kw)
    return mc.Compiled(path=mc.graph_path(case["graph"]), dims=dims, **kw)


def _graph_inputs(case, graph, seed):
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    return [_values(graph["nodes"][n]["shape"], dist, gen) for n, dist in zip(graph["inputs"], INPUTS[case["graph"]])]


def _operands(case, seed):
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    a = _values((case["M"], case["K"]), ("uniform", -1.0, 1.0), gen)
    b = _values((case["K"], case["N"]), ("uniform", -1.0, 1.0), gen)
    if case.get("operands") == 16:
        a, b = (t.to(LOW_PRECISION[case["gemm"]][1]) for t in (a, b))
    return a, b


def prepare(case, seed):
    stream = _ready()
    if "graph" in case:
        compiled = _compile(case, options={"matmul": case["matmul"]} if "matmul" in case else None)
        graph = compiled.graph()
        inputs = _graph_inputs(case, graph, seed)
        outputs = [torch.empty(graph["nodes"][o]["shape"], dtype=torch.float32, device=DEVICE)
                   for o in graph["outputs"]]
        compiled.bind_inputs([t.data_ptr() for t in inputs])
        compiled.bind_outputs([t.data_ptr() for t in outputs])
        torch.cuda.synchronize()
        return {"compiled": compiled, "inputs": inputs, "outputs": outputs, "stream": stream.cuda_stream}
    m, n, k = case["M"], case["N"], case["K"]
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    kernel = mc.resolve_matmul_kernel(case["gemm"], m, n, k, cus)
    splits = mc.matmul_splits(kernel, m, n, k, cus)
    nbytes = mc.matmul_workspace_bytes(kernel, m, n, splits)
    a, b = _operands(case, seed)
    state = {"kernel": mc.matmul_kernel_id(kernel), "a": a, "b": b, "sizes": (m, n, k), "splits": splits,
             "c": torch.empty((m, n), dtype=torch.float32, device=DEVICE),
             "workspace": torch.empty(nbytes // 4, dtype=torch.float32, device=DEVICE) if nbytes else None,
             "dtype": LOW_PRECISION[kernel][0] if case.get("operands") == 16 else 0, "stream": stream.cuda_stream}
    torch.cuda.synchronize()
    return state


def run(state):
    if "compiled" in state:
        state["compiled"].enqueue(state["stream"])
        return state["outputs"]
    a, b, c, ws = state["a"], state["b"], state["c"], state["workspace"]
    m, n, k = state["sizes"]
    workspace = ws.data_ptr() if ws is not None else None
    if state["dtype"]:
        mc.launch_matmul_lowp(state["kernel"], state["dtype"], a.data_ptr(), b.data_ptr(), c.data_ptr(), m, n, k,
                              state["stream"], state["splits"], workspace)
    else:
        mc.launch_matmul(state["kernel"], a.data_ptr(), b.data_ptr(), c.data_ptr(), m, n, k, state["stream"],
                         state["splits"], workspace)
    return c


# ---------------------------------------------------------------- work and results


def work(case):
    """Each input and constant read once and each output written once; two operations per multiply-add, none counted
    for elementwise groups."""
    if "graph" in case and case["graph"] in ELEMENTWISE:
        rows, cols = (case[d] for d in DIMS[case["graph"]])
        per_col = {"gelu_chain": 0, "batchnorm_relu": 4, "row_norm": 2}[case["graph"]]
        per_row = 2 if case["graph"] == "row_norm" else 0
        return {"bytes": 4 * (2 * rows * cols + per_col * cols + per_row * rows), "flops": 0}
    if case.get("graph", "").startswith("mlp"):
        b, d, h = case["B"], case["D"], case["H"]
        vectors = d + h if case["graph"] == "mlp_gelu" else d + 5 * h
        return {"bytes": 4 * (2 * b * d + 2 * d * h + vectors), "flops": 4 * b * d * h}
    m, n, k = case["M"], case["N"], case["K"]
    # A graph's constant operand can be kept in 16 bits; its input x comes in fp32.
    if "graph" in case:
        nbytes = 4 * (m * k + m * n + n) + (2 if "matmul" in case else 4) * k * n
    else:
        size = 2 if case.get("operands") == 16 else 4
        nbytes = size * (m * k + k * n) + 4 * m * n
    return {"bytes": nbytes, "flops": 2 * m * n * k}


def tolerance(case):
    # fp32 arithmetic throughout, or fp32 sums of exact 16-bit products: only the order of the sums, the contraction
    # of a multiply and an add, and tanh's last bits are free. About four times the measured distance from the 64-bit
    # results: 5e-8 for the elementwise graphs, up to 5e-7 for products over K = 4096.
    if "graph" in case and case["graph"] in ELEMENTWISE:
        return {"rel": 2.5e-7}
    return {"rel": 2e-6}


_UNARY = {"neg": torch.neg, "exp": torch.exp, "log": torch.log, "sqrt": torch.sqrt, "relu": torch.relu,
          "sigmoid": torch.sigmoid, "tanh": torch.tanh}
_BINARY = {"add": torch.add, "sub": torch.sub, "mul": torch.mul, "div": torch.div}


def exact(case, seed):
    """The graph as written, node by node, or the product, in float64; operands of the 16-bit matrix cores are
    rounded to their type first, as the kernel's name says."""
    _ready()
    if "gemm" in case:
        a, b = _operands(case, seed)
        if case["gemm"] in LOW_PRECISION:
            a, b = (t.to(LOW_PRECISION[case["gemm"]][1]) for t in (a, b))
        return torch.matmul(a.double(), b.double())
    compiled = _compile(case, passes="none", backend="none")
    graph = compiled.graph()
    nodes = graph["nodes"]
    values = {n: t.double() for n, t in zip(graph["inputs"], _graph_inputs(case, graph, seed))}
    for node in nodes:
        if node["op_name"] == "input":
            continue
        if node["op_name"] == "const":
            values[node["id"]] = torch.from_numpy(compiled.constant(node["id"])).to(DEVICE).double().reshape(node["shape"])
            continue
        args = [values[i] for i in node["inputs"]]
        if node["op_name"] == "matmul":
            if "matmul" in case:
                args = [t.to(LOW_PRECISION[case["matmul"]][1]).double() for t in args]
            values[node["id"]] = torch.matmul(*args)
        else:
            values[node["id"]] = (_UNARY.get(node["op_name"]) or _BINARY[node["op_name"]])(*args)
    return [values[o] for o in graph["outputs"]]
