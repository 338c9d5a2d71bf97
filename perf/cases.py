"""The workloads whose speed is followed: what a program that uses this library has it compute, through the entry
points it calls.  listed() are fixed sizes, draw() gives more of the same ranges, prepare() / run() make the inputs
and one pass, work() and tolerance() say what a pass must move and compute and how exact its results are.

Partitions (JSON and textual MLIR) run through execute_async on the current stream with tensors that stay on the
GPU; single GEMMs and attention run through the package's functions.
"""
import importlib
import importlib.util
import math
import os
import sys

import numpy as np
import torch


def _package():
    """graph-compiler_amd/ has a hyphen in its name: import it by path, from the tree that is the working folder."""
    name = "graph_compiler_amd"
    if name not in sys.modules:
        pkg = os.path.join(os.getcwd(), "graph-compiler_amd")
        spec = importlib.util.spec_from_file_location(name, os.path.join(pkg, "__init__.py"),
                                                      submodule_search_locations=[pkg])
        mod = importlib.util.module_from_spec(spec)
        sys.modules[name] = mod
        spec.loader.exec_module(mod)
    return sys.modules[name]


gc = _package()
ga = importlib.import_module("graph_compiler_amd.graph_api")
mm = importlib.import_module("graph_compiler_amd.mlir_modules")


# ------------------------------------------------------------------------------------------------------- the cases
def listed():
    return [
        # one small f32 layer (matmul + bias + ReLU): the call whose cost is the launch
        {"name": "f32_layer_small", "kind": "f32_layer", "M": 128, "K": 512, "N": 256},
        # a three-layer f32 MLP over a batch that fills no tile evenly (the pattern the reference's harness builds)
        {"name": "f32_mlp_ragged", "kind": "f32_mlp", "M": 1111, "h0": 1000, "h1": 3000, "h2": 1000, "h3": 500},
        # the large square product: every compute unit busy for one round of large tiles
        {"name": "bf16_gemm_large", "kind": "bf16_gemm", "M": 4096, "N": 4096, "K": 4096, "act": "none"},
        # a feed-forward shard of a Llama-sized layer split over eight devices (11008 / 8 = 1376, no multiple of a
        # K block) over an odd number of tokens; weights as torch.nn.Linear stores them, bias and GELU
        {"name": "bf16_linear_shard", "kind": "bf16_linear", "M": 1237, "N": 4096, "K": 1376, "act": "gelu_erf"},
        # the quantised feed-forward layer, prefill and decode
        {"name": "int8_layer_prefill", "kind": "int8_layer", "M": 4096, "K": 4096, "N": 11008},
        {"name": "int8_layer_decode", "kind": "int8_layer", "M": 32, "K": 4096, "N": 11008},
        # attention over a prompt: causal mask as data, as the reference's graph has it
        {"name": "mha_prefill_causal", "kind": "mha", "B": 4, "H": 32, "Sq": 2048, "Sk": 2048, "D": 128, "mask": "causal"},
        # attention of ragged queries over ragged keys (an encoder's output), no mask, head dim 64
        {"name": "mha_cross_ragged", "kind": "mha", "B": 8, "H": 16, "Sq": 500, "Sk": 777, "D": 64, "mask": "none"},
        # attention of one new token per sequence over its cached keys
        {"name": "mha_decode", "kind": "mha", "B": 8, "H": 32, "Sq": 1, "Sk": 4096, "D": 128, "mask": "none"},
        # the second half of a llama-2 decoder layer (projection, two norms, gated feed-forward): decode and prefill
        {"name": "block_decode", "kind": "block", "T": 32, "hidden": 4096, "ffn": 11008},
        {"name": "block_prefill", "kind": "block", "T": 1000, "hidden": 4096, "ffn": 11008},
        # a norm over many rows: memory traffic only
        {"name": "rmsnorm_large", "kind": "rmsnorm", "rows": 16384, "hidden": 4096, "dtype": "bf16"},
    ]


def _log(rng, lo, hi, mult=1):
    """An integer in [lo, hi], uniform in its logarithm, a multiple of `mult`."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return max(mult * ((lo + mult - 1) // mult), min(hi, (v + mult // 2) // mult * mult))


def _mult(rng, coarse, fine):
    """Most sizes are multiples of a hardware-friendly number, some are not."""
    return coarse if rng.random() < 0.6 else fine


def draw(rng):
    kind = rng.choice(["f32_layer", "f32_mlp", "bf16_gemm", "bf16_linear", "int8_layer", "mha_prefill", "mha_decode",
                       "block", "norm"])
    if kind == "f32_layer":
        return {"kind": kind, "M": _log(rng, 1, 512), "K": _log(rng, 16, 2048, _mult(rng, 16, 1)),
                "N": _log(rng, 16, 2048, _mult(rng, 16, 1))}
    if kind == "f32_mlp":
        h = [_log(rng, 64, 3000, _mult(rng, 8, 1)) for _ in range(4)]
        return {"kind": kind, "M": _log(rng, 16, 1200), "h0": h[0], "h1": h[1], "h2": h[2], "h3": h[3]}
    if kind == "bf16_gemm":
        return {"kind": kind, "M": _log(rng, 16, 4096), "N": _log(rng, 64, 4096, _mult(rng, 64, 8)),
                "K": _log(rng, 64, 4096, _mult(rng, 64, 8)), "act": rng.choice(["none", "relu"])}
    if kind == "bf16_linear":
        return {"kind": kind, "M": _log(rng, 1, 2048), "N": _log(rng, 512, 8192, _mult(rng, 64, 8)),
                "K": _log(rng, 512, 4096, _mult(rng, 64, 8)), "act": rng.choice(["none", "relu", "gelu_erf", "gelu_tanh"])}
    if kind == "int8_layer":
        return {"kind": kind, "M": _log(rng, 1, 4096), "K": _log(rng, 512, 4096, _mult(rng, 64, 16)),
                "N": _log(rng, 512, 11008, _mult(rng, 64, 16))}
    if kind == "mha_prefill":
        Sq = _log(rng, 32, 2048)
        causal = rng.random() < 0.5
        return {"kind": "mha", "B": rng.randint(1, 4), "H": rng.choice([8, 12, 16, 32]), "Sq": Sq,
                "Sk": Sq if causal else _log(rng, 32, 1500), "D": rng.choice([64, 128]),
                "mask": "causal" if causal else "none"}
    if kind == "mha_decode":
        Sq = rng.choice([1, 1, 1, 2, 4, 7, 16])
        B, H = rng.choice([1, 2, 4, 8, 16]), rng.choice([8, 16, 32])
        hi = min(8192, 8 * 32 * 4096 // (B * H))
        return {"kind": "mha", "B": B, "H": H, "Sq": Sq, "Sk": _log(rng, 64, hi), "D": rng.choice([64, 128]),
                "mask": "causal" if Sq > 1 else "none"}
    if kind == "block":
        hidden, ffn = rng.choice([(4096, 11008), (2048, 5632), (1024, 2816)])
        return {"kind": kind, "T": _log(rng, 1, 1000), "hidden": hidden, "ffn": ffn}
    return {"kind": rng.choice(["rmsnorm", "layernorm", "softmax"]), "rows": _log(rng, 4, 16384),
            "hidden": _log(rng, 128, 4096, _mult(rng, 64, 4)), "dtype": "bf16"}


# ----------------------------------------------------------------------------------------------------- preparation
class _Partition:
    """A compiled partition with its tensors bound: what a program keeps for as long as it uses a model."""

    def __init__(self, text, mlir, inputs, outputs):
        self.compiler = ga.Compiler()
        status, self.exe = (self.compiler.compile_mlir if mlir else self.compiler.compile)(text)
        if status:
            self.exe = None
            raise RuntimeError("compile -> %d: %s" % (status, ga.api().dnnl_graph_compiler_last_error().decode()))
        self.inputs, self.outputs = inputs, outputs
        self.calls = {}

    def __call__(self):
        stream = torch.cuda.current_stream().cuda_stream
        if stream not in self.calls:
            self.calls[stream] = self.exe.bind(self.inputs, self.outputs, stream)
        status = self.calls[stream]()
        if status:
            raise RuntimeError("execute_async -> %d: %s" % (status, ga.api().dnnl_graph_compiler_last_error().decode()))
        return [t for _, t in self.outputs]

    def __del__(self):
        if self.exe is not None:
            self.exe.close()
        self.compiler.close()


class _Random:
    """Seeded tensors made on the GPU."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(int(seed))

    def normal(self, *shape, std=1.0, dtype=torch.bfloat16):
        return (torch.randn(*shape, device="cuda", generator=self.gen) * std).to(dtype)

    def uniform(self, *shape, lo=-1.0, hi=1.0):
        return torch.rand(*shape, device="cuda", generator=self.gen) * (hi - lo) + lo

    def integers(self, lo, hi, shape, dtype):
        return torch.randint(lo, hi, shape, device="cuda", generator=self.gen, dtype=torch.int32).to(dtype)


def _empty(*shape, dtype=torch.bfloat16):
    return torch.empty(*shape, device="cuda", dtype=dtype)


def _softmax_json(rows, hidden, dtype):
    t = {"dtype": dtype, "shape": [rows, hidden]}
    return ga._graph([{"kind": "SoftMax", "attrs": {"axis": {"type": "s64", "value": -1}},
                       "inputs": [dict(t, id=0)], "outputs": [dict(t, id=1)]}], [0], [1])


def prepare(case, seed):
    r, kind = _Random(seed), case["kind"]
    if kind == "f32_layer":
        M, K, N = case["M"], case["K"], case["N"]
        ins = [(0, r.uniform(M, K)), (1, r.uniform(K, N)), (2, r.uniform(N))]
        return _Partition(ga.matmul_bias_relu_json(M, K, N), False, ins, [(4, _empty(M, N, dtype=torch.float32))])
    if kind == "f32_mlp":
        M, h = case["M"], [case["h0"], case["h1"], case["h2"], case["h3"]]
        ins = [r.uniform(M, h[0])]
        ins += [r.normal(h[i], h[i + 1], std=h[i] ** -0.5, dtype=torch.float32) for i in range(3)]
        ins += [r.normal(h[i + 1], std=0.1, dtype=torch.float32) for i in range(3)]
        return _Partition(mm.mlp(M, h, [True] * 3, "relu", "f32"), True, list(enumerate(ins)),
                          [(len(ins), _empty(M, h[3], dtype=torch.float32))])
    if kind == "bf16_gemm":
        M, N, K = case["M"], case["N"], case["K"]
        return {"A": r.normal(M, K, std=0.1), "B": r.normal(K, N, std=0.1), "act": case["act"]}
    if kind == "bf16_linear":
        M, N, K = case["M"], case["N"], case["K"]
        return {"A": r.normal(M, K), "Bt": r.normal(N, K, std=0.02), "bias": r.normal(N, std=0.02), "act": case["act"]}
    if kind == "int8_layer":
        M, K, N = case["M"], case["K"], case["N"]
        A = r.integers(0, 256, (M, K), torch.uint8)
        W = r.integers(-127, 128, (K, N), torch.int8)
        # scales of a calibrated layer: results of a few units
        scale_w = np.random.RandomState(int(seed) % (1 << 31)).uniform(0.5, 1.5, N) * 2e-2
        text, last = ga.int8_mlp_json(M, K, N, 1.0 / (64.0 * K ** 0.5), 128, scale_w)
        return _Partition(text, False, [(0, A), (1, W), (2, r.normal(N, dtype=torch.float32))], [(last, _empty(M, N))])
    if kind == "mha":
        B, H, Sq, Sk, D = case["B"], case["H"], case["Sq"], case["Sk"], case["D"]
        mask = None
        if case["mask"] == "causal":  # the last query sees every key
            mask = torch.triu(torch.full((Sq, Sk), float("-inf"), device="cuda"), diagonal=1 + Sk - Sq)
        return {"Q": r.normal(B, H, Sq, D), "K": r.normal(B, H, Sk, D), "V": r.normal(B, H, Sk, D), "mask": mask}
    if kind == "block":
        T, H, F = case["T"], case["hidden"], case["ffn"]
        eps = torch.full((1,), 1e-5, device="cuda")
        ins = [r.normal(1, T, H), r.normal(H, H, std=0.02), r.normal(1, T, H), eps, 1 + r.normal(H, std=0.1),
               r.normal(F, H, std=0.02), r.normal(F, H, std=0.02), r.normal(H, F, std=0.02), eps.clone(),
               1 + r.normal(H, std=0.1)]
        return _Partition(mm.decoder_mlp_block(T, H, F), True, list(enumerate(ins)),
                          [(10, _empty(1, T, H)), (11, _empty(1, T, H))])
    rows, hidden = case["rows"], case["hidden"]
    if kind == "rmsnorm":
        ins = [r.normal(1, rows, hidden), torch.full((1,), 1e-5, device="cuda"), 1 + r.normal(hidden, std=0.1)]
        return _Partition(mm.rmsnorm(rows, hidden), True, list(enumerate(ins)), [(3, _empty(1, rows, hidden))])
    if kind == "layernorm":
        ins = [r.normal(rows, hidden), 1 + r.normal(hidden, std=0.1), r.normal(hidden, std=0.1)]
        return _Partition(mm.layernorm(rows, hidden, "bf16"), True, list(enumerate(ins)), [(3, _empty(rows, hidden))])
    if kind == "softmax":
        return _Partition(_softmax_json(rows, hidden, "bf16"), False, [(0, r.normal(rows, hidden, std=2.0))],
                          [(1, _empty(rows, hidden))])
    raise ValueError(kind)


def run(state):
    if isinstance(state, _Partition):
        return state()
    if "Q" in state:
        return gc.mha_fwd_bf16(state["Q"], state["K"], state["V"], state["mask"])
    act = None if state["act"] == "none" else state["act"]
    if "Bt" in state:
        return gc.gemm_bf16_nt(state["A"], state["Bt"], bias=state["bias"], act=act)
    return gc.gemm_bf16(state["A"], state["B"], act=act)


# ---------------------------------------------------------------------------------------------- work and tolerances
def work(case):
    kind = case["kind"]
    if kind == "f32_layer":
        M, K, N = case["M"], case["K"], case["N"]
        return {"bytes": 4 * (M * K + K * N + N + M * N), "flops": 2 * M * K * N}
    if kind == "f32_mlp":
        M, h = case["M"], [case["h0"], case["h1"], case["h2"], case["h3"]]
        weights = sum(h[i] * h[i + 1] + h[i + 1] for i in range(3))
        return {"bytes": 4 * (M * h[0] + weights + M * h[3]), "flops": 2 * M * sum(h[i] * h[i + 1] for i in range(3))}
    if kind in ("bf16_gemm", "bf16_linear"):
        M, N, K = case["M"], case["N"], case["K"]
        return {"bytes": 2 * (M * K + K * N + M * N + (N if kind == "bf16_linear" else 0)), "flops": 2 * M * N * K}
    if kind == "int8_layer":
        M, K, N = case["M"], case["K"], case["N"]
        return {"bytes": M * K + K * N + 4 * 3 * N + 2 * M * N, "flops": 2 * M * N * K}
    if kind == "mha":
        BH, Sq, Sk, D = case["B"] * case["H"], case["Sq"], case["Sk"], case["D"]
        pairs, mask = Sq * Sk, 0
        if case["mask"] == "causal":  # query i sees keys 0 .. Sk - Sq + i
            pairs = sum(max(0, Sk - Sq + i + 1) for i in range(Sq))
            mask = 4 * Sq * Sk
        return {"bytes": 2 * BH * D * (2 * Sq + 2 * Sk) + mask, "flops": 4 * BH * pairs * D}
    if kind == "block":
        T, H, F = case["T"], case["hidden"], case["ffn"]
        return {"bytes": 2 * (H * H + 3 * H * F + 2 * H + 4 * T * H) + 8, "flops": 2 * T * (H * H + 3 * H * F)}
    rows, hidden = case["rows"], case["hidden"]
    vectors = {"rmsnorm": 1, "layernorm": 2, "softmax": 0}[kind]
    return {"bytes": 2 * (2 * rows * hidden + vectors * hidden), "flops": 8 * rows * hidden}


def tolerance(case):
    """Relative errors (2-norm) of another correct implementation of the same precision: about four times what the
    present one shows against a float64 evaluation with no rounding in between (f32 up to 9.4e-7 through three layers;
    bf16 results 1.6e-3 to 3.4e-3 with up to three roundings; the decoder block, nine rounded tensors deep, 5.9e-3)."""
    kind = case["kind"]
    if kind in ("f32_layer", "f32_mlp"):
        return {"rel": 4e-6}
    if kind == "block":
        return {"rel": 2.4e-2}
    return {"rel": 1e-2}
