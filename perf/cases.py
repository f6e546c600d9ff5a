"""Workloads for timing the library through its public entry points.

A case is one call, or one decoder layer's sequence of calls, that a serving process makes:

* ``fused_norm``  `fused_allreduce_layernorm` on a `PartialsBuffer`: sum of the tensor-parallel
                  partials, residual add and RMSNorm, in place, on one rank's rows or on all;
* ``norm``        `RMSNorm` without a reduction: with residual, first layer (`out=`), plain;
* ``quant``       the norm with fp8 / int8 output, static scale or one per token;
* ``linear``      `RowParallelLinear(..., is_tokenweave=True)`: o_proj / down_proj in place;
* ``producer``    `gemm_bf16_nt_partials`: the projections of all ranks in one call;
* ``layer``       `tokenweave_with_fuse_only` or `tokenweave_overlap` on one decoder layer with
                  this rank's o_proj and down_proj, as `weave_plan` decides.

Shapes are those of the shipped weave tables (`MODELS`), of `tokenweave_amd.workloads`, and
generic ones of the unit tests (odd hidden sizes, fp16 and fp32).
"""
import math

import torch

import tokenweave_amd as tw
from tokenweave_amd import _custom_ops as ops

DEV = "cuda"
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}

# shipped weave table -> (hidden size, ranks, inner size of o_proj, of down_proj, eps)
MODELS = {
    "llama_config_8": (8192, 8, 1024, 3584, 1e-5),
    "llama_config_4": (8192, 4, 2048, 7168, 1e-5),
    "qwen2_config_8": (8192, 8, 1024, 3696, 1e-6),
    "qwen2_config_4": (8192, 4, 2048, 7392, 1e-6),
    "mixtral_config_8": (6144, 8, 768, 2048, 1e-5),
}
WEAVE_TOKENS = 1024       # batches from here on may be woven: this GPU then normalises all rows itself
MOST_FLOPS = 1.2e12       # the largest listed case's: nothing drawn costs more
MOST_ELEMENTS = 1 << 29   # of one staging allocation of a drawn norm


def listed():
    return [
        # 64 sequences decoding: one rank's 8 rows of the fused op, twice per layer and token
        {"name": "fused_norm_decode", "kind": "fused_norm", "P": 8, "tokens": 64, "H": 8192, "all": False, "eps": 1e-5},
        # a 2048-token prefill step: one rank's 256 rows
        {"name": "fused_norm_shard", "kind": "fused_norm", "P": 8, "tokens": 2048, "H": 8192, "all": False, "eps": 1e-5},
        # a ragged batch, every row on this GPU
        {"name": "fused_norm_ragged", "kind": "fused_norm", "P": 8, "tokens": 3001, "H": 8192, "all": True, "eps": 1e-6},
        # a long prefill chunk at a hidden size that is no power of two
        {"name": "fused_norm_chunk", "kind": "fused_norm", "P": 8, "tokens": 8192, "H": 6144, "all": True, "eps": 1e-5},
        # add + norm without tensor parallelism, a mid-size step
        {"name": "add_norm_512", "kind": "norm", "mode": "add", "tokens": 512, "H": 8192, "dtype": "bf16"},
        # full-precision tensors, a prefill-size batch at a hidden size of the unit tests
        {"name": "add_norm_fp32", "kind": "norm", "mode": "add", "tokens": 4096, "H": 5120, "dtype": "fp32"},
        # input of an fp8 GEMM: norm and one scale per token
        {"name": "quant_fp8_token", "kind": "quant", "mode": "dyn_fp8", "tokens": 2048, "H": 8192, "dtype": "bf16",
         "residual": True},
        # down_proj of a decode step of 32 sequences
        {"name": "linear_decode", "kind": "linear", "M": 32, "N": 8192, "K": 3584, "bias": False},
        # down_proj of a ragged mixed step at an inner size that is no multiple of 64
        {"name": "linear_ragged", "kind": "linear", "M": 1000, "N": 8192, "K": 3696, "bias": False},
        # o_proj of the larger token split of a 4096-token batch, all eight ranks' partial sums
        {"name": "producer_split", "kind": "producer", "P": 8, "M": 2458, "N": 8192, "K": 1024},
        # a decoder layer while 64 sequences decode (below the weave threshold: fuse only)
        {"name": "layer_decode", "kind": "layer", "model": "llama_config_8", "tokens": 64},
        # a decoder layer of a large prefill batch, woven
        {"name": "layer_prefill", "kind": "layer", "model": "llama_config_8", "tokens": 16384},
    ]


def _log_int(rng, low, high):
    """Spread over the logarithm; half of the larger values are rounded to a multiple of 8."""
    n = int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))
    if n > 64 and rng.random() < 0.5:
        n = (n + 7) // 8 * 8
    return max(low, min(high, n))


def _fused_hidden(rng):
    return rng.choice((8192, 8192, 6144, 5120, 4096, 8 * rng.randint(128, 2048)))


def draw(rng):
    kind = rng.choice(("fused_norm", "fused_norm", "fused_norm", "norm", "norm", "quant", "linear", "linear", "linear",
                       "producer", "layer", "layer"))
    if kind == "fused_norm":
        P, H = rng.choice((8, 8, 8, 4, 4, 2, 3, 5)), _fused_hidden(rng)
        tokens = min(_log_int(rng, 1, 16384), MOST_ELEMENTS // (P * H))
        return {"kind": kind, "P": P, "tokens": tokens, "H": H, "all": rng.random() < 0.5,
                "eps": rng.choice((1e-5, 1e-6))}
    if kind == "norm":
        H = rng.choice((8192, 8192, 6144, 5120, 4096, rng.randint(768, 8199)))
        return {"kind": kind, "mode": rng.choice(("add", "add", "first", "plain")), "tokens": _log_int(rng, 1, 16384),
                "H": H, "dtype": rng.choice(("bf16", "bf16", "fp16", "fp32"))}
    if kind == "quant":
        mode = rng.choice(("dyn_fp8", "dyn_fp8", "dyn_int8", "static_fp8"))
        return {"kind": kind, "mode": mode, "tokens": _log_int(rng, 1, 8192),
                "H": rng.choice((8192, 8192, 6144, 5120, 4096, rng.randint(768, 8199))),
                "dtype": rng.choice(("bf16", "bf16", "fp16")), "residual": rng.random() < 0.7}
    H, P, k_attn, k_mlp, _ = MODELS[rng.choice(sorted(MODELS))] if kind != "layer" else (0, 0, 0, 0, 0)
    if kind == "linear":
        return {"kind": kind, "M": _log_int(rng, 1, 8192), "N": H, "K": rng.choice((k_attn, k_mlp)),
                "bias": rng.random() < 0.25}
    if kind == "producer":
        K = rng.choice((k_attn, k_mlp))
        M = min(_log_int(rng, 1, 4096), int(MOST_FLOPS / (2.0 * P * H * K)))
        return {"kind": kind, "P": P, "M": M, "N": H, "K": K}
    model = rng.choice(sorted(MODELS))
    H, P, k_attn, k_mlp, _ = MODELS[model]
    most = min(16384, int(MOST_FLOPS / (2.0 * H * (k_attn + k_mlp))))
    return {"kind": kind, "model": model, "tokens": max(P, _log_int(rng, P, most) // P * P)}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _normal(shape, g, dtype=torch.bfloat16, mean=0.0, std=1.0):
    t = torch.randn(shape, generator=g, device=DEV, dtype=dtype)
    if std != 1.0:
        t.mul_(std)
    return t.add_(mean) if mean else t


def _rms_norm_layer(H, eps, g, dtype=torch.bfloat16):
    layer = tw.RMSNorm(H, eps=eps, dtype=dtype).to(DEV)
    layer.weight.data.copy_(_normal((H,), g, torch.float32, 1.0, 0.1))
    return layer


def _row_parallel(K, N, ranks, g, bias=False):
    layer = tw.RowParallelLinear(K * ranks, N, bias=bias, tp_rank=0, tp_size=ranks).to(DEV)
    layer.weight.data.copy_(_normal((N, K), g, std=0.02))
    if bias:
        layer.bias.data.copy_(_normal((N,), g, std=0.1))
    return layer


def _staging(P, tokens, H, rank, g):
    """The ranks' partial sums, each slot N(0, 1/P), so that their sum is about N(0, 1)."""
    buf = tw.PartialsBuffer(P, tokens, H, rank=rank, device=DEV)
    for p in range(P):
        buf.slot(p).copy_(_normal((tokens, H), g, std=P ** -0.5))
    return buf


def _copy_stream(made=[]):  # noqa: B006 — one side stream for the process, as a model runner keeps it
    if not made:
        made.append(torch.cuda.Stream())
    return made[0]


class _DecoderLayer:
    """What the schedules need of a model's layer: two norms, `self_attn` and an MLP whose
    row-parallel projections write this rank's partial sums over `hidden_states`.  The
    projections' inputs (attention output, activated gate / up product) are in hand."""

    def __init__(self, case, g):
        H, P, k_attn, k_mlp, eps = MODELS[case["model"]]
        T = case["tokens"]
        self.P, self.rank = P, P // 2
        self.buf = _staging(P, T, H, self.rank, g)
        self.hidden_states = self.buf.hidden_states(T)
        self.residual = _normal((T, H), g)
        self.positions = torch.arange(T, device=DEV)
        self.input_layernorm, self.post_attention_layernorm, self.next_layernorm = (
            _rms_norm_layer(H, eps, g) for _ in range(3))
        self.o_proj, self.down_proj = _row_parallel(k_attn, H, P, g), _row_parallel(k_mlp, H, P, g)
        self.attn_out, self.activated = _normal((T, k_attn), g), _normal((T, k_mlp), g)
        self.first, self.row_bytes = self.hidden_states.data_ptr(), H * 2
        config = tw.load_config("tokenweave_configs/%s.json" % case["model"])
        self.plan = tw.weave_plan(T, config)
        self.copy_stream = _copy_stream()

    def self_attn(self, positions, hidden_states, split_id=0, split_size=0, num_actual_tokens=None, gemm_cus=None):
        n = hidden_states.shape[0]
        first = split_size if split_id else 0
        self.o_proj(self.attn_out[first:first + n], hidden_states, is_tokenweave=True, gemm_cus=gemm_cus)

    def mlp(self, hidden_states, gemm_cus=None):
        first = (hidden_states.data_ptr() - self.first) // self.row_bytes
        self.down_proj(self.activated[first:first + hidden_states.shape[0]], hidden_states, is_tokenweave=True,
                       gemm_cus=gemm_cus)

    def __call__(self):
        T, plan = self.hidden_states.shape[0], self.plan
        if plan is None:
            return tw.tokenweave_with_fuse_only(
                self, self.positions, self.hidden_states, self.residual, self.buf, 1, rank=self.rank,
                world_size=self.P, next_layer_norm=self.next_layernorm, actual_tokens=T,
                nearest_multiple_of_world_size=T, MAX_CTAS_ATTN=0, MAX_CTAS_MLP=0, mlp_fn=self.mlp,
                all_ranks=T >= WEAVE_TOKENS)
        return tw.tokenweave_overlap(
            self, self.positions, self.hidden_states, self.residual, self.buf, 1, end_layer=3, rank=self.rank,
            world_size=self.P, current_stream=torch.cuda.current_stream(), copy_stream=self.copy_stream,
            next_layer_norm=self.next_layernorm, split_size=plan["split_size"], actual_tokens=T,
            num_tokens_padded=T, MAX_CTAS_ATTN=plan["attention_ctas"], MAX_CTAS_MLP=plan["mlp_ctas"],
            mlp_fn=self.mlp, all_ranks=True, gemm_cus=plan["gemm_cus"], mlp_gemm_cus=plan.get("mlp_gemm_cus"))


def _rows(case):
    """Rows of the batch that the fused op of this case works on: all, or the shard of a rank
    in the middle (token counts that the ranks do not divide leave the last ones fewer)."""
    if case["all"]:
        return 0, case["tokens"]
    start, end = tw.shard_bounds(case["tokens"], (case["P"] - 1) // 2, case["P"], "ceil")
    return (start, end) if end > start else (0, 1)


def prepare(case, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    kind = case["kind"]
    if kind == "fused_norm":
        P, T, H = case["P"], case["tokens"], case["H"]
        rank = (P - 1) // 2
        buf = _staging(P, T, H, rank, g)
        return {"kind": kind, "buf": buf, "x": buf.hidden_states(T), "residual": _normal((T, H), g), "P": P,
                "rank": rank, "rows": _rows(case), "layer": _rms_norm_layer(H, case["eps"], g)}
    if kind == "norm":
        T, H, dtype = case["tokens"], case["H"], DTYPES[case["dtype"]]
        return {"kind": kind, "mode": case["mode"], "x": _normal((T, H), g, dtype),
                "residual": _normal((T, H), g, dtype), "layer": _rms_norm_layer(H, 1e-6, g, dtype)}
    if kind == "quant":
        T, H, dtype = case["tokens"], case["H"], DTYPES[case["dtype"]]
        return {"kind": kind, "mode": case["mode"], "x": _normal((T, H), g, dtype),
                "residual": _normal((T, H), g, dtype) if case["residual"] else None,
                "weight": _normal((H,), g, torch.float32, 1.0, 0.1).to(dtype),
                "scale": torch.full((1,), 0.02, device=DEV),
                "out": torch.empty((T, H), dtype=torch.float8_e4m3fn, device=DEV) if case["mode"] == "static_fp8" else None}
    if kind == "linear":
        M, N, K = case["M"], case["N"], case["K"]
        return {"kind": kind, "x": _normal((M, K), g), "layer": _row_parallel(K, N, 8, g, case["bias"]),
                "out": torch.empty((M, N), dtype=torch.bfloat16, device=DEV)}
    if kind == "producer":
        P, M, N, K = case["P"], case["M"], case["N"], case["K"]
        buf = tw.PartialsBuffer(P, M, N, device=DEV)
        return {"kind": kind, "buf": buf, "outs": [buf.slot(p) for p in range(P)],
                "a": [_normal((M, K), g) for _ in range(P)], "b": [_normal((N, K), g, std=0.02) for _ in range(P)]}
    return {"kind": kind, "layer": _DecoderLayer(case, g)}


def run(state):
    kind = state["kind"]
    if kind == "fused_norm":
        x, residual, (start, end) = state["x"], state["residual"], state["rows"]
        tw.fused_allreduce_layernorm(state["layer"], x, residual, state["buf"], 0, state["rank"], state["P"], 0,
                                     row_range=(start, end))
        return x[start:end], residual[start:end]
    if kind == "norm":
        if state["mode"] == "add":
            return state["layer"](state["x"], state["residual"])
        if state["mode"] == "first":
            return state["layer"](state["x"], out=state["residual"]), state["residual"]
        return state["layer"](state["x"])
    if kind == "quant":
        x, residual, w = state["x"], state["residual"], state["weight"]
        if state["mode"] == "static_fp8":
            if residual is None:
                ops.rms_norm_static_fp8_quant(state["out"], x, w, state["scale"], 1e-6)
            else:
                ops.fused_add_rms_norm_static_fp8_quant(state["out"], x, residual, w, state["scale"], 1e-6)
            return state["out"], residual
        dtype = torch.int8 if state["mode"] == "dyn_int8" else torch.float8_e4m3fn
        out, scales = ops.rms_norm_dynamic_per_token_quant(x, w, 1e-6, dtype, None, residual)
        return out, scales, residual
    if kind == "linear":
        return state["layer"](state["x"], state["out"], is_tokenweave=True)[0]
    if kind == "producer":
        ops.gemm_bf16_nt_partials(state["outs"], state["a"], state["b"])
        return state["outs"]
    return state["layer"]()


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _gemm_work(M, N, K):
    return (M * K + N * K + M * N) * 2, 2.0 * M * N * K


def work(case):
    kind = case["kind"]
    if kind == "fused_norm":
        start, end = _rows(case)
        rows, H = end - start, case["H"]
        return {"bytes": ((case["P"] + 3) * rows + 1) * H * 2, "flops": 0}
    if kind == "norm":
        size = DTYPES[case["dtype"]].itemsize
        streams = {"add": 4, "first": 3, "plain": 2}[case["mode"]]
        return {"bytes": (streams * case["tokens"] + 1) * case["H"] * size, "flops": 0}
    if kind == "quant":
        T, H = case["tokens"], case["H"]
        streams = 6 if case["residual"] else 2
        return {"bytes": (streams + 1) * T * H + 2 * H + (0 if case["mode"] == "static_fp8" else 4 * T), "flops": 0}
    if kind == "linear":
        n_bytes, flops = _gemm_work(case["M"], case["N"], case["K"])
        return {"bytes": n_bytes + (case["N"] * 2 if case["bias"] else 0), "flops": flops}
    if kind == "producer":
        n_bytes, flops = _gemm_work(case["M"], case["N"], case["K"])
        return {"bytes": case["P"] * n_bytes, "flops": case["P"] * flops}
    # A layer: two projections and two norms.  This rank's partial sum is written by a projection
    # and read by the norm behind it: not counted.  The other ranks' sums are new before each norm.
    H, P, k_attn, k_mlp, _ = MODELS[case["model"]]
    T = case["tokens"]
    rows = T if T >= WEAVE_TOKENS else T // P
    n_bytes = sum((T * k + H * k) * 2 for k in (k_attn, k_mlp)) + 2 * ((P - 1 + 3) * rows + 1) * H * 2
    return {"bytes": n_bytes, "flops": 2.0 * T * H * (k_attn + k_mlp)}


def tolerance(case):
    """16-bit results of fp32 sums in another order: most values the same, the rest one rounding
    step (2^-7 of the value in bf16) apart.  fp8 codes: a step is an eighth of the value."""
    kind = case["kind"]
    if kind == "quant":
        if case["mode"] == "dyn_int8":
            return {"rel": 5e-3, "max": 2e-2, "differ": 5e-3}
        return {"rel": 1e-2, "max": 0.13}
    if case.get("dtype") == "fp32":
        return {"rel": 1e-5, "max": 1e-4}
    if kind == "layer":
        return {"rel": 1e-2, "max": 4e-2}
    return {"rel": 5e-3, "max": 2e-2}
