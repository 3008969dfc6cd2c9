"""The work that a user of this package has it do, as cases that can be timed.

A case is one pass of one linear layer (or norm layer, or mixture-of-experts projection) through the public
operators, the way a serving loop calls them: fresh activations in hand, weights already on the GPU.  `listed()`
names the representative ones, `draw()` gives others of the same ranges, `prepare()` makes what a program holds
before the call, `run()` is the pass, `work()` what the pass cannot do without, `tolerance()` how far another
correct implementation may be from it.
"""
import math

import torch

import flashnn_amd
from flashnn_amd import workloads

DEV = "cuda:0"
_TYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}
EPS = 1e-6


def listed():
    return [
        # the smallest call: one token through an attention projection with int8 weights; latency and host time
        dict(name="w8 1 token", kind="weight_only", bits=8, group=0, m=1, n=4096, k=4096, dtype="fp16", zp=False,
             bias=False),
        # a small decode batch, activations quantised per token, square projection
        dict(name="a8w8 16 tokens", kind="a8w8", m=16, n=4096, k=4096, dtype="fp16", out="fp16"),
        # one token through the wide FFN projection of a large model, int4 weights in groups of 128: the weight stream
        dict(name="w4 1 token", kind="weight_only", bits=4, group=128, m=1, n=28672, k=8192, dtype="bf16", zp=True,
             bias=False),
        # the same layer for a batch of 64 decoding sequences
        dict(name="w4 64 tokens", kind="weight_only", bits=4, group=128, m=64, n=28672, k=8192, dtype="bf16", zp=True,
             bias=False),
        # the same layer for a short prompt
        dict(name="w4 256 tokens", kind="weight_only", bits=4, group=128, m=256, n=28672, k=8192, dtype="bf16", zp=True,
             bias=False),
        # a ragged batch through the FFN-down projection of a model sharded over 8 GPUs: K is 69.5 times 128
        dict(name="a8w8 764 tokens ragged", kind="a8w8", m=764, n=13312, k=8896, dtype="bf16", out="bf16"),
        # prefill of 2048 tokens through a fused QKV projection
        dict(name="a8w8 2048 tokens", kind="a8w8", m=2048, n=12288, k=4096, dtype="fp16", out="bf16"),
        # norm + quantisation + projection of a large prefill, all on the GPU
        dict(name="rmsnorm a8w8 8192 tokens", kind="rms_a8w8", m=8192, n=8192, k=8192, dtype="bf16", out="bf16"),
        # a prompt through the first projection of a mixture of experts, int8; the block size callers take by default
        dict(name="moe a8w8 4096 tokens", kind="moe_a8w8", tokens=4096, experts=8, top_k=2, n=28672, k=4096, block=64,
             dtype="fp16", routed_weight=False),
        # decoding through the same layer with int4 experts in groups of 128: every expert's weights, few rows each
        dict(name="moe a16w4 16 tokens", kind="moe_a16w4", tokens=16, experts=8, top_k=2, n=28672, k=4096, group=128,
             block=16, dtype="bf16", routed_weight=False),
        # a prompt through it: weights decoded once per row block
        dict(name="moe a16w4 1024 tokens", kind="moe_a16w4", tokens=1024, experts=8, top_k=2, n=28672, k=4096, group=128,
             block=64, dtype="bf16", routed_weight=True),
        # a layer norm with quantisation over a prefill, an odd number of rows: memory traffic alone
        dict(name="layernorm quant 4001 rows", kind="norm", op="layernorm_dquant", m=4001, k=8192, dtype="bf16"),
    ]


def _log_int(rng, lo, hi):
    """An integer from lo to hi, even over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


# (N, K) of the linear layers the package is quoted on, and of the sharded decoder layers of its benchmark sweep
_LINEAR = ([(n, k) for k, n in workloads.A8W8_PREFILL_SHAPES.values()] + [(n, k) for k, n in workloads.A16W8_DECODE_SHAPES] +
           [(workloads.A16W4_SHAPE[1], workloads.A16W4_SHAPE[0]), (8192, 8192)] + workloads.sharded_model_gemm_shapes())


def _linear_shape(rng, k_step, n_step):
    """Half the time a layer of the list (where its sizes fit the steps), else a generic one."""
    if rng.random() < 0.5:
        return rng.choice([s for s in _LINEAR if s[0] % n_step == 0 and s[1] % k_step == 0])
    n = _log_int(rng, 1024 // n_step, 32768 // n_step) * n_step
    k = _log_int(rng, 1024 // k_step, 16384 // k_step) * k_step
    return n, k


_MOST_FLOPS = 2 * 8192 ** 3     # of the listed cases' larger ones: what a drawn case costs at most


def draw(rng):
    kind = rng.choice(["a8w8"] * 3 + ["rms_a8w8"] * 2 + ["w8"] * 2 + ["w4"] * 4 + ["packed"] + ["moe_a8w8"] * 2 +
                      ["moe_a16w4"] * 2 + ["norm"] * 2)
    if kind in ("a8w8", "rms_a8w8"):
        n, k = _linear_shape(rng, 32, 16)
        m = _log_int(rng, 1, min(8192, _MOST_FLOPS // (2 * n * k)))
        dtype = rng.choice(["fp16", "bf16"])
        return dict(kind=kind, m=m, n=n, k=k, dtype=dtype, out=dtype if kind == "a8w8" and dtype == "fp16" else "bf16")
    if kind in ("w8", "w4"):
        group = 128 if kind == "w4" or rng.random() < 0.25 else 0
        n, k = _linear_shape(rng, 128, 32)
        m = _log_int(rng, 1, 1024 if n * k <= 1 << 28 else 256)
        return dict(kind="weight_only", bits=8 if kind == "w8" else 4, group=group, m=m, n=n, k=k,
                    dtype=rng.choice(["fp16", "bf16"]), zp=kind == "w4" and rng.random() < 0.75, bias=rng.random() < 0.25)
    if kind == "packed":
        n, k = rng.choice([(28672, 8192), (8192, 8192), (4096, 4096), (12288, 4096), (22016, 4096), (8192, 28672)])
        return dict(kind="packed", m=_log_int(rng, 1, 64), n=n, k=k, dtype=rng.choice(["fp16", "bf16"]),
                    bias=rng.random() < 0.25)
    if kind in ("moe_a8w8", "moe_a16w4"):
        # few large experts or many small ones, as such layers come
        experts, top_k, n, k = rng.choice([(8, 2, 28672, 4096), (8, 2, 4096, 14336), (16, 2, 12288, 4096), (64, 6, 2816, 2048)])
        tokens = _log_int(rng, 1, 4096 if kind == "moe_a8w8" else 2048)
        per_expert = tokens * top_k / experts
        block = 16 if per_expert <= 16 else rng.choice([32, 64]) if per_expert <= 64 else rng.choice([64, 64, 128])
        case = dict(kind=kind, tokens=tokens, experts=experts, top_k=top_k, n=n, k=k, block=block,
                    dtype=rng.choice(["fp16", "bf16"]), routed_weight=rng.random() < 0.5)
        if kind == "moe_a16w4":
            case["group"] = 0 if k > 8192 else rng.choice([0, 128])     # long rows come with one scale per channel
        return case
    return dict(kind="norm", op=rng.choice(["rmsnorm", "layernorm", "layernorm_dquant", "dynamic_quant"]),
                m=_log_int(rng, 1, 8192), k=_log_int(rng, 64, 1112) * 16, dtype=rng.choice(["fp16", "bf16"]))


# ------------------------------------------------------------------------------------------------ inputs


class _Maker:
    """Seeded random tensors on the GPU with the distributions the operators meet."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(int(seed))

    def uniform(self, shape, lo, hi, dtype):
        return torch.empty(shape, dtype=torch.float32, device=DEV).uniform_(lo, hi, generator=self.g).to(dtype)

    def activations(self, m, k, dtype):
        """N(0, 1), one channel of a hundred twenty times as large."""
        x = torch.randn((m, k), dtype=torch.float32, device=DEV, generator=self.g)
        outliers = torch.randperm(k, device=DEV, generator=self.g)[: max(1, k // 100)]
        x[:, outliers] *= 20.0
        return x.to(dtype)

    def int8(self, *shape):
        return torch.randint(-127, 128, shape, dtype=torch.int8, device=DEV, generator=self.g)

    def nibbles(self, *shape):
        """Bytes of two uniform signed nibbles."""
        return torch.randint(-128, 128, shape, dtype=torch.int8, device=DEV, generator=self.g)

    def zero_points(self, shape, dtype):
        """Whole numbers from -8 to 7: uint4 zero points in the operators' signed form."""
        return torch.randint(-8, 8, shape, device=DEV, generator=self.g).to(dtype)


def prepare(case, seed):
    make = _Maker(seed)
    kind, dtype = case["kind"], _TYPES[case["dtype"]]
    st = {"case": case}
    if kind == "norm":
        op = case["op"]
        st["x"] = make.activations(case["m"], case["k"], dtype)
        if op == "dynamic_quant":
            st["op"] = flashnn_amd.DynamicQuantize()
        else:
            cls = {"rmsnorm": flashnn_amd.RMSNorm, "layernorm": flashnn_amd.LayerNorm,
                   "layernorm_dquant": flashnn_amd.LayernormDquant}[op]
            st["op"] = cls(case["k"]).to(device=DEV, dtype=dtype).requires_grad_(False)
            st["op"].weight.copy_(make.uniform((case["k"],), 0.5, 1.5, dtype))
            if op != "rmsnorm":
                st["op"].bias.copy_(make.uniform((case["k"],), -0.5, 0.5, dtype))
    elif kind in ("a8w8", "rms_a8w8"):
        n, k = case["n"], case["k"]
        st["x"] = make.activations(case["m"], k, dtype)
        st["w"] = make.int8(n, k)
        st["ws"] = make.uniform((n,), 1e-3, 1e-2, torch.float32)
        st["gemm"] = flashnn_amd.GemmA8W8(_TYPES[case["out"]])
        if kind == "a8w8":
            st["quant"] = flashnn_amd.DynamicQuantize()
        else:
            st["quant"] = flashnn_amd.RMSNormDquant(k, EPS).to(DEV).requires_grad_(False)
            st["quant"].weight.copy_(make.uniform((k,), 0.5, 1.5, torch.float32))
    elif kind in ("weight_only", "packed"):
        n, k = case["n"], case["k"]
        bits, group = (4, 128) if kind == "packed" else (case["bits"], case["group"])
        tables = (n,) if group == 0 else (k // group, n)
        st["x"] = make.activations(case["m"], k, dtype)
        w = make.int8(n, k) if bits == 8 else make.nibbles(n // 2, k)
        scale = make.uniform(tables, 1e-3, 1e-2, torch.float16)
        zp = make.zero_points(tables, torch.float16) if kind == "packed" or case["zp"] else None
        st["bias"] = make.uniform((n,), -1.0, 1.0, dtype) if case["bias"] else None
        st["gemm"] = flashnn_amd.GemmWeightOnly(dtype)
        if kind == "packed":
            st["packed"] = st["gemm"].prepack(w, scale, zp)
        else:
            st["w"], st["scale"], st["zp"] = w, scale, zp
    else:
        m, e, top_k, n, k = case["tokens"], case["experts"], case["top_k"], case["n"], case["k"]
        scores = torch.randn((m, e), dtype=torch.float32, device=DEV, generator=make.g)
        weights, ids = torch.topk(torch.softmax(scores, -1), top_k, dim=-1)
        st["topk_weights"], st["topk_ids"] = weights.contiguous(), ids.to(torch.int32)
        st["routing"] = [t.to(DEV) for t in workloads.moe_align_block_size(st["topk_ids"].cpu(), case["block"], e)]
        st["x"] = make.activations(m, k, dtype)
        if kind == "moe_a8w8":
            st["w"] = make.int8(e, n, k)
            st["ws"] = make.uniform((e, n), 1e-3, 1e-2, torch.float32)
            st["quant"] = flashnn_amd.DynamicQuantize()
        else:
            tables = (e, n) if case["group"] == 0 else (e, n, k // case["group"])
            st["w"] = make.nibbles(e, n // 2, k)
            st["scale"] = make.uniform(tables, 1e-3, 1e-2, dtype)
            st["zp"] = make.zero_points(tables, dtype)
    return st


# ------------------------------------------------------------------------------------------------ one pass


def run(st):
    case = st["case"]
    kind, x = case["kind"], st["x"]
    if kind == "norm":
        return st["op"](x)
    if kind in ("a8w8", "rms_a8w8"):
        q, s = st["quant"](x)
        return st["gemm"](q, st["w"], s, st["ws"])
    if kind == "weight_only":
        return st["gemm"](x, st["w"], st["scale"], st["bias"], st["zp"])
    if kind == "packed":
        return st["gemm"].forward_prepacked(x, st["packed"], st["bias"])
    sorted_ids, expert_ids, used = st["routing"]
    out = torch.empty((case["tokens"], case["top_k"], case["n"]), dtype=x.dtype, device=x.device)
    if kind == "moe_a8w8":
        q, s = st["quant"](x)
        return flashnn_amd.fused_moe_a8w8_forward(q, st["w"], out, s, st["ws"], st["topk_weights"], st["topk_ids"],
                                                  sorted_ids, expert_ids, used, case["routed_weight"], case["top_k"],
                                                  case["block"])
    return flashnn_amd.fused_moe_a16w4_forward(x, st["w"], out, st["scale"], st["zp"], st["topk_weights"], st["topk_ids"],
                                               sorted_ids, expert_ids, used, case["routed_weight"], case["top_k"],
                                               case["block"])


# ------------------------------------------------------------------------------------------------ what a pass needs


def work(case):
    kind = case["kind"]
    if kind == "norm":
        m, k = case["m"], case["k"]
        to_int8 = case["op"] in ("layernorm_dquant", "dynamic_quant")
        vectors = {"dynamic_quant": 0, "rmsnorm": 1, "layernorm": 2, "layernorm_dquant": 2}[case["op"]]
        return {"bytes": m * k * (3 if to_int8 else 4) + vectors * 2 * k + (2 * m if to_int8 else 0), "flops": 0}
    if kind in ("a8w8", "rms_a8w8"):
        # activations in, weights and their scales in, the product out; the int8 activations need not reach memory
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": 2 * m * k + n * k + 4 * n + 2 * m * n + (4 * k if kind == "rms_a8w8" else 0), "flops": 2 * m * n * k}
    if kind in ("weight_only", "packed"):
        m, n, k = case["m"], case["n"], case["k"]
        bits, group, zp = (4, 128, True) if kind == "packed" else (case["bits"], case["group"], case["zp"])
        tables = n if group == 0 else n * (k // group)
        return {"bytes": n * k * bits // 8 + 2 * tables * (2 if zp else 1) + 2 * m * k + 2 * m * n + (2 * n if case["bias"] else 0),
                "flops": 2 * m * n * k}
    m, e, top_k, n, k = case["tokens"], case["experts"], case["top_k"], case["n"], case["k"]
    used = e * (1.0 - (1.0 - top_k / e) ** m)       # experts that at least one of m evenly routed tokens reaches
    per_expert = n * k + 4 * n if kind == "moe_a8w8" else n * k // 2 + 4 * (n if case["group"] == 0 else n * (k // case["group"]))
    return {"bytes": int(used * per_expert) + 2 * m * k + 2 * m * top_k * n, "flops": 2 * m * top_k * n * k}


def tolerance(case):
    """Against the same formulas in 64 bits, and with fp32 sums taken in another order, the operators measure (relative
    2-norm; most, over the value): int8 products 9e-6 / one last bit in bf16, 3e-6 / one last bit in fp16; behind the fused
    norm 9e-5 / 1.2e-2, where int8 values on a tie flip; weight-only products 9e-5 where scales are applied to fp32 sums and
    8.5e-4 (bf16 out), 3.3e-4 (fp16 out) where every weight is rounded to fp16 as the plain formula does; norms 7e-6 / one
    last bit, 9e-8 of the int8 values.  About four times that is allowed; a last bit is 2^-7 of the value in bf16 at most and
    2^-10 in fp16."""
    kind = case["kind"]
    bf16 = case["dtype"] == "bf16"
    if kind == "norm":
        if case["op"] == "dynamic_quant":
            return "exact"
        few = 2.0 / math.sqrt(case["m"] * case["k"])      # a single last bit, or value, of a small tensor
        return {"rel": 3e-5 + few * (2 ** -8 if bf16 else 2 ** -11), "max": 3e-2 if bf16 else 6e-3, "differ": 1e-6 + few * few}
    if kind in ("a8w8", "moe_a8w8"):
        to_bf16 = (case["out"] if kind == "a8w8" else case["dtype"]) == "bf16"
        return {"rel": 4e-5, "max": 1.6e-2} if to_bf16 else {"rel": 1.2e-5, "max": 2e-3}
    if kind == "rms_a8w8":
        return {"rel": 4e-4, "max": 5e-2}
    return {"rel": 3.5e-3, "max": 3.2e-2} if bf16 else {"rel": 1.3e-3, "max": 8e-3}
