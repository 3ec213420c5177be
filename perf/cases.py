"""What the speed of this framework is measured on: calls of its public modules and operators as a model runtime makes them.

Sizes are those of bench.py, BASELINE.md and the tests: Qwen3-27B-like linears (5120 / 17408), the Q8_0 matrix of 4096 x 4096,
FP8 E4M3 weights with 128 x 128 block scales, MiniMax-M2 layers (hidden 3072, 48 / 8 heads of 128, 256 experts of 1536, top-8).
`draw` spreads over the ranges these stand for: one activation row up to prompts of 2048 tokens, every block format, the three
activation types, matrices from a key / value projection up to an up projection, expert sets of 64 to 256.

Weights carry the code distribution a Gaussian matrix quantizes to (the codebook formats: uniform indices and signs), activations
are N(0, 1).  A state owns its tensors; nothing is shared between states.
"""
from __future__ import annotations

import math

import torch

from pocketllm_amd import codebooks
from pocketllm_amd import ops
from pocketllm_amd.cuda_loader import load_cuda_kernel
from pocketllm_amd.minimax_block import ExpertLayer, MiniMaxAttention, MiniMaxBlock, MiniMaxM2Args, MiniMaxMoE, RMSNorm
from pocketllm_amd.quant_types import GGUF_BLOCK_BYTES, GGUF_DENSE_TYPE_IDS
from pocketllm_amd.quantized_ops import Q8_0GGUFLinear, QuantizedGGUFLinear
from pocketllm_amd.quantized_tensor import QuantizedGGUFTensor

DEV = "cuda:0"
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
DTYPE_BYTES = {"bf16": 2, "f16": 2, "f32": 4}

HIDDEN, HEADS, KV_HEADS, HEAD_DIM = 3072, 48, 8, 128        # a MiniMax-M2 layer
EXPERTS, EXPERT_INTER, TOP_K = 256, 1536, 8


# ---- the cases ---------------------------------------------------------------------------------------------------------

def listed() -> list[dict]:
    return [
        # one token through a Q8_0 projection, float32 activations: the smallest call
        dict(name="q8_0_decode", kind="q8_0", n=4096, k=4096, t=1, dtype="f32"),
        # one token through a query / output projection and through an up projection: what a generated token consists of
        dict(name="q4_k_decode", kind="linear", type="q4_k", n=5120, k=5120, t=1, dtype="bf16"),
        dict(name="q5_k_decode_wide", kind="linear", type="q5_k", n=17408, k=5120, t=1, dtype="bf16"),
        dict(name="fp8_decode_wide", kind="fp8", n=17408, k=5120, t=1, dtype="bf16"),
        # a small batch of sequences (or drafted tokens) through a down projection
        dict(name="q6_k_batch", kind="linear", type="q6_k", n=5120, k=17408, t=7, dtype="f16"),
        # a short prompt through Q8_0, a prompt through an up projection, a long one of odd length through a down projection
        dict(name="q8_0_prompt", kind="q8_0", n=4096, k=4096, t=203, dtype="bf16"),
        dict(name="q4_k_prompt", kind="linear", type="q4_k", n=17408, k=5120, t=512, dtype="bf16"),
        dict(name="q5_k_prompt_long", kind="linear", type="q5_k", n=5120, k=17408, t=1999, dtype="f16"),
        # the FP8 linear with activations quantized to E4M3 as well
        dict(name="fp8_native_prompt", kind="fp8_native", n=17408, k=5120, t=512, dtype="bf16"),
        # the routed experts of one layer for a prompt whose routes are known
        dict(name="experts_prompt", kind="experts", w13="iq2_xxs", w2="iq1_m", experts=EXPERTS, dim=HIDDEN, inter=EXPERT_INTER, top_k=TOP_K, t=256, dtype="bf16"),
        # a whole layer: one generated token against 2047 stored positions, and a prompt
        dict(name="layer_decode", kind="layer", t=1, past=2047),
        dict(name="layer_prompt", kind="layer", t=1024, past=0),
    ]


def _spread(rng, lo: int, hi: int) -> int:
    """An integer of [lo, hi], spread over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _matrix(rng, k_unit: int) -> tuple[int, int]:
    """Rows and columns of a projection: 1024 .. 17408 each, rows of any multiple of 8 with now and then an odd one."""
    n, k = _spread(rng, 1024, 17408), _spread(rng, 1024, 17408)
    n = n if rng.random() < 0.15 else max(8, n // 8 * 8)
    k = max(k_unit, k // k_unit * k_unit)
    while n * k > 17408 * 5120:
        n, k = max(8, n * 3 // 4 // 8 * 8), max(k_unit, k * 3 // 4 // k_unit * k_unit)
    return n, k


def draw(rng) -> dict:
    kind = rng.choices(("linear", "q8_0", "fp8", "fp8_native", "experts", "layer"), weights=(6, 2, 2, 1, 2, 2))[0]
    dtype = rng.choices(("bf16", "f16", "f32"), weights=(5, 3, 2))[0]
    tokens = 1 if rng.random() < 0.3 else _spread(rng, 1, 2048)
    if kind == "linear":
        names = ("q4_k", "q5_k", "q6_k", "q2_k", "iq4_xs", "iq3_xxs", "iq2_xs", "iq2_xxs", "iq1_m")
        n, k = _matrix(rng, 256)
        return dict(kind=kind, type=rng.choices(names, weights=(4, 4, 3, 1, 1, 1, 1, 1, 1))[0], n=n, k=k, t=tokens, dtype=dtype)
    if kind == "q8_0":
        n, k = _matrix(rng, 256 if rng.random() < 0.8 else 64)
        t = tokens if tokens == 1 else _spread(rng, 2, 512)
        while t * n * k > 320 * 4096 * 4096:
            t = max(1, t // 2)
        return dict(kind=kind, n=n, k=k, t=t, dtype=dtype)
    if kind == "fp8":
        n, k = _matrix(rng, 256 if rng.random() < 0.8 else 128)
        tokens = tokens if k % 256 == 0 else min(tokens, 512)
        # float32 activations of few rows keep float32 arithmetic; prompts come in 16-bit types
        return dict(kind=kind, n=n, k=k, t=tokens, dtype=dtype if tokens < 16 else ("bf16" if dtype == "f32" else dtype))
    if kind == "fp8_native":
        n, k = _matrix(rng, 128)
        return dict(kind=kind, n=n, k=k, t=max(2, tokens), dtype="bf16" if dtype == "f32" else dtype)
    if kind == "experts":
        w13, w2 = rng.choices((("iq2_xxs", "iq1_m"), ("q4_k", "q4_k"), ("iq2_xxs", "q2_k"), ("q4_k", "q6_k")), weights=(4, 2, 1, 1))[0]
        experts, dim, inter = rng.choice(((256, 3072, 1536), (128, 2048, 768), (64, 2048, 1408), (128, 3072, 1536)))
        inter = inter // 256 * 256
        return dict(kind=kind, w13=w13, w2=w2, experts=experts, dim=dim, inter=inter, top_k=rng.choice((4, 6, 8)), t=_spread(rng, 1, 1024),
                    dtype="bf16" if dtype == "f32" else dtype)
    if tokens == 1:
        return dict(kind="layer", t=1, past=_spread(rng, 16, 4095))
    return dict(kind="layer", t=_spread(rng, 2, 1024), past=0)


# ---- inputs ------------------------------------------------------------------------------------------------------------

class _Source:
    """Random tensors of one seed on the GPU."""

    def __init__(self, seed: int):
        self.gen = torch.Generator(device=DEV)
        self.gen.manual_seed(int(seed) * 7919 + 17)

    def ints(self, lo: int, hi: int, *shape) -> torch.Tensor:
        return torch.randint(lo, hi, shape, device=DEV, dtype=torch.uint8, generator=self.gen)

    def normal(self, *shape, dtype=torch.float32) -> torch.Tensor:
        return torch.randn(shape, device=DEV, dtype=dtype, generator=self.gen)

    def uniform(self, lo: float, hi: float, *shape) -> torch.Tensor:
        return torch.rand(shape, device=DEV, generator=self.gen) * (hi - lo) + lo

    def codes(self, top: int, *shape) -> torch.Tensor:
        """Unsigned codes 0 .. top as a Gaussian weight quantizes to: centred, the ends about 2.3 standard deviations out."""
        c = self.normal(*shape, dtype=torch.float16)
        return c.mul_(top / 4.6).add_(top / 2.0).round_().clamp_(0, top).to(torch.uint8)


def _half_bytes(v: torch.Tensor) -> torch.Tensor:
    return v.to(torch.float16).unsqueeze(-1).view(torch.uint8)


def _k4_scale_bytes(sc: torch.Tensor, mn: torch.Tensor) -> torch.Tensor:
    """Eight 6-bit scales and minima -> the 12 bytes of a Q4_K / Q5_K block."""
    lo_s, hi_s, lo_m, hi_m = sc[..., :4], sc[..., 4:], mn[..., :4], mn[..., 4:]
    return torch.cat((lo_s | ((hi_s >> 4) << 6), lo_m | ((hi_m >> 4) << 6), (hi_s & 15) | ((hi_m & 15) << 4)), dim=-1)


def _blocks(src: _Source, type_name: str, lead: tuple[int, ...], sigma: float) -> torch.Tensor:
    """Valid blocks [*lead, block bytes] whose weights have a standard deviation of about `sigma`."""
    if type_name in ("q4_k", "q5_k"):
        top = 15 if type_name == "q4_k" else 31
        sc = src.ints(30, 64, *lead, 8)
        mn = (sc.to(torch.int16) + src.ints(0, 9, *lead, 8).to(torch.int16) - 4).clamp_(0, 63).to(torch.uint8)
        d = src.uniform(0.8, 1.2, *lead) * (sigma * 4.6 / top / 47.0)
        head = torch.cat((_half_bytes(d), _half_bytes(d * (top / 2.0)), _k4_scale_bytes(sc, mn)), dim=-1)
        q = src.codes(top, *lead, 8, 32)
        lo, hi = q[..., 0::2, :], q[..., 1::2, :]
        nibbles = ((lo & 15) | ((hi & 15) << 4)).flatten(-2)
        if type_name == "q4_k":
            return torch.cat((head, nibbles), dim=-1).contiguous()
        qh = torch.zeros(*lead, 32, dtype=torch.uint8, device=DEV)
        for g in range(8):
            qh |= (q[..., g, :] >> 4) << g
        return torch.cat((head, qh, nibbles), dim=-1).contiguous()
    if type_name == "q2_k":
        sc = src.ints(7, 16, *lead, 16)
        d = src.uniform(0.8, 1.2, *lead) * (sigma * 1.5 / 11.0)
        q = src.codes(3, *lead, 2, 4, 32)
        packed = (q[..., 0, :] | (q[..., 1, :] << 2) | (q[..., 2, :] << 4) | (q[..., 3, :] << 6)).flatten(-2)
        return torch.cat((sc | (sc << 4), packed, _half_bytes(d), _half_bytes(d * 1.5)), dim=-1).contiguous()
    if type_name == "q6_k":
        q = src.codes(63, *lead, 2, 4, 32)
        ql = torch.cat(((q[..., 0, :] & 15) | ((q[..., 2, :] & 15) << 4), (q[..., 1, :] & 15) | ((q[..., 3, :] & 15) << 4)), dim=-1).flatten(-2)
        qh = ((q[..., 0, :] >> 4) | ((q[..., 1, :] >> 4) << 2) | ((q[..., 2, :] >> 4) << 4) | ((q[..., 3, :] >> 4) << 6)).flatten(-2)
        d = src.uniform(0.8, 1.2, *lead) * (sigma * 4.6 / 63.0 / 95.0)
        return torch.cat((ql, qh, src.ints(64, 128, *lead, 16), _half_bytes(d)), dim=-1).contiguous()
    # the codebook formats: indices, signs and local scales uniform, block scale in a narrow range
    blocks = src.ints(0, 256, *lead, GGUF_BLOCK_BYTES[GGUF_DENSE_TYPE_IDS[type_name]])
    rms = {"iq2_xxs": 59.0, "iq2_xs": 59.0, "iq3_xxs": 130.0, "iq4_xs": 1170.0, "iq1_m": 7.3}[type_name]      # of a weight at d = 1
    d = (src.uniform(0.8, 1.2, *lead) * (sigma / rms)).to(torch.float16)
    if type_name == "iq1_m":                    # the scale's four nibbles sit on top of four 12-bit scale words
        bits = d.view(torch.int16).to(torch.int32)
        for i in range(4):
            blocks[..., 49 + 2 * i] = (blocks[..., 49 + 2 * i] & 15) | (((bits >> (4 * i)) & 15) << 4).to(torch.uint8)
    else:
        blocks[..., 0:2] = _half_bytes(d)
    return blocks


def _q8_0_blocks(src: _Source, n: int, k: int, sigma: float) -> torch.Tensor:
    q = src.normal(n, k // 32, 32, dtype=torch.float16).mul_(127 / 2.5).round_().clamp_(-127, 127).to(torch.int8).view(torch.uint8)
    d = src.uniform(0.8, 1.2, n, k // 32) * (sigma * 2.5 / 127)
    return torch.cat((_half_bytes(d), q), dim=-1).contiguous()


def _fp8_weight(src: _Source, n: int, k: int, sigma: float) -> tuple[torch.Tensor, torch.Tensor]:
    codes = src.normal(n, k, dtype=torch.float16).mul_(448 / 4.5).clamp_(-448, 448).to(torch.float8_e4m3fn)
    return codes, src.uniform(0.8, 1.2, (n + 127) // 128, (k + 127) // 128) * (sigma * 4.5 / 448)


def _linear(src: _Source, type_name: str, n: int, k: int, name: str = "") -> QuantizedGGUFLinear:
    blocks = _blocks(src, type_name, (n, k // 256), k ** -0.5)
    return QuantizedGGUFLinear(QuantizedGGUFTensor.from_blocks(blocks, type_name, k, source_name=name))


def _layer(src: _Source, past: int, steps: int) -> MiniMaxBlock:
    args = MiniMaxM2Args(dim=HIDDEN, n_heads=HEADS, n_kv_heads=KV_HEADS, head_dim=HEAD_DIM, rope_dim=64, rope_base=5.0e6, n_routed_experts=EXPERTS,
                         top_k=TOP_K, moe_inter_dim=EXPERT_INTER, norm_eps=1e-6)
    gamma = lambda width: src.uniform(0.7, 1.3, width)
    attention = MiniMaxAttention(args, _linear(src, "q5_k", HEADS * HEAD_DIM, HIDDEN, "q"), _linear(src, "q5_k", KV_HEADS * HEAD_DIM, HIDDEN, "k"),
                                 _linear(src, "q5_k", KV_HEADS * HEAD_DIM, HIDDEN, "v"), _linear(src, "q5_k", HIDDEN, HEADS * HEAD_DIM, "o"),
                                 RMSNorm(gamma(HEADS * HEAD_DIM), args.norm_eps), RMSNorm(gamma(KV_HEADS * HEAD_DIM), args.norm_eps))
    expert = lambda name, n, k: QuantizedGGUFTensor.from_blocks(_blocks(src, name, (EXPERTS, n, k // 256), k ** -0.5), name, k)
    experts = ExpertLayer(expert("iq2_xxs", EXPERT_INTER, HIDDEN), expert("iq2_xxs", EXPERT_INTER, HIDDEN), expert("iq1_m", HIDDEN, EXPERT_INTER))
    gate = src.normal(EXPERTS, HIDDEN) * (HIDDEN ** -0.5)
    block = MiniMaxBlock(args, gamma(HIDDEN), gamma(HIDDEN), attention, MiniMaxMoE(args, gate, src.normal(EXPERTS) * 0.1, experts))
    block.reset_cache(1, past + steps)
    if past:
        for store in (attention.store.keys, attention.store.values):
            store[:, :, :past] = src.normal(1, KV_HEADS, past, HEAD_DIM, dtype=torch.float16)
    return block


# ---- one pass ----------------------------------------------------------------------------------------------------------

def prepare(case: dict, seed: int) -> dict:
    src, kind = _Source(seed), case["kind"]
    if kind == "layer":
        return dict(case=case, block=_layer(src, case["past"], case["t"]), x=src.normal(1, case["t"], HIDDEN, dtype=torch.float16))
    dtype = DTYPES[case["dtype"]]
    if kind == "experts":
        e, d, i, k13, k2 = case["experts"], case["dim"], case["inter"], case["w13"], case["w2"]
        w1, w3 = (_blocks(src, k13, (e, i, d // 256), d ** -0.5) for _ in range(2))
        w2 = _blocks(src, k2, (e, d, i // 256), i ** -0.5)
        ids = sorted({GGUF_DENSE_TYPE_IDS[k13], GGUF_DENSE_TYPE_IDS[k2]} & {0, 2})
        grids = [codebooks.grid_tensor_for_type(t).to(DEV) for t in ids]
        grid = grids[0] if len(grids) == 1 else (tuple(grids) if grids else torch.empty(0, dtype=torch.int8, device=DEV))
        weights, chosen = torch.softmax(src.normal(case["t"], e), dim=-1).topk(case["top_k"], dim=-1)
        weights = weights / weights.sum(dim=-1, keepdim=True)
        return dict(case=case, w1=w1, w3=w3, w2=w2, grid=grid, chosen=chosen.contiguous(), weights=weights.contiguous(),
                    x=src.normal(case["t"], d, dtype=dtype))
    n, k = case["n"], case["k"]
    x = src.normal(case["t"], k, dtype=dtype)
    if kind == "linear":
        return dict(case=case, layer=_linear(src, case["type"], n, k), x=x)
    if kind == "q8_0":
        return dict(case=case, layer=Q8_0GGUFLinear(_q8_0_blocks(src, n, k, k ** -0.5), k), x=x)
    weight, scale = _fp8_weight(src, n, k, k ** -0.5)
    return dict(case=case, weight=weight, scale=scale, x=x)


def run(state: dict):
    case, x = state["case"], state["x"]
    kind = case["kind"]
    if kind in ("linear", "q8_0"):
        return state["layer"](x)
    if kind == "fp8":
        return ops.soft_fp8_blockfp8_gemm(x, state["weight"], state["scale"])
    if kind == "fp8_native":
        codes, scales = ops.act_quant(x)
        return ops.fp8_gemm(codes, scales, state["weight"], state["scale"])
    if kind == "experts":
        mod = load_cuda_kernel()
        ids = [GGUF_DENSE_TYPE_IDS[case[w]] for w in ("w13", "w2")]
        if case["t"] == 1:
            return mod.gguf_moe_single_token_forward(x, state["chosen"][0], state["weights"][0], state["w1"], state["w3"], state["w2"], 0.0)
        _, tokens, weights, seg = mod.moe_group_routes(state["chosen"], state["weights"], 0, case["experts"])
        return mod.gguf_moe_prefill_grouped_forward(x, tokens, weights, seg, state["w1"], state["w3"], state["w2"], case["dim"], ids[0],
                                                    case["dim"], ids[0], case["inter"], ids[1], state["grid"], 0.0)
    with torch.inference_mode():
        block = state["block"]
        y = block(x, case["past"])
        return y, block.attention.store.keys, block.attention.store.values


# ---- what a pass cannot do without -------------------------------------------------------------------------------------

def _weight_bytes(type_name: str, n: int, k: int) -> float:
    return n * (k / 256) * GGUF_BLOCK_BYTES[GGUF_DENSE_TYPE_IDS[type_name]]


def _experts_work(w13: str, w2: str, experts: int, dim: int, inter: int, top_k: int, t: int) -> tuple[float, float]:
    touched = experts * (1.0 - (1.0 - top_k / experts) ** t)
    return touched * (2 * _weight_bytes(w13, inter, dim) + _weight_bytes(w2, dim, inter)), 2.0 * t * top_k * 3 * dim * inter


def work(case: dict) -> dict:
    kind, t = case["kind"], case["t"]
    if kind == "layer":
        q, kv, length = HEADS * HEAD_DIM, KV_HEADS * HEAD_DIM, case["past"] + t
        w = sum(_weight_bytes("q5_k", n, k) for n, k in ((q, HIDDEN), (kv, HIDDEN), (kv, HIDDEN), (HIDDEN, q))) + 4 * EXPERTS * HIDDEN
        eb, ef = _experts_work("iq2_xxs", "iq1_m", EXPERTS, HIDDEN, EXPERT_INTER, TOP_K, t)
        flops = 2.0 * t * HIDDEN * (2 * q + 2 * kv + EXPERTS) + ef + 4.0 * q * t * (case["past"] + (t + 1) / 2)
        return dict(bytes=w + eb + 4 * t * HIDDEN + 2 * 2 * length * kv, flops=flops)
    if kind == "experts":
        eb, ef = _experts_work(case["w13"], case["w2"], case["experts"], case["dim"], case["inter"], case["top_k"], t)
        return dict(bytes=eb + t * case["dim"] * (DTYPE_BYTES[case["dtype"]] + 4), flops=ef)
    n, k, item = case["n"], case["k"], DTYPE_BYTES[case["dtype"]]
    if kind == "linear":
        weights, out = _weight_bytes(case["type"], n, k), 2
    elif kind == "q8_0":
        weights, out = n * (k / 32) * 34, 2
    else:
        weights, out = n * k + 4 * math.ceil(n / 128) * math.ceil(k / 128), 4
    return dict(bytes=weights + t * (k * item + n * out), flops=2.0 * t * n * k)


def tolerance(case: dict) -> dict:
    """About four times what a float64 restatement of each call shows: 1.7e-3 in 16-bit results; float32 results of FP8 weights
    2.1e-4 where operands are rounded to fp16 and 1e-7 (summation order) below 16 rows; FP8 by FP8 1.4e-5; experts 4.2e-4 (two
    chained products, the hidden values between them at 16 bits or less).  A layer stores fp16 between its operators, and a near
    tie between two experts may fall the other way for a few of its tokens."""
    if case["kind"] == "fp8":
        return {"rel": 1e-3 if case["t"] >= 16 else 1e-5}
    return {"rel": {"linear": 7e-3, "q8_0": 7e-3, "fp8_native": 6e-5, "experts": 2e-3, "layer": 1e-2}[case["kind"]]}
