"""The attention core of the decoder block (pocketllm_amd/attention_core.py) against a plain numpy statement of half-split rotary
embedding and causal grouped-query attention (what src/models/minimax_m2/architecture.py:197-266 computes).  CPU only."""
import numpy as np
import pytest
import torch

from pocketllm_amd import _ffi
from pocketllm_amd.attention_core import KeyValueCache, RotaryTable, grouped_query_attention


def _rope_np(x, first, rope_dim, base):
    half = rope_dim // 2
    f = np.arange(first, first + x.shape[1])[:, None] * (base ** (-(2.0 * np.arange(half)) / rope_dim))[None, :]
    s, c = np.sin(f)[None, :, None, :], np.cos(f)[None, :, None, :]
    x1, x2 = x[..., :half], x[..., half:rope_dim]
    return np.concatenate([x1 * c - x2 * s, x1 * s + x2 * c, x[..., rope_dim:]], axis=-1)


def test_rotary_table_matches_the_pairwise_rotation_and_grows():
    rng = np.random.default_rng(0)
    x = rng.standard_normal((2, 5, 4, 16))
    table = RotaryTable(8, 10000.0, torch.device("cpu"), head_dim=16, positions=4)
    for first in (0, 3, 700):                # 700 lies beyond the first table: it has to grow
        got = table.rotate(torch.from_numpy(x).float(), first).numpy()
        assert np.abs(got - _rope_np(x, first, 8, 10000.0)).max() < 2e-5
    whole = RotaryTable(16, 5.0e6, torch.device("cpu"))                        # rope_dim == head_dim, no tail
    assert np.abs(whole.rotate(torch.from_numpy(x).float(), 11).numpy() - _rope_np(x, 11, 16, 5.0e6)).max() < 2e-5
    none = RotaryTable(0, 10000.0, torch.device("cpu"), head_dim=16)
    assert none.rotate(torch.from_numpy(x), 5) is not None and torch.equal(none.rotate(torch.from_numpy(x), 5), torch.from_numpy(x))


def test_grouped_query_attention_is_causal_softmax_attention_over_the_store():
    rng = np.random.default_rng(1)
    batch, heads, kv_heads, dim = 2, 4, 2, 16
    cache = KeyValueCache(kv_heads, dim, torch.device("cpu"), torch.float32)
    ks, vs = [], []
    first = 0
    for steps in (3, 5, 1):                  # a prefill, a second chunk at a non-zero position, one decode step (the store grows on the way)
        k, v = rng.standard_normal((batch, steps, kv_heads, dim)), rng.standard_normal((batch, steps, kv_heads, dim))
        q = rng.standard_normal((batch, steps, heads, dim))
        ks.append(k)
        vs.append(v)
        cache.write(torch.from_numpy(k).float(), torch.from_numpy(v).float(), first)
        keys, values = cache.read(batch, first + steps)
        got = grouped_query_attention(torch.from_numpy(q).float(), keys, values, first).numpy()
        all_k, all_v = np.concatenate(ks, axis=1), np.concatenate(vs, axis=1)
        want = np.zeros((batch, steps, heads, dim))
        for b in range(batch):
            for t in range(steps):
                for h in range(heads):
                    kk, vv = all_k[b, :first + t + 1, h // (heads // kv_heads)], all_v[b, :first + t + 1, h // (heads // kv_heads)]
                    s = kk @ q[b, t, h] / np.sqrt(dim)
                    p = np.exp(s - s.max())
                    want[b, t, h] = (p / p.sum()) @ vv
        assert np.abs(got - want.reshape(batch, steps, heads * dim)).max() < 1e-5
        first += steps
    assert cache.keys.size(2) >= first


class _HostOperators:
    """The operators that MiniMaxAttention calls, over one dense matrix per blocks tensor."""

    def __init__(self):
        self.dense = {}
        self.prompt_calls = []

    def gguf_quant_gemm_prefill_forward(self, x, blocks, row_elems, type_id, grid, out_dtype=torch.bfloat16):
        return (x.float() @ self.dense[id(blocks)].t()).to(out_dtype)

    def gguf_quant_gemm_multi_forward(self, x, blocks, row_elems, type_id, grid, *, norm_weight=None, eps=0.0, out_dtype=torch.bfloat16):
        assert norm_weight is None
        return [self.gguf_quant_gemm_prefill_forward(x, b, row_elems, type_id, grid, out_dtype=out_dtype) for b in blocks]

    def attention_prompt_forward(self, q, k, v, *rest, **options):
        self.prompt_calls.append((q.dtype, k.dtype, v.dtype))
        assert q.dtype in (torch.float16, torch.bfloat16) and k.dtype == q.dtype and v.dtype == q.dtype
        return None                          # (no kernel for the shape: the framework's operators run)


class _HostNorm:
    eps = 1e-6

    def __init__(self, out_dtype=torch.float16):
        self.weight, self.out_dtype = None, out_dtype

    def __call__(self, x):
        return torch.nn.functional.rms_norm(x.float(), x.shape[-1:], eps=self.eps).to(self.out_dtype)


def _host_attention(classes, out_dtypes=(torch.float16,) * 3, norm_dtype=torch.float16, o_proj=None, attention_class=None):
    """A MiniMaxAttention of 2 / 1 heads of 128 on the CPU: projections of the given classes and result types over random matrices."""
    from pocketllm_amd.minimax_block import MiniMaxAttention, MiniMaxM2Args
    from pocketllm_amd.quantized_tensor import QuantizedGGUFTensor

    gen = torch.Generator().manual_seed(5)
    ops = _HostOperators()
    args = MiniMaxM2Args(dim=256, n_heads=2, n_kv_heads=1, head_dim=128, rope_dim=64, rope_base=1e4, n_routed_experts=4, top_k=2, moe_inter_dim=256,
                         norm_eps=1e-6)
    lin = []
    for cls, dtype, n in zip(classes, out_dtypes, (256, 128, 128)):
        blocks = torch.zeros((n, 1, 176), dtype=torch.uint8)
        p = cls(QuantizedGGUFTensor.from_blocks(blocks, "q5_k", 256, source_name="p"), out_dtype=dtype)
        p._cuda = ops
        ops.dense[id(p.tensor.blocks)] = torch.randn(n, 256, generator=gen) / 16
        lin.append(p)
    out_weight = torch.randn(256, 256, generator=gen) / 16
    o = o_proj or (lambda h: (h.float() @ out_weight.t()).to(torch.float16))
    attn = (attention_class or MiniMaxAttention)(args, *lin, o, _HostNorm(norm_dtype), _HostNorm(norm_dtype))
    attn._cuda = ops
    return args, attn, ops


needs_library = pytest.mark.skipif(not _ffi.LIB_PATH.exists(), reason="libpllm_hip.so not built")


@needs_library
@pytest.mark.parametrize("steps", [6, 70])
def test_prompts_keep_the_types_and_calls_of_their_modules(steps):
    """Projections return their modules' type at every row count, an output projection is any callable, and a block calls its attention."""
    from pocketllm_amd.minimax_block import MiniMaxAttention, MiniMaxBlock
    from pocketllm_amd.quantized_ops import QuantizedGGUFLinear

    class Twice(QuantizedGGUFLinear):
        def __call__(self, x):
            return 2.0 * super().__call__(x)

    class Marked(MiniMaxAttention):
        def __call__(self, x, start_pos):
            return torch.full_like(super().__call__(x, start_pos), 3.0)

    x = torch.randn(1, steps, 256, generator=torch.Generator().manual_seed(6)).to(torch.float16)
    for classes in ((QuantizedGGUFLinear,) * 3, (QuantizedGGUFLinear, Twice, QuantizedGGUFLinear)):
        for dtypes in ((torch.float16,) * 3, (torch.float32, torch.float16, torch.float16)):
            _, attn, ops = _host_attention(classes, dtypes)
            for got, p in zip(attn.project_qkv(x), (attn.q_proj, attn.k_proj, attn.v_proj)):
                want = x.float() @ ops.dense[id(p.tensor.blocks)].t()
                want = want.to(p.out_dtype) * (2.0 if type(p) is Twice else 1.0)
                assert got.dtype == p.out_dtype and torch.allclose(got.float(), want.float(), rtol=2e-3, atol=1e-3)
            assert attn(x, 0).shape == x.shape
    with pytest.raises(ValueError):                                            # a width that the projections do not take
        attn.project_qkv(x[..., :128])
    args, attn, _ = _host_attention((QuantizedGGUFLinear,) * 3, attention_class=Marked)
    block = MiniMaxBlock(args, torch.ones(256), torch.ones(256), attn, lambda stream, residual, input_norm: residual)
    block.attn_norm = _HostNorm()
    assert torch.equal(block(x, 0), x + 3.0)


@needs_library
def test_prompt_operator_takes_one_16_bit_type_only(monkeypatch):
    """Projections of mixed or 32-bit result types, and normalisations of another type or class, run the framework's operators; the first is
    offered to the prompt operator."""
    from pocketllm_amd import minimax_block
    from pocketllm_amd.quantized_ops import QuantizedGGUFLinear

    class OtherNorm(_HostNorm):
        pass

    monkeypatch.setattr(minimax_block, "RMSNorm", _HostNorm)
    f16, bf16, f32 = torch.float16, torch.bfloat16, torch.float32
    x = torch.randn(1, 6, 256, generator=torch.Generator().manual_seed(6)).to(f16)
    for dtypes, norm_dtype, offered in (((f16,) * 3, f16, 1), ((bf16,) * 3, f16, 1), ((bf16, f16, bf16), f16, 0), ((f32,) * 3, f16, 0),
                                        ((f16, f16, f32), f16, 0), ((f16,) * 3, f32, 0)):
        _, attn, ops = _host_attention((QuantizedGGUFLinear,) * 3, dtypes, norm_dtype)
        want = attn.context(x, 0)
        attn._fused_step = True
        assert torch.equal(attn.context(x, 0), want) and len(ops.prompt_calls) == offered
        attn.k_norm = OtherNorm(norm_dtype)
        assert torch.equal(attn.context(x, 0), want) and len(ops.prompt_calls) == offered
