"""Attention of several new positions (pllm_attention_prompt through attention_prompt_forward) against a float64 statement of the same
arithmetic (reference: src/models/minimax_m2/architecture.py:158-266): RMS normalisation of q and k over their whole width, half-split
rotary phases, the new rows in the stores, causal grouped-query softmax attention.  Tolerance, rel-L2 of a query's output: the turned
queries and keys are rounded to 16 bits twice (relative 2^-12 in fp16, 2^-9 in bf16, independent over 128 products of a score of about
unit variance), the softmax weights and the output once more: 2e-3 and 1.5e-2."""
import numpy as np
import pytest
import torch

from pocketllm_amd.attention_core import RotaryTable
from pocketllm_amd.cuda_loader import load_cuda_kernel

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _statement(q, k, v, keys, values, first, heads, kv_heads, qw, kw, eps, cos, sin, rope_dim):
    q, k, v, keys, values = (t.double().cpu() for t in (q, k, v, keys, values))
    batch, steps = q.shape[:2]
    half = rope_dim // 2

    def norm(x, w):
        return x if w is None else x * torch.rsqrt((x * x).mean(dim=-1, keepdim=True) + eps) * w.double().cpu()

    def turn(x):                                  # [batch, steps, heads, 128]
        if rope_dim == 0:
            return x
        partner = torch.cat((x[..., half:2 * half], x[..., :half], x[..., 2 * half:]), dim=-1)
        return x * cos.double().cpu()[None, :, None] + partner * sin.double().cpu()[None, :, None]

    qh = turn(norm(q, qw).view(batch, steps, heads, 128))
    kh = turn(norm(k, kw).view(batch, steps, kv_heads, 128)).permute(0, 2, 1, 3)
    all_k = torch.cat((keys[:batch, :, :first], kh), dim=2)
    all_v = torch.cat((values[:batch, :, :first], v.view(batch, steps, kv_heads, 128).permute(0, 2, 1, 3)), dim=2)
    group = heads // kv_heads
    seen = torch.arange(first + steps)[None, :] <= first + torch.arange(steps)[:, None]
    out = torch.empty(batch, steps, heads, 128, dtype=torch.float64)
    for h in range(heads):
        scores = qh[:, :, h] @ all_k[:, h // group].transpose(1, 2).contiguous() / np.sqrt(128)
        out[:, :, h] = torch.softmax(scores.masked_fill(~seen, float("-inf")), dim=-1) @ all_v[:, h // group]
    return out.reshape(batch, steps, heads * 128), kh


@pytest.mark.parametrize("heads,kv_heads,rope_dim,batch,steps,first,normed", [
    (48, 8, 64, 1, 2, 0, True), (48, 8, 64, 1, 127, 1, True), (6, 2, 128, 2, 128, 0, True), (8, 8, 0, 1, 129, 63, False), (6, 1, 32, 3, 33, 300, True),
    (8, 1, 64, 1, 300, 0, True), (64, 32, 64, 1, 65, 0, False), (4, 2, 20, 1, 40, 0, True)])
@pytest.mark.parametrize("dtype,new_dtype,tol", [(torch.float16, torch.float16, 2e-3), (torch.bfloat16, torch.bfloat16, 1.5e-2),
                                                 (torch.float16, torch.bfloat16, 2e-3)])
def test_prompt_matches_the_float64_statement(heads, kv_heads, rope_dim, batch, steps, first, normed, dtype, new_dtype, tol):
    mod = load_cuda_kernel()
    assert mod is not None and torch.cuda.is_available()
    gen = torch.Generator(device="cpu").manual_seed(steps + first)
    capacity = first + steps + 5
    table = RotaryTable(rope_dim, 1.0e4, torch.device(DEV), head_dim=128, positions=capacity)
    cos, sin = table.span(first, steps)
    qw = (torch.rand(heads * 128, generator=gen) + 0.5).to(DEV) if normed else None
    kw = (torch.rand(kv_heads * 128, generator=gen) + 0.5).to(DEV) if normed else None
    keys, values = ((torch.randn(batch + 1, kv_heads, capacity, 128, generator=gen)).to(DEV).to(dtype) for _ in range(2))
    values[:, :, first + steps:] = float("nan")              # behind the last position: never used
    keys[:, :, first + steps:] = float("nan")
    q = torch.randn(batch, steps, heads * 128, generator=gen).to(DEV).to(new_dtype)
    k, v = (torch.randn(batch, steps, kv_heads * 128, generator=gen).to(DEV).to(new_dtype) for _ in range(2))
    want, want_k = _statement(q, k, v, keys, values, first, heads, kv_heads, qw, kw, 1e-6, cos, sin, rope_dim)
    before = keys.clone(), values.clone()
    print(f"case attention prompt heads={heads}/{kv_heads} batch={batch} steps={steps} first={first} {new_dtype} {dtype}", flush=True)
    got = mod.attention_prompt_forward(q, k, v, keys, values, first, q_norm_weight=qw, k_norm_weight=kw, eps=1e-6, cos_rows=cos, sin_rows=sin,
                                       rope_dim=rope_dim)
    torch.cuda.synchronize()
    got = got.double().cpu()
    err = (got - want).norm(dim=-1) / want.norm(dim=-1)
    assert err.max() <= tol, (err.max(), err.argmax())
    new = slice(first, first + steps)
    assert torch.equal(values[:batch, :, new], v.view(batch, steps, kv_heads, 128).permute(0, 2, 1, 3).to(dtype))
    assert ((keys[:batch, :, new].double().cpu() - want_k).norm() / want_k.norm()) <= tol / 2
    for store, old in zip((keys, values), before):           # nothing else in the stores has changed
        store[:batch, :, new] = 0
        old[:batch, :, new] = 0
        assert torch.equal(store.view(torch.int16), old.view(torch.int16))
    # another head dimension: declined, not refused
    small = torch.zeros(1, 1, 4, 64, dtype=dtype, device=DEV)
    row = torch.zeros(1, 2, 64, dtype=dtype, device=DEV)
    assert mod.attention_prompt_forward(row, row, row, small, small.clone(), 0) is None


@pytest.mark.parametrize("sign", [-1.0, 1.0])
@pytest.mark.parametrize("first", [0, 70])
@pytest.mark.parametrize("dtype,size,small,tol", [(torch.bfloat16, 1.0e16, 1.0e-16, 1.5e-2), (torch.float16, 1.3e4, 2.0e-5, 2e-3)])
def test_prompt_with_very_large_scores(dtype, size, small, tol, first, sign):
    """Scores up to 1e34 in magnitude (below and above zero) beside ordinary ones: the weights of a query with such scores are one and zeros.  The keys'
    factors lie 1 / 64 apart, so no rounding of a score changes which is largest."""
    mod = load_cuda_kernel()
    gen = torch.Generator(device="cpu").manual_seed(3)
    heads, kv_heads, steps = 4, 2, 64
    unit = (1.0 + torch.arange(128) / 128.0) * torch.where(torch.rand(128, generator=gen) < 0.5, -1.0, 1.0)
    factor = lambda n: 1.0 + torch.randperm(64, generator=gen)[torch.arange(n) % 64] / 64.0
    rows = torch.where(torch.arange(steps) % 2 == 0, torch.tensor(size, dtype=torch.float64), torch.tensor(small, dtype=torch.float64))
    q = (unit[None, None, None, :] * rows[None, :, None, None]).expand(1, steps, heads, 128).reshape(1, steps, -1).to(dtype).to(DEV)
    k = (sign * size * unit[None, None, None, :] * factor(steps)[None, :, None, None]).expand(1, steps, kv_heads, 128).reshape(1, steps, -1).to(dtype).to(DEV)
    v = torch.randn(1, steps, kv_heads * 128, generator=gen).to(DEV).to(dtype)
    keys, values = (torch.randn(1, kv_heads, first + steps, 128, generator=gen).to(DEV).to(dtype) for _ in range(2))
    keys[:, :, :first] = (sign * size * unit * 0.5).to(dtype).to(DEV) if sign > 0 else (sign * size * unit * 2.5).to(dtype).to(DEV)     # never the largest
    want, _ = _statement(q, k, v, keys, values, first, heads, kv_heads, None, None, 1e-6, None, None, 0)
    print(f"case attention prompt large scores {dtype} first={first} sign={sign}", flush=True)
    got = mod.attention_prompt_forward(q, k, v, keys, values, first)
    torch.cuda.synchronize()
    err = (got.double().cpu() - want).norm(dim=-1) / want.norm(dim=-1)
    assert err.max() <= tol, (err.max(), err.argmax())


@pytest.mark.parametrize("heads,kv_heads,batch,steps,first", [
    (8, 2, 1, 192, 0), (8, 2, 1, 193, 0),             # three and four tiles of 64 keys
    (8, 8, 1, 40, 217), (6, 1, 1, 130, 1000),         # five tiles of one block; two blocks behind a long past
    (16, 4, 17, 66, 574), (16, 4, 17, 66, 510)])      # 272 blocks of ten tiles and of nine, more than compute units
@pytest.mark.parametrize("dtype,tol", [(torch.float16, 2e-3), (torch.bfloat16, 1.5e-2)])
def test_two_groups_of_waves_share_a_blocks_keys(heads, kv_heads, batch, steps, first, dtype, tol):
    """Both sides of the lines from which a form with two groups of waves took the tiles of a query block in turn (one group takes them all now), against the
    statement in float64; the tolerance of the other sizes: the weights of the values are rounded as there."""
    mod = load_cuda_kernel()
    gen = torch.Generator(device="cpu").manual_seed(heads + steps + first)
    rows = min(batch, 2)
    draw = lambda *shape: torch.randn(rows, *shape, generator=gen).to(dtype).repeat(-(-batch // rows), *[1] * len(shape))[:batch].to(DEV)
    keys, values = draw(kv_heads, first + steps, 128), draw(kv_heads, first + steps, 128)
    q, k, v = draw(steps, heads * 128), draw(steps, kv_heads * 128), draw(steps, kv_heads * 128)
    few = [t[:rows].clone() for t in (q, k, v, keys, values)]
    print(f"case attention prompt groups heads={heads}/{kv_heads} batch={batch} steps={steps} first={first} {dtype}", flush=True)
    got = mod.attention_prompt_forward(q, k, v, keys, values, first)
    torch.cuda.synchronize()
    want, _ = _statement(*few, first, heads, kv_heads, None, None, 0.0, None, None, 0)
    err = (got[:rows].double().cpu() - want).norm(dim=-1) / want.norm(dim=-1)
    assert err.max() <= tol, (err.max(), err.argmax())
    assert torch.equal(got, got[:rows].repeat(-(-batch // rows), 1, 1)[:batch])


@pytest.mark.parametrize("sign", [-1.0, 1.0])
@pytest.mark.parametrize("dtype,size,small,tol", [(torch.bfloat16, 1.0e16, 1.0e-16, 1.5e-2), (torch.float16, 1.3e4, 2.0e-5, 2e-3)])
def test_prompt_with_very_large_scores_over_five_tiles(dtype, size, small, tol, sign):
    test_prompt_with_very_large_scores(dtype, size, small, tol, 200, sign)


@pytest.mark.parametrize("heads,kv_heads,steps,first", [(8, 2, 193, 0), (8, 8, 40, 217), (16, 4, 66, 574), (48, 8, 300, 100)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_a_sequence_alone_and_in_a_batch(heads, kv_heads, steps, first, dtype):
    """A sequence's outputs are the same bits alone and in a batch whose query blocks are more than the compute units."""
    mod = load_cuda_kernel()
    gen = torch.Generator(device="cpu").manual_seed(heads + steps + first)
    batch = 2 * -(-257 // (2 * heads * -(-steps // 128)))
    draw = lambda *shape: torch.randn(2, *shape, generator=gen).to(dtype).repeat(batch // 2, *[1] * len(shape)).to(DEV)
    args = [draw(steps, heads * 128), draw(steps, kv_heads * 128), draw(steps, kv_heads * 128), draw(kv_heads, first + steps, 128), draw(kv_heads, first + steps, 128)]
    few = [t[:2].clone() for t in args]
    print(f"case attention prompt alone heads={heads}/{kv_heads} batch={batch} steps={steps} first={first} {dtype}", flush=True)
    got = mod.attention_prompt_forward(*args, first)
    torch.cuda.synchronize()
    assert torch.equal(got, got[:2].repeat(batch // 2, 1, 1))
    for r in range(2):
        assert torch.equal(mod.attention_prompt_forward(*(t[r:r + 1].contiguous() for t in few), first)[0], got[r])
