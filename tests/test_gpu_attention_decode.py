"""The one-operator decode step of attention (pllm_attention_decode through attention_decode_forward) against a float64
statement of the same arithmetic (reference: src/models/minimax_m2/architecture.py:158-266 for one query position): RMS
normalisation of q and k over their whole width, half-split rotary phases, the new row in the stores, grouped-query softmax
attention over positions 0 .. pos.  Tolerance: rel-L2 <= 3e-3 in fp16 and <= 1.5e-2 in bf16 (the operator rounds the normalized
and the turned values and its output to the 16-bit type; the statement does not)."""
import numpy as np
import pytest
import torch

from pocketllm_amd.attention_core import RotaryTable
from pocketllm_amd.cuda_loader import load_cuda_kernel

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _statement(q, k_new, v_new, keys, values, pos, heads, kv_heads, qw, kw, eps, cos, sin, rope_dim):
    """float64 on the CPU; keys / values [batch, kv_heads, >= pos, 128] hold positions 0 .. pos - 1."""
    q, k_new, v_new, keys, values = (t.double().cpu() for t in (q, k_new, v_new, keys, values))
    batch, dim = q.size(0), 128
    half = rope_dim // 2

    def norm(x, w):
        return x if w is None else x * torch.rsqrt((x * x).mean(dim=-1, keepdim=True) + eps) * w.double().cpu()

    def turn(x):                                  # [batch, heads, 128]
        if rope_dim == 0:
            return x
        partner = torch.cat((x[..., half:2 * half], x[..., :half], x[..., 2 * half:]), dim=-1)
        return x * cos.double().cpu() + partner * sin.double().cpu()

    qh = turn(norm(q, qw).view(batch, heads, dim))
    kh = turn(norm(k_new, kw).view(batch, kv_heads, dim))
    all_k = torch.cat((keys[:batch, :, :pos], kh.unsqueeze(2)), dim=2)              # [batch, kv_heads, pos + 1, 128]
    all_v = torch.cat((values[:batch, :, :pos], v_new.view(batch, kv_heads, 1, dim)), dim=2)
    group = heads // kv_heads
    qg = qh.view(batch, kv_heads, group, dim)
    scores = torch.einsum("bkgd,bkld->bkgl", qg, all_k) / np.sqrt(dim)
    out = torch.einsum("bkgl,bkld->bkgd", torch.softmax(scores, dim=-1), all_v)
    return out.reshape(batch, heads * dim), kh


@pytest.mark.parametrize("dtype,tol", [(torch.float16, 3e-3), (torch.bfloat16, 1.5e-2)])
def test_decode_step_matches_the_float64_statement(dtype, tol):
    mod = load_cuda_kernel()
    assert mod is not None and torch.cuda.is_available()
    gen = torch.Generator(device="cpu").manual_seed(11)
    cases = (  # heads, kv_heads, rope_dim, batch, positions, norm weights
        (48, 8, 64, 1, (0, 5, 63, 64, 65, 700, 2047), True),
        (16, 2, 128, 2, (1, 64, 130), True),
        (8, 8, 0, 3, (3, 127, 128), False),
        (12, 4, 32, 1, (255, 256), True),
    )
    for heads, kv_heads, rope_dim, batch, positions, with_norm in cases:
        capacity = max(positions) + 1
        table = RotaryTable(rope_dim, 1.0e4, torch.device(DEV), head_dim=128, positions=capacity)
        qw = (torch.rand(heads * 128, generator=gen) + 0.5).to(DEV) if with_norm else None
        kw = (torch.rand(kv_heads * 128, generator=gen) + 0.5).to(DEV) if with_norm else None
        for pos in positions:
            keys = (torch.randn(batch + 1, kv_heads, capacity, 128, generator=gen) * 0.7).to(DEV).to(dtype)
            values = torch.randn(batch + 1, kv_heads, capacity, 128, generator=gen).to(DEV).to(dtype)
            q = (torch.randn(batch, heads * 128, generator=gen) * 2.0).to(DEV).to(dtype)
            k_new = torch.randn(batch, kv_heads * 128, generator=gen).to(DEV).to(dtype)
            v_new = torch.randn(batch, kv_heads * 128, generator=gen).to(DEV).to(dtype)
            cos, sin = table.rows(pos)
            want, want_k = _statement(q, k_new, v_new, keys, values, pos, heads, kv_heads, qw, kw, 1e-6, cos, sin, rope_dim)
            keys_before, values_before = keys.clone(), values.clone()
            print(f"case attention decode {dtype} heads={heads}/{kv_heads} rope={rope_dim} batch={batch} pos={pos}", flush=True)
            got = mod.attention_decode_forward(q, k_new, v_new, keys, values, pos, q_norm_weight=qw, k_norm_weight=kw, eps=1e-6,
                                               cos_row=cos, sin_row=sin, rope_dim=rope_dim)
            torch.cuda.synchronize()
            assert got.shape == (batch, heads * 128) and got.dtype == dtype
            err = (got.double().cpu() - want).norm() / want.norm()
            assert err <= tol, f"rel-L2 {err:.3e}"
            # the stores: position pos of the first `batch` sequences holds the new rows, nothing else moved
            new_k = keys[:batch, :, pos].double().cpu()
            assert (new_k - want_k).norm() / want_k.norm() <= tol
            assert torch.equal(values[:batch, :, pos], v_new.view(batch, kv_heads, 128))
            keys_before[:batch, :, pos] = keys[:batch, :, pos]
            values_before[:batch, :, pos] = values[:batch, :, pos]
            assert torch.equal(keys, keys_before) and torch.equal(values, values_before)


def test_decode_step_rejects_what_it_does_not_take():
    mod = load_cuda_kernel()
    keys = torch.zeros(1, 2, 8, 64, device=DEV, dtype=torch.float16)       # 64-wide heads
    q = torch.zeros(1, 4 * 64, device=DEV, dtype=torch.float16)
    kv = torch.zeros(1, 2 * 64, device=DEV, dtype=torch.float16)
    with pytest.raises(RuntimeError):
        mod.attention_decode_forward(q, kv, kv, keys, keys.clone(), 0)
    keys = torch.zeros(1, 1, 8, 128, device=DEV, dtype=torch.float16)      # sixteen query heads on one key/value head
    q = torch.zeros(1, 16 * 128, device=DEV, dtype=torch.float16)
    kv = torch.zeros(1, 128, device=DEV, dtype=torch.float16)
    with pytest.raises(RuntimeError):
        mod.attention_decode_forward(q, kv, kv, keys, keys.clone(), 0)
    with pytest.raises(RuntimeError):                                      # position outside the stores
        mod.attention_decode_forward(torch.zeros(1, 128, device=DEV, dtype=torch.float16), kv, kv, keys, keys.clone(), 8)


@pytest.mark.parametrize("dtype,step,tol", [(torch.float16, 2.0 ** -10, 3e-3), (torch.bfloat16, 2.0 ** -7, 1.5e-2)])
@pytest.mark.parametrize("heads,kv_heads,batch,pos", [
    (48, 8, 5, 447),          # seven runs of one slice of 64 keys, two to a workgroup; the new key the last of its slice
    (48, 8, 5, 448),          # ... the only one of its slice
    (64, 8, 11, 200),         # two workgroups of two runs
    (32, 32, 1, 700),         # one query head per key/value head, runs of two slices, the last of one
    (8, 2, 34, 1024),         # two workgroups per compute unit, of three runs, the last of two
    (10, 2, 600, 65)])        # five query heads, more rows than places: both runs of a row in one workgroup
def test_several_slices_in_one_workgroup(heads, kv_heads, batch, pos, dtype, step, tol):
    """Rows of a batch that is large enough for workgroups to walk over several slices, against the statement in float64 and against the same rows
    called alone: at most one step of their type apart (the same bits since the runs of slices go by one sequence)."""
    mod = load_cuda_kernel()
    gen = torch.Generator(device="cpu").manual_seed(heads + batch + pos)
    table = RotaryTable(64, 1.0e4, torch.device(DEV), head_dim=128, positions=pos + 1)
    qw, kw = ((torch.rand(h * 128, generator=gen) + 0.5).to(DEV) for h in (heads, kv_heads))
    rows = min(batch, 3)                                        # (rows repeat with this period)
    draw = lambda size, *shape: (torch.randn(rows, *shape, generator=gen) * size).to(dtype).repeat(-(-batch // rows), *[1] * len(shape))[:batch].to(DEV)
    keys, values = draw(0.7, kv_heads, pos + 1, 128), draw(1.0, kv_heads, pos + 1, 128)
    keys[:, :, pos:], values[:, :, pos:] = float("nan"), float("nan")      # (the new position's row is written by the call)
    q, k_new, v_new = draw(2.0, heads * 128), draw(1.0, kv_heads * 128), draw(1.0, kv_heads * 128)
    cos, sin = table.rows(pos)
    run = lambda s: mod.attention_decode_forward(q[s].contiguous(), k_new[s].contiguous(), v_new[s].contiguous(), keys[s].contiguous(), values[s].contiguous(), pos,
                                                 q_norm_weight=qw, k_norm_weight=kw, eps=1e-6, cos_row=cos, sin_row=sin, rope_dim=64)
    print(f"case attention decode slices {dtype} heads={heads}/{kv_heads} batch={batch} pos={pos}", flush=True)
    got = run(slice(None))
    torch.cuda.synchronize()
    few = [t[:rows] for t in (q, k_new, v_new, keys, values)]
    want, _ = _statement(*few, pos, heads, kv_heads, qw, kw, 1e-6, cos, sin, 64)
    assert (got[:rows].double().cpu() - want).norm() / want.norm() <= tol
    assert torch.equal(got, got[:rows].repeat(-(-batch // rows), 1)[:batch])
    for r in range(rows):
        alone, row = run(slice(r, r + 1)).float(), got[r:r + 1].float()
        assert ((alone - row).abs() <= step * torch.maximum(alone.abs(), row.abs()) + 2.0 ** -24).all()


@pytest.mark.parametrize("dtype,tol", [(torch.float16, 3e-3), (torch.bfloat16, 1.5e-2)])
@pytest.mark.parametrize("heads,kv_heads,batch,pos", [
    (48, 8, 5, 448),          # eight runs of one slice of 64 keys, two to a workgroup
    (64, 8, 11, 200),         # two workgroups of two runs
    (8, 8, 3, 5000),          # runs of three slices, the last of one, three runs to a workgroup
    (16, 16, 2, 1500),        # one query head per key/value head: runs of one slice where runs of two would leave compute units idle
    (16, 8, 1, 3100),         # ... of two, as there would be more than the merge takes at a time
    (8, 2, 34, 1024),         # two workgroups per compute unit, of three runs, the last of two
    (10, 2, 600, 65)])        # more rows than places: both runs of a row in one workgroup
def test_a_sequence_alone_and_in_a_batch(heads, kv_heads, batch, pos, dtype, tol):
    """A sequence's outputs are the same bits alone and in any batch (the runs of slices that are added up one after the other go by one sequence),
    and within the tolerance of the other sizes of the statement in float64."""
    mod = load_cuda_kernel()
    gen = torch.Generator(device="cpu").manual_seed(heads + batch + pos)
    rows = min(batch, 3)                                        # (rows repeat with this period)
    draw = lambda size, *shape: (torch.randn(rows, *shape, generator=gen) * size).to(dtype).repeat(-(-batch // rows), *[1] * len(shape))[:batch].to(DEV)
    args = [draw(1.0, heads * 128), draw(1.0, kv_heads * 128), draw(1.0, kv_heads * 128), draw(0.7, kv_heads, pos + 1, 128), draw(1.0, kv_heads, pos + 1, 128)]
    few = [t[:rows].clone() for t in args]
    print(f"case attention decode alone {dtype} heads={heads}/{kv_heads} batch={batch} pos={pos}", flush=True)
    got = mod.attention_decode_forward(*args, pos)
    torch.cuda.synchronize()
    want, _ = _statement(*few, pos, heads, kv_heads, None, None, 1e-6, None, None, 0)
    assert (got[:rows].double().cpu() - want).norm() / want.norm() <= tol
    for r in range(rows):
        assert torch.equal(mod.attention_decode_forward(*(t[r:r + 1].contiguous() for t in few), pos), got[r:r + 1])


@pytest.mark.parametrize("sign", [-1.0, 1.0])
@pytest.mark.parametrize("pos", [40, 300, 9000])              # one slice, runs of one, runs of two
@pytest.mark.parametrize("dtype,size,tol", [(torch.bfloat16, 1.0e16, 1.5e-2), (torch.bfloat16, 1.8e18, 1.5e-2), (torch.float16, 1.3e4, 3e-3)])
def test_decode_step_with_very_large_scores(dtype, size, tol, pos, sign):
    """Scores of up to 2e38 in magnitude, above and below zero, in every other head, whose dot products pass the largest float before they are scaled (1.8e18),
    beside heads of ordinary scores: one key of each sequence is the largest by half, so such a head's weights are one and zeros, whatever the rounding."""
    mod = load_cuda_kernel()
    gen = torch.Generator(device="cpu").manual_seed(pos)
    heads, kv_heads, batch = 8, 2, 3
    unit = (1.0 + torch.arange(128) / 128.0) * torch.where(torch.rand(128, generator=gen) < 0.5, -1.0, 1.0)
    rows = torch.where(torch.arange(heads) % 2 == 0, torch.tensor(size, dtype=torch.float64), torch.tensor(0.04 / size, dtype=torch.float64))
    factor = torch.full((batch, pos + 1), 1.0 if sign > 0 else 2.0)
    for b, at in enumerate((pos, pos - 1, pos // 2)):                      # the new key, one of its slice, one further back
        factor[b, at] = 3.0 - factor[b, at]
    q = (unit * rows[:, None]).reshape(1, -1).expand(batch, -1).to(dtype).contiguous().to(DEV)
    keys = (sign * size * unit * factor[:, None, :, None]).expand(batch, kv_heads, pos + 1, 128).to(dtype).contiguous().to(DEV)
    k_new = keys[:, :, pos].reshape(batch, -1).clone()
    keys[:, :, pos] = float("nan")                                         # (written by the call)
    values = torch.randn(batch, kv_heads, pos + 1, 128, generator=gen).to(DEV).to(dtype)
    v_new = torch.randn(batch, kv_heads * 128, generator=gen).to(DEV).to(dtype)
    want, _ = _statement(q, k_new, v_new, keys, values, pos, heads, kv_heads, None, None, 1e-6, None, None, 0)
    print(f"case attention decode large scores {dtype} {size} pos={pos} sign={sign}", flush=True)
    got = mod.attention_decode_forward(q, k_new, v_new, keys, values, pos)
    torch.cuda.synchronize()
    err = (got.double().cpu() - want).view(batch, heads, 128).norm(dim=-1) / want.view(batch, heads, 128).norm(dim=-1)
    assert err.max() <= tol, err
