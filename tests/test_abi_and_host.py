"""CPU-only checks: the C-ABI library loads and exports what include/pllm_hip.h declares, the ctypes
table matches the header, and the host-side helpers (encoders, codebooks, loader contract) behave."""
import ctypes
import re
from pathlib import Path

import numpy as np
import pytest
import torch

from oracle import gguf_oracle as O
from pocketllm_amd import _ffi, block_codec as C, codebooks, cuda_loader, quant_types

ROOT = Path(__file__).resolve().parents[1]
HEADER = (ROOT / "include" / "pllm_hip.h").read_text()


def _declared():
    text = re.sub(r"/\*.*?\*/", "", HEADER, flags=re.S)
    return sorted(set(re.findall(r"\b(pllm_[a-z0-9_]+)\s*\(", text)))


def test_header_and_ctypes_table_agree():
    assert _declared() == sorted(_ffi.SIGNATURES)


def test_every_declaration_cites_the_reference_or_says_it_has_no_counterpart():
    for name in _declared():
        pos = HEADER.index(name + "(")
        comment = HEADER[:pos].rsplit("/*", 1)[-1]
        if name in ("pllm_status_string", "pllm_abi_version") or name.endswith("_workspace_bytes") or name == "pllm_fp8_block_gemm":
            continue        # documented together with their neighbours
        assert ("src/" in comment) or ("cpp_engine/" in comment) or ("no counterpart" in comment), name


@pytest.mark.skipif(not _ffi.LIB_PATH.exists(), reason="libpllm_hip.so not built")
def test_library_exports_every_declared_symbol():
    lib = ctypes.CDLL(str(_ffi.LIB_PATH))
    for name in _declared():
        assert hasattr(lib, name), name
    loaded = _ffi.load_library()
    assert loaded.pllm_abi_version() >= 1
    assert [loaded.pllm_gguf_block_bytes(t) for t in range(5)] == [66, 84, 56, 144, 176]
    assert loaded.pllm_gguf_block_bytes(9) == 0
    assert loaded.pllm_status_string(-4) == b"workspace too small"
    # pure host arithmetic of the ABI
    assert loaded.pllm_gguf_quant_gemm_workspace_bytes(3, 1, 5120, 5120, 20) >= 5120 * 2.5
    assert loaded.pllm_gguf_quant_gemm_workspace_bytes(42, 1, 5120, 5120, 20) == 0
    assert loaded.pllm_gguf_moe_workspace_bytes(1, 8, 3072, 1536) > 8 * 3072 * 4


@pytest.mark.skipif(not _ffi.LIB_PATH.exists(), reason="libpllm_hip.so not built")
def test_rows_beyond_32_bit_offsets_are_left_to_the_row_kernels():
    """The kernels of several activation rows address 64 of them with 32-bit byte offsets: from 2^25 columns on (three Q8_0 rows, five Q2_K
    rows), the workspace is that of the kernels that take row by row."""
    lib = _ffi.load_library()

    def q8_0(rows, blocks):
        return lib.pllm_q8_0_gemm_workspace_bytes(rows, 32 * blocks, 1, blocks)

    def q2_k(rows, blocks):
        return lib.pllm_gguf_quant_gemm_workspace_bytes(1, rows, 256 * blocks, 1, blocks)

    assert q8_0(3, 2**20) > 3 * q8_0(1, 2**20) and q2_k(5, 2**17) * 4 > q2_k(4, 2**17) * 5
    for columns in (2**25 + 256, 38_400_000):
        assert q8_0(3, columns // 32) == 3 * q8_0(1, columns // 32)
        assert q2_k(5, columns // 256) * 4 == q2_k(4, columns // 256) * 5


def _bytes_with_the_height_by_token_count(rows, n, bpr, cus=256):
    """Workspace of a prompt whose tile height follows the token count and the share of the machine the tiles fill: staged fp16 rows, their
    scales, and float32 tiles of the slices that the tiles beyond whole rounds are cut in."""
    cols, low, high = -(-n // 256), -(-rows // 128), -(-rows // 256)
    height = 128 if high * cols * 4 <= cus or (low % 2 and low * cols <= cus) else 256
    left = -(-rows // height) * cols % cus
    slices, best = 1, None
    for s in range(1, min(16, bpr) + 1) if left else ():
        cost = -(-left * s // cus) / s * (8.8 * bpr) + (2.0 * left * s * height * 1024 / 5.0e6 if s > 1 else 0.0)
        if best is None or cost < best - 1e-9:
            slices, best = s, cost
    up = lambda b: (b + 255) // 256 * 256
    return up(rows * bpr * 512) + up(rows * 4) + (left * slices * height * 1024 if slices > 1 else 0)


@pytest.mark.skipif(not _ffi.LIB_PATH.exists() or torch.cuda.is_available(), reason="the library's figures for 256 compute units, which it takes without a device")
def test_prompts_that_the_static_scratch_holds_stay_within_it():
    """Whatever plan a prompt's tiles take, a call that fits the library's own array with the tile height by token count still fits it, in
    every format: the entry without a workspace goes by this figure."""
    lib = _ffi.load_library()
    limit, held = 16 << 20, 0
    named = [(600, 17408, 5120), (1300, 5120, 5120), (320, 16384, 4096), (400, 17408, 3072), (277, 14592, 3584), (1500, 4096, 4096), (1100, 8192, 3072), (900, 8192, 4096)]
    sweep = [(rows, n, k) for rows in range(129, 2048, 61) for n in (1000, 3072, 4096, 6144, 8192, 12288, 14336, 17408) for k in (1024, 3072, 4096, 5120, 8192)]
    for rows, n, k in named + sweep:
        before = _bytes_with_the_height_by_token_count(rows, n, k // 256)
        got = [lib.pllm_gguf_quant_gemm_workspace_bytes(t, rows, k, n, k // 256) for t in range(9)]
        if before <= limit:
            held += 1
            assert max(got) <= limit, (rows, n, k, got)
    assert held > 300
    # a format asks for its own plan: 90 tiles of 128 rows in two slices for Q4_K and FP8 weights, 48 of 256 rows in four for IQ3_XXS and Q6_K
    rows, n, k = 1793, 1336, 3072
    staged = rows * k * 2 + (rows * 4 + 255) // 256 * 256
    got = [lib.pllm_gguf_quant_gemm_workspace_bytes(t, rows, k, n, k // 256) - staged for t in (3, 6, 8)]
    assert got == [90 * 2 * 128 * 1024, 48 * 4 * 256 * 1024, 48 * 4 * 256 * 1024]
    assert lib.pllm_fp8_block_gemm_workspace_bytes(rows, k, n) - staged == 90 * 2 * 128 * 1024
    # the 16 tiles of 128 rows beyond a round: in eleven slices for Q4_K, twelve for FP8 weights, sixteen for Q6_K
    staged = 512 * 5120 * 2 + 512 * 4
    got = [lib.pllm_gguf_quant_gemm_workspace_bytes(t, 512, 5120, 17408, 20) - staged for t in (3, 8)]
    assert got == [16 * 11 * 128 * 1024, 16 * 16 * 128 * 1024]
    assert lib.pllm_fp8_block_gemm_workspace_bytes(512, 5120, 17408) - staged == 16 * 12 * 128 * 1024


@pytest.mark.skipif(not _ffi.LIB_PATH.exists(), reason="libpllm_hip.so not built")
def test_routed_experts_take_no_more_workspace_than_their_tile_matmuls_hold():
    """Several tokens' experts as tile matmuls: fp16 rows and scales of the routes' activations and hidden values, float32 gate, up and down products.
    Callers keep this figure, so what else the products need finds its place inside it."""
    lib = _ffi.load_library()
    up = lambda b: (b + 255) // 256 * 256
    staged = lambda rows, width: up(rows * ((width + 255) // 256) * 512) + up(rows * 4)
    for tokens, routes, dim, inter in [(512, 4096, 2048, 768), (512, 4096, 3072, 1536), (256, 2048, 3072, 1536), (64, 512, 2048, 1408)]:
        tiles = staged(routes, dim) + staged(routes, inter) + 2 * up(routes * inter * 4) + up(routes * dim * 4) + 256
        assert lib.pllm_gguf_moe_workspace_bytes(tokens, routes, dim, inter) == tiles


@pytest.mark.skipif(not _ffi.LIB_PATH.exists(), reason="libpllm_hip.so not built")
def test_native_host_path_declines_tensors_without_memory():
    """The wrapper tensors inside vmap, jvp and grad are torch.Tensor exactly and own no memory: the native functions leave them to the Python
    path, which states the error."""
    from pocketllm_amd import _bindings

    seen = {}

    def note(name):
        def f(x):
            seen[name] = _bindings.dense_tensor(x)
            return (x * x).sum()
        return f

    x = torch.randn(3, 4)
    torch.vmap(note("vmap"))(x)
    torch.func.grad(note("grad"))(x)
    torch.func.jvp(note("jvp"), (x,), (torch.ones_like(x),))
    assert seen == {"vmap": False, "grad": False, "jvp": False}
    assert _bindings.dense_tensor(x) and _bindings.dense_tensor(torch.nn.Parameter(x))
    assert not _bindings.dense_tensor(x.t()) and not _bindings.dense_tensor(x.to_sparse()) and not _bindings.dense_tensor(None)


def test_loader_contract_module_or_none(monkeypatch, tmp_path):
    monkeypatch.setattr(cuda_loader, "_NATIVE_MOD", None)
    monkeypatch.setattr(_ffi, "_LIB", None)
    monkeypatch.setattr(_ffi, "LIB_PATH", tmp_path / "missing.so")
    assert cuda_loader.load_cuda_kernel() is None
    from pocketllm_amd.quantized_ops import Q8_0GGUFLinear
    with pytest.raises(RuntimeError, match="native HIP library is required"):
        Q8_0GGUFLinear(torch.zeros(2, 1, 34, dtype=torch.uint8), 32)
    from pocketllm_amd import ops
    with pytest.raises(RuntimeError, match="no CPU path"):
        ops.q8_0_weight_gemm(torch.zeros(1, 32), torch.zeros(2, 1, 34, dtype=torch.uint8))


def test_operators_without_the_native_host_path(monkeypatch):
    """The extension with the native host path only makes calls cheaper: where it does not load, the operator module says so once and every call takes
    the Python path."""
    import importlib.util
    import sys

    import pocketllm_amd

    monkeypatch.delattr(pocketllm_amd, "_bindings", raising=False)
    monkeypatch.setitem(sys.modules, "pocketllm_amd._bindings", None)
    spec = importlib.util.spec_from_file_location("hip_kernel_alone", _ffi.LIB_PATH.with_name("hip_kernel.py"))
    mod = importlib.util.module_from_spec(spec)
    with pytest.warns(RuntimeWarning, match="_bindings.so is not built or does not load"):
        spec.loader.exec_module(mod)
    x, w1, w2, rw = torch.zeros(1, 512), torch.zeros(2, 4, 2, 144, dtype=torch.uint8), torch.zeros(2, 512, 1, 144, dtype=torch.uint8), torch.ones(1)
    with pytest.raises(RuntimeError, match="x and blocks must be CUDA tensors"):
        mod.gguf_quant_gemm_forward(x, w1[0], 512, 3, torch.empty(0, dtype=torch.int8))
    with pytest.raises(RuntimeError, match="all tensors must be CUDA tensors"):
        mod.q8_0_gemm_forward(x, torch.zeros(4, 16, 34, dtype=torch.uint8), 512)
    with pytest.raises(RuntimeError, match="CUDA"):
        mod.gguf_moe_single_token_accumulate_forward(x, torch.zeros(1, dtype=torch.int64), rw, w1, w1, w2, 0.0, torch.zeros(1, 512))


@pytest.mark.skipif(not _ffi.LIB_PATH.exists(), reason="libpllm_hip.so not built")
def test_operator_names_of_the_reference_extension_exist():
    mod = cuda_loader.load_cuda_kernel()
    for name in ("q8_0_gemm_forward", "gguf_quant_gemm_forward", "gguf_quant_gemm_prefill_forward", "gguf_quant_gemm_pair_forward",
                 "gguf_quant_embedding_forward", "gguf_q2k_gemm_dp4a_forward", "gguf_moe_prefill_grouped_forward",
                 "gguf_moe_single_token_iq2_q2k_forward", "gguf_moe_single_token_iq1m_forward", "moe_group_routes",
                 "gguf_single_token_route_slots"):
        assert hasattr(mod, name), name


@pytest.mark.skipif(not _ffi.LIB_PATH.exists(), reason="libpllm_hip.so not built")
def test_argument_checks_run_before_any_gpu_work():
    mod = cuda_loader.load_cuda_kernel()
    x = torch.zeros(1, 512)
    blocks = torch.zeros(4, 2, 144, dtype=torch.uint8)
    with pytest.raises(RuntimeError, match="x and blocks must be CUDA tensors"):
        mod.gguf_quant_gemm_forward(x, blocks, 512, 3, torch.empty(0, dtype=torch.int8))
    with pytest.raises(RuntimeError, match="all tensors must be CUDA tensors"):
        mod.q8_0_gemm_forward(x, torch.zeros(4, 16, 34, dtype=torch.uint8), 512)


def test_type_table():
    assert quant_types.GGUF_DENSE_TYPE_IDS["q4_k"] == 3 and quant_types.GGUF_DENSE_TYPE_NAMES[2] == "iq1_m"
    assert quant_types.block_bytes_for_type(4) == 176
    with pytest.raises(RuntimeError, match="unsupported GGUF quant type_id"):
        quant_types.block_bytes_for_type(17)


def test_codebooks_agree_with_oracle_copy():
    np.testing.assert_array_equal(codebooks.iq2xxs_signed_grid(), O.iq2xxs_signed_grid())
    np.testing.assert_array_equal(codebooks.iq1_grid(), O.iq1_grid_i8())
    assert tuple(codebooks.get_iq2xxs_signed_grid_tensor().shape) == (256, 128, 8)
    assert codebooks.get_iq1_grid_tensor().dtype == torch.int8
    np.testing.assert_array_equal(codebooks.iq2xs_grid(), O.iq2xs_grid_u8())
    np.testing.assert_array_equal(codebooks.iq3xxs_grid(), O.iq3xxs_grid_u8())
    # the packed tensor for type ids 5 and 6: entry x sign pattern, IQ3_XXS entries doubled under the two sign halves
    packed = codebooks.get_iq2xs_iq3xxs_signed_grid_tensor()
    assert packed.dtype == torch.int8 and packed.numel() == 512 * 128 * 8 + 256 * 128 * 8
    xs, xxs = codebooks.iq2xs_signed_grid(), codebooks.iq3xxs_signed_grid()
    ks = codebooks.ksigns()
    for g, s_ in ((0, 0), (511, 127), (300, 77)):
        sign = np.where((ks[s_] >> np.arange(8)) & 1, -1, 1)
        np.testing.assert_array_equal(xs[g, s_], O.iq2xs_grid_u8()[g].astype(np.int16) * sign)
        np.testing.assert_array_equal(xxs[g % 256, s_], np.tile(O.iq3xxs_grid_u8()[g % 256].astype(np.int16), 2) * sign)
    assert codebooks.grid_tensor_for_type(3).numel() == 0 and codebooks.grid_tensor_for_type(6).numel() == packed.numel()


@pytest.mark.parametrize("name,enc,bits", [("q4_k", C.quantize_q4_k, 4), ("q5_k", C.quantize_q5_k, 5), ("q2_k", C.quantize_q2_k, 2)])
def test_kquant_encoders_round_trip(name, enc, bits):
    rng = np.random.default_rng(3)
    w = (rng.standard_normal((8, 700)) * 0.02).astype(np.float32)       # ragged K: padded with zeros
    blocks = enc(w)
    assert blocks.shape == (8, 3, O.BLOCK_BYTES[name]) and blocks.dtype == np.uint8
    back = O.dequant_rows(blocks, name, 700)
    err = np.abs(back - w).max()
    assert err < 0.1 * 2.0 ** (4 - bits) * 0.02 * 4 + 1e-3, err


def test_q8_0_packer_matches_reference_recipe():
    rng = np.random.default_rng(4)
    w = rng.standard_normal((5, 70)).astype(np.float32)
    blocks = C.pack_q8_0(w)
    assert blocks.shape == (5, 3, 34)
    # the recipe of tests/test_q8_0_cuda.py:12-24, restated with torch
    padded = torch.zeros(5, 96)
    padded[:, :70] = torch.from_numpy(w)
    view = padded.view(5, 3, 32)
    scales = view.abs().amax(dim=2).clamp_min(1e-6) / 127.0
    q = torch.clamp(torch.round(view / scales.unsqueeze(-1)), -127, 127).to(torch.int8)
    np.testing.assert_array_equal(blocks[..., 2:], q.numpy().view(np.uint8))
    np.testing.assert_array_equal(blocks[..., :2], scales.to(torch.float16).view(torch.uint8).view(5, 3, 2).numpy())


def test_fp8_block_encoder():
    rng = np.random.default_rng(5)
    w = (rng.standard_normal((130, 260)) * 0.02).astype(np.float32)
    codes, scale = C.quantize_fp8_block(w)
    assert codes.shape == (130, 260) and scale.shape == (2, 3)
    back = O.dequant_fp8_block(codes, scale)
    assert np.abs(back - w).max() <= np.abs(w).max() / 448 * 16 + 1e-9      # half an ulp at 3 mantissa bits
    assert ((codes & 0x7f) != 0x7f).all()


def test_random_iq_blocks_have_finite_scales():
    rng = np.random.default_rng(6)
    for name, gen in (("iq2_xxs", C.random_iq2_xxs), ("iq1_m", C.random_iq1_m)):
        blocks = gen(rng, 3, 2)
        vals = O.dequant_rows(blocks, name)
        assert np.isfinite(vals).all() and vals.std() > 0


def test_product_never_touches_the_oracle():
    """The oracle is test infrastructure: nothing under the package imports, reads or links it."""
    import pathlib
    root = pathlib.Path(__file__).resolve().parents[1] / "pocketllm_amd"
    for path in list(root.glob("*.py")) + list((root / "csrc").glob("*")):
        if path.is_file() and path.suffix in (".py", ".hip", ".h", ".inc"):
            assert "oracle" not in path.read_text(errors="replace"), path.name
