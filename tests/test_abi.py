"""The C ABI: the shared library loads and exports exactly what include/quarot_hip.h declares.
No kernel is launched here; argument errors are returned before any launch."""
import ctypes
import pathlib
import re

import pytest

from quarot_amd import _lib

ROOT = pathlib.Path(__file__).resolve().parent.parent
HEADER = ROOT / "include" / "quarot_hip.h"


@pytest.fixture(scope="module")
def lib():
    if not _lib.LIB_PATH.exists():          # built beforehand normally; build only if nothing is there
        from quarot_amd import build
        build.build(verbose=False)
    return _lib.lib()


def declared_symbols():
    text = re.sub(r"/\*.*?\*/", "", HEADER.read_text(), flags=re.S)
    return sorted(set(re.findall(r"\b(qr_[a-z0-9_]+)\s*\(", text)))


def test_header_declares_expected_entry_points():
    syms = declared_symbols()
    for must in ("qr_hadamard", "qr_sym_quant_f16_i4", "qr_quantize_rows_f16_i4", "qr_hadamard_quantize_f16_i4",
                 "qr_matmul_i4_i32", "qr_sym_dequant_i32_f16", "qr_linear_i4_f16", "qr_kv_quant_f16_i4",
                 "qr_kv_dequant_i4_f16", "qr_version", "qr_strerror", "qr_rmsnorm_quantize_f16_i4", "qr_heads_hadamard_quantize_f16_i4", "qr_quantized_linear_workspace_bytes", "qr_quantized_linear_f16", "qr_kv_quant_append_batch_decode_f16_i4", "qr_kv_append_f16", "qr_batch_decode_f16",
                 "qr_workspace_bytes", "qr_linear_i4_f16_ws", "qr_linear_i4_f16_static", "qr_f6_bytes", "qr_convert_i4_f6",
                 "qr_linear_f6_f16"):
        assert must in syms


def test_library_exports_every_declared_symbol(lib):
    raw = ctypes.CDLL(str(_lib.LIB_PATH))
    for name in declared_symbols():
        assert hasattr(raw, name), name
    assert sorted(_lib.SIGNATURES) == declared_symbols()


def test_version_and_error_text(lib):
    assert lib.qr_version() >= 100
    assert lib.qr_strerror(0) == b"success"
    for code in (-1, -2, -3, -4, -5, -6, -7):
        assert len(lib.qr_strerror(code)) > 5
    assert b"unknown" in lib.qr_strerror(-99)


def test_argument_errors_are_returned_before_any_launch(lib):
    one = ctypes.c_void_p(16)       # never dereferenced: every call below must fail validation first
    assert lib.qr_matmul_i4_i32(one, one, 4, 4, 100, one, None) == -2          # K % 64 != 0
    assert lib.qr_matmul_i4_i32(one, one, 4, 4, 1 << 18, one, None) == -2      # accumulator would overflow
    assert lib.qr_matmul_i4_i32(None, one, 4, 4, 64, one, None) == -1
    assert lib.qr_matmul_i4_i32(ctypes.c_void_p(8), one, 4, 4, 64, one, None) == -4
    assert lib.qr_matmul_i4_i32(one, one, 0, 4, 64, None, None) == 0           # empty: nothing to do
    assert lib.qr_matmul_i4_i32(one, one, -1, 4, 64, one, None) == -2
    assert lib.qr_linear_i4_f16(one, None, one, one, None, 4, 4, 64, one, None) == -1
    assert lib.qr_sym_quant_f16_i4(None, one, 3, 8, one, None) == -1
    assert lib.qr_sym_quant_f16_i4(one, one, 0, 8, one, None) == 0
    assert lib.qr_quantize_rows_f16_i4(one, 1.0, 3, 0, one, one, None) == -2   # max over an empty axis
    assert lib.qr_sym_dequant_i32_f16(one, one, None, 2, 2, one, None) == -1
    assert lib.qr_hadamard(one, one, 2, 100, 1, None, 0, 1.0, None) == -2      # not a power of two
    assert lib.qr_hadamard(one, one, 2, 172 * 3, 172, one, 0, 1.0, None) == -2
    assert lib.qr_hadamard(one, one, 2, 1 << 16, 1, None, 0, 1.0, None) == -3  # longer than one workgroup's LDS
    assert lib.qr_hadamard(one, one, 2, 64, 1, None, 7, 1.0, None) == -5
    assert lib.qr_hadamard(one, one, 2, 11008, 172, None, 0, 1.0, None) == -1  # hadK missing
    assert lib.qr_hadamard_quantize_f16_i4(one, 2, 64, 1, None, 0, 1.0, 1.0, None, one, None, None) == -1
    assert lib.qr_hadamard_quantize_f16_i4(one, 2, 64, 1, None, 0, 1.0, 1.0, ctypes.c_void_p(20), one, None, None) == -4  # codes: 8-byte aligned
    assert lib.qr_kv_quant_f16_i4(one, 4, 100, 0, one, one, one, None) == -3
    assert lib.qr_kv_quant_f16_i4(one, 4, 128, 3, one, one, one, None) == -5
    assert lib.qr_kv_dequant_i4_f16(one, one, one, 0, 128, one, None) == 0
    # the entry point with the built-in scratch buffer: a shape beyond the buffer is refused by size alone
    assert lib.qr_workspace_bytes(768, 3072, 65536) > (32 << 20)
    assert lib.qr_linear_i4_f16_static(one, one, one, one, None, 768, 3072, 65536, one, None) == -7
    assert lib.qr_linear_i4_f16_static(one, one, one, one, None, 128, 4096, 100, one, None) == -2


def test_workspace_query_needs_no_gpu(lib):
    """qr_workspace_bytes is pure host arithmetic: non-zero exactly for prompts of a few hundred tokens
    whose tiles would leave most CUs idle, a whole number of [M, N] int32 slabs."""
    assert lib.qr_workspace_bytes(2048, 4096, 11008) == 0          # enough tiles
    assert lib.qr_workspace_bytes(8, 8192, 28672) == 0             # decode batches use the decode kernel
    assert lib.qr_workspace_bytes(512, 11008, 4096) == 0           # short K: nothing to split
    for m, n, k in ((256, 4096, 11008), (128, 4096, 4096), (96, 8192, 8192), (256, 8192, 28672)):
        ws = lib.qr_workspace_bytes(m, n, k)
        assert ws > 0 and ws % (m * n * 4) == 0 and 2 <= ws // (m * n * 4) <= 16
    assert lib.qr_workspace_bytes(0, 4096, 4096) == 0 and lib.qr_workspace_bytes(256, 4096, 100) == 0
    one = ctypes.c_void_p(16)
    assert lib.qr_linear_i4_f16_ws(one, None, one, one, None, 4, 4, 64, one, None, 0, None) == -1
    assert lib.qr_linear_i4_f16_ws(one, one, one, one, None, 4, 4, 100, one, None, 0, None) == -2


def test_fp6_path_sizes_and_argument_errors_need_no_gpu(lib):
    """The FP6 matrix path: a converted operand is 6 bits per value; argument errors come back before any launch."""
    assert lib.qr_f6_bytes(2048, 11008) == 2048 * 11008 * 3 // 4
    assert lib.qr_f6_bytes(0, 4096) == 0 and lib.qr_f6_bytes(16, 100) == 0
    one = ctypes.c_void_p(16)
    assert lib.qr_convert_i4_f6(one, 4, 100, one, None) == -2                   # K % 64 != 0
    assert lib.qr_convert_i4_f6(None, 4, 64, one, None) == -1
    assert lib.qr_convert_i4_f6(ctypes.c_void_p(8), 4, 64, one, None) == -4
    assert lib.qr_convert_i4_f6(one, 0, 64, one, None) == 0
    assert lib.qr_linear_f6_f16(one, one, one, one, None, 4, 4, 100, one, None) == -2
    assert lib.qr_linear_f6_f16(one, None, one, one, None, 4, 4, 64, one, None) == -1
    assert lib.qr_linear_f6_f16(ctypes.c_void_p(8), one, one, one, None, 4, 4, 64, one, None) == -4
    assert lib.qr_linear_f6_f16(one, one, one, one, None, 1 << 20, 4, 8192, one, None) == -3   # operand beyond 32-bit offsets
    assert lib.qr_linear_f6_f16(one, one, one, one, None, 0, 4, 64, one, None) == 0


def test_quantized_linear_workspace_and_argument_errors_need_no_gpu(lib):
    """The single-call layer entry point: its workspace holds the codes (M K / 2 bytes), the scales
    (2 M bytes), each rounded up to 16 bytes, and the GEMM's own scratch; argument errors are
    reported before anything is launched."""
    assert lib.qr_quantized_linear_workspace_bytes(1, 8192, 28672) == 14336 + 16
    assert lib.qr_quantized_linear_workspace_bytes(2048, 4096, 11008) == 2048 * 5504 + 4096
    m, n, k = 256, 4096, 11008
    assert lib.qr_quantized_linear_workspace_bytes(m, n, k) == m * k // 2 + 512 + lib.qr_workspace_bytes(m, n, k)
    assert lib.qr_quantized_linear_workspace_bytes(0, n, k) == 0
    one = ctypes.c_void_p(16)
    args = (one, 4, 64, 0, None, 0, 1.0, 1.0, one, one, None, 4, one)
    assert lib.qr_quantized_linear_f16(*args, None, 0, None) == -6                 # no workspace
    assert lib.qr_quantized_linear_f16(*args, one, 100, None) == -6                # too small (needs 128 + 16)
    assert lib.qr_quantized_linear_f16(*args, ctypes.c_void_p(24), 4096, None) == -6   # misaligned
    assert lib.qr_quantized_linear_f16(one, 4, 100, 0, None, 0, 1.0, 1.0, one, one, None, 4, one, one, 4096, None) == -2
    assert lib.qr_quantized_linear_f16(None, 4, 64, 0, None, 0, 1.0, 1.0, one, one, None, 4, one, one, 4096, None) == -1
    assert lib.qr_quantized_linear_f16(one, 0, 64, 0, None, 0, 1.0, 1.0, one, one, None, 4, one, None, 0, None) == 0
    assert b"workspace" in lib.qr_strerror(-6)


def test_missing_library_fails_loudly(monkeypatch, tmp_path):
    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.setattr(_lib, "LIB_PATH", tmp_path / "nope.so")
    with pytest.raises(RuntimeError, match="no CPU or PyTorch fallback"):
        _lib.lib()


def test_plan_names_a_kernel_for_every_shape_and_stays_within_the_workspace(lib):
    """qr_linear_plan: a name for every shape that the product takes, scratch that is a whole number of [M, N] int32 slabs, no more
    than offered, and the same plan again when only that much is offered; NULL for shapes that are refused."""
    seen = set()
    used = ctypes.c_size_t()
    for m in (1, 2, 4, 5, 7, 8, 24, 40, 48, 64, 65, 128, 300, 333, 777, 1260, 2048, 8191, 32768):
        for n in (1, 100, 128, 520, 4096, 5120, 8192, 12288, 28672, 57344):
            for k in (64, 1088, 4096, 11008, 28672, 131008):
                offered = lib.qr_workspace_bytes(m, n, k)
                name = lib.qr_linear_plan(m, n, k, offered, ctypes.byref(used))
                assert name and used.value <= offered and used.value % (m * n * 4) == 0, (m, n, k)
                assert (b"sliced" in name) == (used.value > 0)
                assert lib.qr_linear_plan(m, n, k, used.value, None) == name
                assert b"sliced" not in lib.qr_linear_plan(m, n, k, 0, None)
                seen.add(name)
    assert len(seen) == 11 and lib.qr_linear_plan(1 << 17, 128, 131008, 0, None) == b"gemm_i4_kernel", seen
    for bad in ((0, 1, 64), (1, 0, 64), (1, 1, 0), (1, 1, 100), (1, 1, 131072), (1 << 31, 1, 64)):
        assert lib.qr_linear_plan(*bad, 0, None) is None


def test_plan_of_five_small_tiles_per_cu(lib):
    """64 x 64 tiles, five on the busiest CU, against a K of 4096 and more: 128-row tiles on the FP6 matrix path take them, light weights or
    heavy (measured, 64 x 64 / 128 x 256 in us: 58 / 50, 71 / 59, 138 / 110, 89 / 75, 147 / 118, 74 / 58, 45 / 38, 42 / 37.5, 25.2 / 23.8;
    at K = 2048 they are even, 16.4 / 16.6)."""
    for m, n, k in ((1260, 4096, 11008), (1000, 5120, 13824), (2560, 2048, 28672), (1280, 4096, 17920), (600, 8192, 28672),
                    (300, 13824, 13824), (640, 8192, 8192), (300, 13824, 8192), (1280, 4096, 4096)):
        assert lib.qr_linear_plan(m, n, k, 0, None) == b"gemm_spk_kernel", (m, n, k)
    assert lib.qr_linear_plan(1280, 4096, 1024, 0, None) == b"gemm_mid_kernel<64,64>"


def test_plan_of_very_wide_outputs(lib):
    """The large tiles store through 32-bit offsets from a tile's first row: 256 rows of fp16 up to 2^23 columns, 128 up to 2^24."""
    for n in ((1 << 22) - 8, 1 << 22, 4500000):
        assert lib.qr_linear_plan(256, n, 1856, 0, None) == b"gemm_sp256_kernel", n
    for n in (1 << 24, (1 << 25) + 64):
        assert lib.qr_linear_plan(256, n, 192, 0, None).startswith(b"gemm_mid_kernel"), n


def test_plan_counts_the_cost_of_an_output_that_ends_inside_a_tile(lib):
    """A last column of tiles that the output's edge cuts, and rows of no whole 16-byte pieces, leave the small tiles element by element,
    the 128 x 128 ones slowest (measured: 9 us on 64 x 64 tiles, 14 on 128 x 128, for the first shape)."""
    for m, n, k in ((133, 11112, 1024), (5568, 448, 448), (440, 5568, 128), (3000, 704, 704), (1001, 2649, 768), (106, 18581, 256)):
        assert lib.qr_linear_plan(m, n, k, 0, None) == b"gemm_mid_kernel<64,64>", (m, n, k)
    offered = lib.qr_workspace_bytes(83, 5120, 13824)           # (18 us in slices of K, 22 in one launch)
    assert b"sliced" in lib.qr_linear_plan(83, 5120, 13824, offered, None)


def test_plan_counts_columns_left_in_a_cut_tile_and_weights_that_no_cache_holds(lib):
    """Eight columns left in the last 128 x 128 tile cost little (measured: 13.4 us, 15.2 on 64 x 64 tiles); 130 MB of weights are read from
    memory, twice by 64-row tiles (45 us on 128 x 128, 63 on 64 x 64); a long K in as many slices as pay (30 us in four, 34 in two)."""
    for m, n, k in ((76, 24584, 2176), (111, 28736, 9024)):
        assert lib.qr_linear_plan(m, n, k, 0, None) == b"gemm_mid_kernel<128,128>", (m, n, k)
    used = ctypes.c_size_t()
    lib.qr_linear_plan(100, 4096, 28672, lib.qr_workspace_bytes(100, 4096, 28672), ctypes.byref(used))
    assert used.value == 4 * 100 * 4096 * 4


def test_plan_spreads_tokens_only_where_weights_from_memory_leave_a_lead(lib):
    """Few tokens, spread, against wide weights, packed: the loop waits for weights that come from memory (measured with the tokens spread / in one
    launch, in us: 36.1 / 30.6, 36.5 / 31.8, 50.5 / 45.8, 25.8 / 23.9, 35.5 / 29.8, 35.6 / 29.7, 43.3 / 38.2, 27.1 / 23.6, 61.9 / 59.5, 64.3 / 60.1);
    with more tokens to a tile, and with the weights spread, the lead is there (29.6 / 33.1, 61.3 / 72.8, 30.7 / 35.4, 37.5 / 40.6, 123 / 140)."""
    for m, n, k in ((160, 27648, 5120), (200, 27648, 5120), (256, 28672, 8192), (333, 12288, 4096), (333, 15360, 5120), (400, 13824, 5120),
                    (512, 10240, 8192), (512, 11008, 4096), (65, 57344, 8192), (128, 57344, 8192)):
        assert lib.qr_linear_spread_bytes(m, n, k) == 0, (m, n, k)
    for m, n, k in ((333, 22016, 4096), (400, 28672, 8192), (700, 12288, 4096), (1024, 12288, 4096), (1024, 28672, 8192), (1777, 8192, 28672),
                    (8191, 5120, 5120), (32768, 11008, 4096), (2048, 5120, 5120), (2048, 8192, 8192)):
        assert lib.qr_linear_spread_bytes(m, n, k) > 0, (m, n, k)
