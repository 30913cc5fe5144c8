"""The GEMM on the FP6 matrix path straight from packed nibbles (128-, 192- and 256-row tiles) and on 96 x 64 tiles, bit for bit: int32 sums against exact integer
sums (fp32 products of chunks of K: integers below 2^24), fp16 outputs against the epilogue's rounded operations on those sums."""
import ctypes

import pytest
import torch

from quarot_amd import _lib

pytestmark = pytest.mark.gpu


def _codes(packed):
    low, high = (packed & 15).to(torch.int8), (packed >> 4).to(torch.int8)
    return torch.stack(((low ^ 8) - 8, (high ^ 8) - 8), -1).flatten(1)


def _sums(a, b):
    total = torch.zeros(a.shape[0], b.shape[0], dtype=torch.int32, device=a.device)
    for k in range(0, a.shape[1], 8192):
        total += (_codes(a[:, k:k + 8192]).float() @ _codes(b[:, k:k + 8192]).float().T).to(torch.int32)
    return total


def _operand(rows, k, kind, gen):
    if kind == "random":
        return torch.randint(0, 256, (rows, k // 2), dtype=torch.uint8, device="cuda", generator=gen)
    if kind in ("high", "turn", "signs"):
        r = torch.randint(0, 256, (rows, k // 2), dtype=torch.uint8, device="cuda", generator=gen)
        x = (r & 0x11) | 0x66                                # codes 6 and 7
        if kind == "turn":                                   # codes -8 and -7 up to where the accumulators are first corrected
            x[:, :24576] = (r[:, :24576] & 0x11) | 0x88
        if kind == "signs":                                  # 6, 7, -7 and -6 (a nibble and its complement)
            x ^= (r & 0x02) // 0x02 * 0x0F
            x ^= (r & 0x20) // 0x20 * 0xF0
        return x
    x = torch.full((rows, k // 2), 0x77, dtype=torch.uint8, device="cuda")     # the largest and smallest sums, with and without the offset
    x[::3] = 0x88
    x[1::7] = 0
    return x


def _compare(m, n, k, kind):
    lib = _lib.lib()
    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    a, b = _operand(m, k, "high" if kind == "cancel" else kind, gen), _operand(n, k, "signs" if kind == "cancel" else kind, gen)
    sa = (torch.rand(m, 1, device="cuda", generator=gen) * 0.1 + 0.01).half()
    sb = (torch.rand(n, device="cuda", generator=gen) * 0.01 + 0.001).half()
    bias = torch.randn(n, device="cuda", generator=gen).half()
    want = _sums(a, b)
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    c = torch.full((m + 1, n), 7, dtype=torch.int32, device="cuda")            # (a guard row behind the output)
    assert lib.qr_matmul_i4_i32(p(a), p(b), m, n, k, p(c), None) == 0
    assert torch.equal(c[:m], want) and bool((c[m] == 7).all())
    scaled = (sa * sb) * want.float().half()
    for bi in (None, bias):
        y = torch.full((m + 1, n), 7, dtype=torch.float16, device="cuda")
        assert lib.qr_linear_i4_f16(p(a), p(sa), p(b), p(sb), p(bi) if bi is not None else None, m, n, k, p(y), None) == 0
        assert torch.equal(y[:m], scaled if bi is None else scaled + bi) and bool((y[m] == 7).all())


@pytest.mark.parametrize("m,n,k,kernel", [
    # one row, a remainder and a whole last tile in both directions; K of one stage, of a ragged last stage, of a whole one
    (2049, 4100, 192, "gemm_sp256_kernel"), (2305, 5124, 64, "gemm_sp256_kernel"), (2040, 4099, 320, "gemm_sp256_kernel"),
    (2048, 5120, 1088, "gemm_sp256_kernel"), (1025, 8201, 2112, "gemm_sp256_kernel"), (8200, 2050, 448, "gemm_sp256_kernel"),
    (2040, 4096, 4096, "gemm_spk_kernel"), (1800, 8197, 832, "gemm_spk_kernel"), (2047, 4088, 11008, "gemm_spk_kernel"),
    (4353, 4099, 2112, "gemm_sp256_tail_kernel"), (4600, 4104, 4096, "gemm_sp256_tail_kernel"),
    # around the points where the accumulators are corrected by the row sums (every 49152 k), and the longest K
    (520, 9000, 49152, "gemm_spk_kernel"), (520, 9000, 49216, "gemm_spk_kernel"), (513, 16388, 131008, "gemm_sp256_kernel"),
])
@pytest.mark.parametrize("kind", ["random", "extreme"])
def test_gemm_of_large_tiles_bit_exact(m, n, k, kernel, kind):
    assert _lib.lib().qr_linear_plan(m, n, k, 0, None) == kernel.encode()
    _compare(m, n, k, kind)


# Three and more tiles per workgroup, whose pipeline runs on from one tile into the next: 192- and 256-row tiles and whole rounds before a
# last one of 128-row tiles, K that ends inside a stage, an odd and an even number of stages.
@pytest.mark.parametrize("m,n,k,kernel", [
    (9000, 9003, 704, "gemm_sp256_kernel"), (12500, 5124, 448, "gemm_sp256_kernel"),           # 192 rows
    (24900, 4100, 576, "gemm_sp256_kernel"), (9216, 5120, 1344, "gemm_sp256_kernel"),          # 256 rows
    (11700, 4100, 576, "gemm_sp256_tail_kernel"), (16640, 4160, 832, "gemm_sp256_tail_kernel"), (6145, 16388, 320, "gemm_sp256_tail_kernel"),
    (20000, 5121, 1088, "gemm_sp256_tail_kernel")])
def test_gemm_of_many_large_tiles_bit_exact(m, n, k, kernel):
    assert _lib.lib().qr_linear_plan(m, n, k, 0, None) == kernel.encode()
    _compare(m, n, k, "random")


# Sums of products of codes + 8, of either parity, up to 14.2 million of the 16.8 million that fp32 holds exactly: "high" 10.3 million
# before a correction, "turn" 3 million of small products corrected and 11 million of large ones on top, "cancel" 5.7 million that come to
# a few thousand in the end, so that fp16 outputs are finite.  Walks of three tiles whose turn (two stages before the end) meets the
# correction every 192 stages: 192, 193 and 194 stages.
@pytest.mark.parametrize("m,n,k,kernel", [
    (520, 9000, 49152, "gemm_spk_kernel"), (520, 9000, 98304, "gemm_spk_kernel"), (513, 16388, 131008, "gemm_sp256_kernel"),
    (11776, 4096, 49152, "gemm_sp256_kernel"), (11700, 4090, 49408, "gemm_sp256_kernel"), (11776, 4096, 49664, "gemm_sp256_kernel"),
    (8450, 4100, 49408, "gemm_sp256_tail_kernel")])
@pytest.mark.parametrize("kind", ["high", "turn", "cancel"])
def test_large_sums_of_either_parity_bit_exact(m, n, k, kernel, kind):
    assert _lib.lib().qr_linear_plan(m, n, k, 0, None) == kernel.encode()
    _compare(m, n, k, kind)


@pytest.mark.parametrize("m,n,k", [
    # one 96 x 64 tile on each CU: whole tiles, one row or column into the last one, K that ends inside a stage, rows of no whole
    # 16-byte pieces; the last two: two tiles on a CU
    (333, 4096, 4096), (192, 8192, 11008), (193, 5377, 4160), (385, 3200, 4160), (260, 5440, 2048), (96, 10241, 4160), (95, 12300, 8256), (385, 3000, 4160),
    (257, 10241, 4160), (257, 10241, 11008)])
@pytest.mark.parametrize("kind", ["random", "extreme"])
def test_gemm_of_96_row_tiles_bit_exact(m, n, k, kind):
    assert _lib.lib().qr_linear_plan(m, n, k, 0, None) == b"gemm_mid_kernel<96,64>"
    _compare(m, n, k, kind)


@pytest.mark.parametrize("m,n,k", [(190, 8131, 2112), (275, 5437, 1600)])       # (three 64 x 64 tiles on a CU)
@pytest.mark.parametrize("kind", ["random", "extreme"])
def test_gemm_of_64_row_tiles_bit_exact(m, n, k, kind):
    _compare(m, n, k, kind)


# (at most one 64 x 64 tile on a CU and weights on either side of 10 MB: four stage buffers or three; whole and ragged tiles, K that ends
# inside a stage, walks of ten stages and of several hundred)
@pytest.mark.parametrize("m,n,k", [(65, 8190, 2560), (128, 8192, 2432), (128, 8192, 2496), (127, 5121, 4160), (249, 4095, 11072), (70, 512, 65536)])
@pytest.mark.parametrize("kind", ["random", "extreme"])
def test_gemm_of_64_row_tiles_with_a_cu_each_bit_exact(m, n, k, kind):
    assert _lib.lib().qr_linear_plan(m, n, k, 0, None) == b"gemm_mid_kernel<64,64>"
    _compare(m, n, k, kind)


# (up to 64 rows, K whole: 16 rows ask for all stage buffers at once and 17 for the later ones behind the first stage; five buffers with a CU each, or
# three; ragged last tiles and stages)
@pytest.mark.parametrize("m,n,k", [(8, 12288, 4096), (16, 12280, 4160), (17, 12280, 4160), (17, 12288, 4096), (16, 22009, 4096), (64, 15361, 5120)])
@pytest.mark.parametrize("kind", ["random", "extreme"])
def test_gemm_of_64_row_tiles_of_one_row_bit_exact(m, n, k, kind):
    assert _lib.lib().qr_linear_plan(m, n, k, 0, None) == b"gemm_mid_kernel<64,64>"
    _compare(m, n, k, kind)


# (slices of K; 70 rows: four buffers by the weights' size; up to 64 rows: four with at most one slice on a CU, or three)
@pytest.mark.parametrize("m,n,k", [(70, 512, 65536), (193, 2500, 16448), (48, 5120, 13824), (23, 5100, 13888), (64, 4096, 11008), (48, 5120, 20480)])
@pytest.mark.parametrize("kind", ["random", "extreme"])
def test_gemm_of_64_row_tiles_in_slices_of_k_bit_exact(m, n, k, kind):
    lib, used = _lib.lib(), ctypes.c_size_t()
    assert lib.qr_linear_plan(m, n, k, lib.qr_workspace_bytes(m, n, k), ctypes.byref(used)) == b"gemm_mid_kernel<64,64> (K sliced) + dequant_slabs_kernel"
    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    a, b = _operand(m, k, kind, gen), _operand(n, k, kind, gen)
    sa = (torch.rand(m, 1, device="cuda", generator=gen) * 0.1 + 0.01).half()
    sb = (torch.rand(n, device="cuda", generator=gen) * 0.01 + 0.001).half()
    ws = torch.full((used.value + 4096,), 0xA5, dtype=torch.uint8, device="cuda")
    y = torch.full((m + 1, n), 7, dtype=torch.float16, device="cuda")
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    assert lib.qr_linear_i4_f16_ws(p(a), p(sa), p(b), p(sb), None, m, n, k, p(y), p(ws), used.value, None) == 0
    assert torch.equal(y[:m], (sa * sb) * _sums(a, b).float().half()) and bool((y[m] == 7).all()) and bool((ws[used.value:] == 0xA5).all())


@pytest.mark.parametrize("m,n,k", [(333, 4096, 4096), (2048, 4096, 1088)])      # 96 x 64 tiles, 128 or more rows
@pytest.mark.parametrize("shift", [1, 4])
def test_scales_and_bias_may_start_anywhere(m, n, k, shift):
    lib = _lib.lib()
    gen = torch.Generator(device="cuda").manual_seed(m)
    a, b = _operand(m, k, "random", gen), _operand(n, k, "random", gen)
    sa = (torch.rand(m + shift, 1, device="cuda", generator=gen) * 0.1 + 0.01).half()[shift:]
    sb = (torch.rand(n + shift, device="cuda", generator=gen) * 0.01 + 0.001).half()[shift:]
    bias = torch.randn(n + shift, device="cuda", generator=gen).half()[shift:]
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    y = torch.empty(m, n, dtype=torch.float16, device="cuda")
    assert lib.qr_linear_i4_f16(p(a), p(sa), p(b), p(sb), p(bias), m, n, k, p(y), None) == 0
    assert torch.equal(y, (sa * sb) * _sums(a, b).float().half() + bias)


def test_ragged_rows_of_an_operand_that_ends_below_4_gib():
    """262657 x 16352 bytes = 2^32 - 32: pieces past the end of a row must lie beyond even this operand's last byte."""
    m, n, k = 262657, 256, 32704
    assert m * k // 2 == 2**32 - 32 and _lib.lib().qr_linear_plan(m, n, k, 0, None).startswith(b"gemm_sp")
    gen = torch.Generator(device="cuda").manual_seed(k)
    a = torch.empty(m, k // 2, dtype=torch.uint8, device="cuda")
    for rows in a.split(1 << 15):
        rows.copy_(_operand(rows.shape[0], k, "random", gen))
    b = _operand(n, k, "random", gen)
    sa, sb = torch.ones(m, 1, device="cuda").half(), torch.full((n,), 0.001, device="cuda").half()
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    y = torch.empty(m, n, dtype=torch.float16, device="cuda")
    assert _lib.lib().qr_linear_i4_f16(p(a), p(sa), p(b), p(sb), None, m, n, k, p(y), None) == 0
    for rows in (slice(0, 300), slice(m // 2, m // 2 + 300), slice(m - 300, m)):
        assert torch.equal(y[rows], (sa[rows] * sb) * _sums(a[rows], b).float().half())


@pytest.mark.parametrize("m,n,k,int32", [
    (257, (1 << 22) + 8, 192, False), (130, (1 << 23) - 8, 128, False), (129, 5592403, 192, True), (140, (1 << 23) + 3, 64, False)])
def test_outputs_of_millions_of_columns(m, n, k, int32):
    """Either side of what 256, 192 and 128 rows of an output reach through 32-bit offsets; the output inside guard bands."""
    lib = _lib.lib()
    gen = torch.Generator(device="cuda").manual_seed(n)
    a = _operand(m, k, "random", gen)
    b = torch.randint(0, 256, (n, k // 2), dtype=torch.uint8, device="cuda", generator=gen)
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    out = torch.full((m + 2, n), 7, dtype=torch.int32 if int32 else torch.float16, device="cuda")
    y = out.view(-1)[8:8 + m * n].view(m, n)
    if int32:
        assert lib.qr_matmul_i4_i32(p(a), p(b), m, n, k, p(y), None) == 0
    else:
        sa = (torch.rand(m, 1, device="cuda", generator=gen) * 0.1 + 0.01).half()
        sb = (torch.rand(n, device="cuda", generator=gen) * 0.01 + 0.001).half()
        assert lib.qr_linear_i4_f16(p(a), p(sa), p(b), p(sb), None, m, n, k, p(y), None) == 0
    assert bool((out.view(-1)[:8] == 7).all()) and bool((out.view(-1)[8 + m * n:] == 7).all())
    step = 1 << 19
    for at in range(0, n, step):
        want = _sums(a, b[at:at + step])
        assert torch.equal(y[:, at:at + step], want if int32 else (sa * sb[at:at + step]) * want.float().half()), at
