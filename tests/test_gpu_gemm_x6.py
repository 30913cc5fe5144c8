"""The GEMM whose operand of fewer rows is spread to six bits in the caller's scratch first (gemm_x6.hip), bit for bit against the oracle of the
other large tiles: both operands as the spread one, every tile size, edges of tiles and of K, walks over several tiles per compute unit, the
largest sums; the scratch's limits; the Python entry points with and without room for it."""
import ctypes

import pytest
import torch

import quarot_amd
from quarot_amd import _lib
from test_gpu_gemm_tiles import _operand, _sums

pytestmark = pytest.mark.gpu


class _Refuses:
    def __getattr__(self, name):
        return lambda *a: None


@pytest.fixture
def general_route(monkeypatch):
    def switch():
        monkeypatch.setattr(quarot_amd, "_host", _Refuses())
        monkeypatch.setattr(_lib, "host", _Refuses())
    return switch


_p = lambda t: ctypes.c_void_p(t.data_ptr() if t is not None else None)


def _linear(a, sa, b, sb, bias, ws, ws_bytes, y=None):
    (m, half_k), n = a.shape, b.shape[0]
    if y is None:
        y = torch.full((m + 1, n), 7, dtype=torch.float16, device="cuda")        # (a guard row behind the output)
    rc = _lib.lib().qr_linear_i4_f16_ws(_p(a), _p(sa), _p(b), _p(sb), _p(bias), m, n, 2 * half_k, _p(y), _p(ws), ws_bytes, None)
    assert rc == 0
    return y


def _operands(m, n, k, kind):
    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    a, b = _operand(m, k, "high" if kind == "cancel" else kind, gen), _operand(n, k, "signs" if kind == "cancel" else kind, gen)
    sa = (torch.rand(m, 1, device="cuda", generator=gen) * 0.1 + 0.01).half()
    sb = (torch.rand(n, device="cuda", generator=gen) * 0.01 + 0.001).half()
    return a, sa, b, sb, torch.randn(n, device="cuda", generator=gen).half()


def _plan(m, n, k, ws_bytes):
    return _lib.lib().qr_linear_plan(m, n, k, ws_bytes, None).decode()


@pytest.mark.parametrize("tile,m,n,k,kind", [
    ("128,256", 257, 36144, 320, "random"), ("160,256", 257, 43624, 320, "random"), ("192,256", 1615, 11784, 320, "random"),
    ("224,256", 441, 29448, 320, "extreme"), ("256,256", 673, 32776, 320, "random"), ("256,128", 36099, 296, 320, "random"),
    ("256,160", 24577, 296, 320, "extreme"), ("256,192", 24833, 344, 320, "random"), ("256,224", 29955, 440, 320, "random"),
    ("256,256", 32769, 680, 320, "random"), (None, 3001, 12296, 576, "random"), (None, 2305, 7432, 1088, "extreme"),
    (None, 5003, 4104, 512, "random"), (None, 1777, 8192, 3712, "high"), (None, 2303, 4096, 131008, "turn"), (None, 2303, 4096, 131008, "cancel"),
    (None, 9000, 4096, 32768, "extreme")])
def test_spread_operand_bit_exact(tile, m, n, k, kind):
    need = _lib.lib().qr_linear_spread_bytes(m, n, k)
    assert need > 0 and "gemm_x6" in _plan(m, n, k, need) and (tile is None or f"<{tile}>" in _plan(m, n, k, need)), _plan(m, n, k, need)
    a, sa, b, sb, bias = _operands(m, n, k, kind)
    scaled = (sa * sb) * _sums(a, b).float().half()
    ws = torch.full((need + 4096,), 0xA5, dtype=torch.uint8, device="cuda")       # (nothing in it is read before it is written)
    for bi in (None, bias):
        y = _linear(a, sa, b, sb, bi, ws, need)
        assert torch.equal(y[:m], scaled if bi is None else scaled + bi) and bool((y[m] == 7).all())
        assert bool((ws[need:] == 0xA5).all())
        ws[:need] = 0xFF


def test_scratch_limits_and_outputs_that_the_other_kernels_take():
    m, n, k = 24577, 296, 320
    L = _lib.lib()
    need, used = L.qr_linear_spread_bytes(m, n, k), ctypes.c_size_t()
    assert "gemm_x6" in L.qr_linear_plan(m, n, k, need + 999, ctypes.byref(used)).decode() and used.value == need
    for less in (0, 16, need - 1):
        assert "x6" not in _plan(m, n, k, less)
    assert L.qr_workspace_bytes(m, n, k) == 0 and L.qr_linear_spread_bytes(m, n + 4, k) == 0      # rows of no whole 16-byte pieces
    assert L.qr_linear_spread_bytes(m, n, 256) == 0 and L.qr_linear_spread_bytes(m, n, 100) == 0 and L.qr_linear_spread_bytes(0, n, k) == 0
    assert L.qr_linear_spread_bytes(64, n, k) == 0 and L.qr_linear_spread_bytes(32768, 28672, 28672) == 0      # beyond 512 MiB
    a, sa, b, sb, bias = _operands(m, n, k, "random")
    want = (sa * sb) * _sums(a, b).float().half() + bias
    ws = torch.zeros(need + 16, dtype=torch.uint8, device="cuda")
    for room, at in ((need, 0), (need - 1, 0), (need, 8)):                        # enough, a byte too little, not aligned
        assert torch.equal(_linear(a, sa, b, sb, bias, ws[at:], room)[:m], want)
    y = torch.full((m * n + 8,), 7, dtype=torch.float16, device="cuda")           # an output that starts 8 bytes after a 16-byte boundary
    _linear(a, sa, b, sb, bias, ws, need, y[4:])
    assert torch.equal(y[4:-4].view(m, n), want) and bool((y[:4] == 7).all()) and bool((y[-4:] == 7).all())


def test_python_entry_points_with_and_without_room_for_it(general_route):
    """The module's two calls give it the scratch; a GPU too full for that (here: a limit on this process) takes the one launch, same bits."""
    m, n, k = 4096, 8192, 8192
    gen = torch.Generator(device="cuda").manual_seed(3)
    torch.cuda.empty_cache()                                                      # (no large block with a hole in it)
    x = torch.empty(m, k, dtype=torch.float16, device="cuda").normal_(generator=gen)
    w = _operand(n, k, "random", gen)
    sw = (torch.rand(n, 1, device="cuda", generator=gen) * 0.01).half()
    need = _lib.lib().qr_linear_spread_bytes(m, n, k)
    assert need > 20 << 20
    q, s = quarot_amd.quantize_rows(x)
    want = _linear(q, s, w, sw, None, None, 0)[:m].clone()
    for route in ("native", "general"):
        for call, least in ((lambda: quarot_amd.linear_i4(q, s, w, sw), 2 * m * n), (lambda: quarot_amd.quantized_linear(x, w, sw), 2 * m * n + m * k // 2)):
            for full in (False, True):
                torch.cuda.synchronize()
                torch.cuda.empty_cache()
                before = torch.cuda.memory_allocated()
                torch.cuda.reset_peak_memory_stats()
                if full:
                    total = torch.cuda.get_device_properties(0).total_memory
                    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + least + 0.5 * need) / total)
                try:
                    y = call()
                finally:
                    torch.cuda.set_per_process_memory_fraction(1.0)
                assert (torch.cuda.max_memory_allocated() - before >= least + need) != full
                assert torch.equal(y, want), (route, full)
                del y
        general_route()


def test_scratch_of_a_shape_after_many_others():
    """The native route keeps the sizes of a thread's last shapes: more of them than it keeps, and the first again."""
    m, n, k = 4096, 8192, 4096
    gen = torch.Generator(device="cuda").manual_seed(6)
    q, w = _operand(m, k, "random", gen), _operand(n, k, "random", gen)
    s, sw = (torch.rand(m, 1, device="cuda", generator=gen) * 0.1).half(), (torch.rand(n, 1, device="cuda", generator=gen) * 0.01).half()
    need = _lib.lib().qr_linear_spread_bytes(m, n, k)
    want = (s * sw.view(-1)) * _sums(q, w).float().half()

    def check():
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        held = torch.cuda.memory_allocated()
        y = quarot_amd._host.linear(q, s, w, sw, None)
        assert torch.cuda.max_memory_allocated() - held >= 2 * m * n + need > 2 * m * n and torch.equal(y, want)

    check()
    for rows in range(1, 300, 2):                            # (with slices of K and without, on either side of the fused tokens)
        y = quarot_amd._host.linear(q[:rows], s[:rows], w[:1024], sw[:1024], None)
        assert torch.equal(y, want[:rows, :1024]), rows
        if rows % 50 == 1:
            check()


def test_a_full_gpu_is_asked_for_the_scratch_once(general_route):
    """A refusal costs the allocator's whole cache: of ten calls on a GPU without room one asks, and the first with room again has its scratch."""
    m, n, k = 4096, 8192, 8192
    gen = torch.Generator(device="cuda").manual_seed(5)
    q, w = _operand(m, k, "random", gen), _operand(n, k, "random", gen)
    s, sw = (torch.rand(m, 1, device="cuda", generator=gen) * 0.1).half(), (torch.rand(n, 1, device="cuda", generator=gen) * 0.01).half()
    need, total = _lib.lib().qr_linear_spread_bytes(m, n, k), torch.cuda.get_device_properties(0).total_memory
    assert need > 20 << 20
    want = quarot_amd.linear_i4(q, s, w, sw)
    failed = lambda: sum(torch.cuda.memory_stats()[name] for name in ("num_alloc_retries", "num_ooms"))
    for route in ("native", "general"):
        quarot_amd.linear_i4(q, s, w, sw)                                         # (with room: whatever was refused before is forgotten)
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
        holes = [torch.empty(b["size"], dtype=torch.uint8, device="cuda") for segment in torch.cuda.memory_snapshot() for b in segment["blocks"]
                 if b["state"] == "inactive" and b["size"] >= 1 << 20]            # (what is free in memory that others keep)
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + 2 * m * n + 0.5 * need) / total)
        before = failed()
        try:
            for _ in range(10):
                assert torch.equal(quarot_amd.linear_i4(q, s, w, sw)[::64], want[::64]), route
        finally:
            torch.cuda.set_per_process_memory_fraction(1.0)
        del holes
        assert 1 <= failed() - before <= 2, route                                # (one request: its retry, and its failure)
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        held = torch.cuda.memory_allocated()
        assert torch.equal(quarot_amd.linear_i4(q, s, w, sw), want), route
        assert torch.cuda.max_memory_allocated() - held >= 2 * m * n + need, route
        general_route()


def test_replays_of_a_captured_call():
    m, n, k = 4096, 8192, 4096
    gen = torch.Generator(device="cuda").manual_seed(4)
    x, w = torch.randn(m, k, device="cuda", generator=gen).half(), _operand(n, k, "random", gen)
    sw = (torch.rand(n, 1, device="cuda", generator=gen) * 0.01).half()
    quarot_amd.quantized_linear(x, w, sw)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        quarot_amd.quantized_linear(x, w, sw)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = quarot_amd.quantized_linear(x, w, sw)
    for i in range(4):
        x.copy_(torch.randn(m, k, device="cuda", generator=gen).half())
        want = quarot_amd.quantized_linear(x, w, sw)
        y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want), i
