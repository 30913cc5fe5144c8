"""The native host side of the entry points (csrc/host.cpp): same results and shapes as the general route of the Python
wrappers, and None -- which sends a call down that route -- for whatever is not its plain case."""
import pytest
import torch

import quarot_amd
from quarot_amd import _lib
from quarot_amd.transformers import kv_cache as kv

pytestmark = pytest.mark.gpu
host = quarot_amd._host


class _Refuses:
    """A host module that refuses every call: the wrappers take their general route."""

    def __getattr__(self, name):
        return lambda *args: None


@pytest.fixture
def general_route(monkeypatch):
    def switch():
        monkeypatch.setattr(quarot_amd, "_host", _Refuses())
        monkeypatch.setattr(_lib, "host", _Refuses())
    return switch


@pytest.mark.parametrize("lead", [(1,), (7,), (2, 3), (1, 70), (2, 1, 3)])
def test_same_results_and_shapes_as_the_general_route(lead, general_route):
    torch.manual_seed(len(lead))
    x = torch.randn(*lead, 11008, device="cuda").half()
    nn = quarot_amd.nn
    with torch.device("cuda"):
        lin = nn.Linear4bit(11008, 320, bias=True).half()
        plain = nn.Linear4bit(11008, 320).half()
    lin.weight_scales.uniform_(1e-3, 2e-3), plain.weight_scales.uniform_(1e-3, 2e-3), lin.bias.normal_()
    xh = torch.randn(*lead, 40, 128, device="cuda").half()
    modules = [nn.Quantizer(0.9), lambda y: quarot_amd.rmsnorm(y, 11008), nn.RMSNormQuantizer(11008, input_clip_ratio=0.95), nn.OnlineHadamard(11008).cuda(),
               nn.OnlineHadamard(11008, force_fp32=True).cuda(), nn.OnlineHadamardQuantizer(11008).cuda(),
               nn.OnlineHadamardQuantizer(11008, force_fp32=True).cuda(), nn.HeadsHadamardQuantizer(40).cuda(),
               nn.Linear4bitSequential(nn.Quantizer(), lin), nn.Linear4bitSequential(nn.OnlineHadamard(11008).cuda(), nn.Quantizer(), plain),
               torch.nn.Sequential(nn.Quantizer(), lin)]
    run = lambda: [m(xh if isinstance(m, nn.HeadsHadamardQuantizer) else x) for m in modules]
    got = run()
    general_route()
    for a, b in zip(got, run()):
        if isinstance(a, quarot_amd.PackedQuantizedTensor):
            assert a.scales_x.shape == b.scales_x.shape and torch.equal(a.scales_x.view(torch.int16), b.scales_x.view(torch.int16))
            a, b = a.quantized_x, b.quantized_x
        assert a.shape == b.shape and a.dtype == b.dtype
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))


def test_refuses_what_is_not_its_plain_case():
    x = torch.randn(4, 128, device="cuda").half()
    for bad in (x.cpu(), x.float(), x.t(), x[:, ::2], x[:0], x[0, 0], torch.nn.Module(), None, 3):
        assert host.quantize_rows(bad, 1.0) is None
    assert host.quantize_rows(x, "1.0") is None
    assert isinstance(host.quantize_rows(torch.nn.Parameter(x, requires_grad=False), 1.0), tuple)
    q, s = host.quantize_rows(x, 1.0)
    w, sw = torch.zeros(8, 64, dtype=torch.uint8, device="cuda"), torch.ones(8, 1, device="cuda").half()
    assert host.linear(q, s, w, sw, None).shape == (4, 8)
    for args in ((q, s[:2], w, sw, None), (q, s, w[:, :32], sw, None), (q, s, w, sw[:4], None), (q, s, w, sw, sw[:4].view(-1)),
                 (q, s, w, sw.float(), None), (q.cpu(), s, w, sw, None), (q, s, None, sw, None)):
        assert host.linear(*args) is None
    with pytest.raises(TypeError):
        host.linear(q, s)


@pytest.mark.parametrize("batch,length,page", [(1, 1, 16), (3, 16, 16), (5, 17, 16), (2, 4001, 128), (40, 300, 5)])
def test_page_tables_in_one_launch(batch, length, page, general_route):
    c = kv.MultiLayerPagedKVCache4Bit(batch, page, length, "cuda", 1, 1, 128)
    c.length = length
    got = c.get_cache_specs_for_flash_infer(None)
    general_route()
    c._specs = None
    want = c.get_cache_specs_for_flash_infer(None)
    for name in ("kv_indptr", "kv_indices", "last_page_offset"):
        assert got[name].dtype == torch.int32 and torch.equal(got[name], want[name]), name


def test_rmsnorm_under_transforms_tracers_and_forward_mode():
    """What torch's operations took before there was a kernel, RMSNorm still takes."""
    import torch.autograd.forward_ad as fwad
    from torch.fx.experimental.proxy_tensor import make_fx
    norm = quarot_amd.nn.RMSNorm(64)
    x, t = torch.randn(2, 5, 3, 64, device="cuda").half().unbind(0)
    plain = norm(x)
    want = torch.func.jvp(lambda y: norm(y.float()), (x,), (t,))[1]           # (fp32 rows: always torch)
    assert torch.equal(torch.func.vmap(norm)(x), norm(x.clone()))
    near = lambda a: torch.testing.assert_close(a.float(), want, rtol=1e-3, atol=2e-3)      # fp16 results of values up to ~4
    near(torch.func.jvp(norm, (x,), (t,))[1])
    with fwad.dual_level():
        near(fwad.unpack_dual(norm(fwad.make_dual(x, t))).tangent)
    more = torch.cat([x, x])
    for traced in (make_fx(norm)(x), torch.jit.trace(norm, x)):
        torch.testing.assert_close(traced(x * 2), plain, rtol=1e-3, atol=1e-3)
    assert torch.jit.trace(norm, x)(more).shape == more.shape and torch.jit.script(norm)(x).shape == x.shape
    leaf = x.clone().requires_grad_()
    assert norm(leaf).requires_grad and not norm(x).requires_grad


def test_out_of_memory_keeps_its_type():
    n = 1 << 15
    q, s = torch.zeros(n, 32, dtype=torch.uint8, device="cuda"), torch.ones(n, 1, device="cuda").half()
    torch.cuda.empty_cache()
    allowed = torch.cuda.memory_reserved() + 2 ** 30
    torch.cuda.set_per_process_memory_fraction(allowed / torch.cuda.mem_get_info()[1])
    try:
        with pytest.raises(torch.OutOfMemoryError):                           # 2 GiB of output
            host.linear(q, s, q, s, None)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)


def test_decode_workspace_made_under_capture_is_not_kept():
    """The arrival counters of such a workspace are zeroed by replays of that graph only: an eager step without a replay
    makes its own."""
    g = torch.Generator(device="cuda").manual_seed(3)
    rnd = lambda n: torch.randn(1, n, 4, 128, generator=g, device="cuda").half()
    k0, v0, step = rnd(2048), rnd(2048), [rnd(1) for _ in range(3)]
    caches = [kv.MultiLayerPagedKVCache4Bit(1, 16, 2100, "cuda", 1, 4, 128) for _ in range(2)]
    for c in caches:
        c.pages.zero_(), c.scales.zero_()
        c.update(k0, v0, 0)
        c._decode_ws = c._decode_ws_key = None
    run = lambda c: c.update(step[0], step[1], 0)(step[2])
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = run(caches[0])
    assert caches[0]._decode_ws is None
    for _ in range(3):
        graph.replay()
        caches[1].length = 2048
        want = run(caches[1])
        assert torch.equal(captured, want)
    assert torch.equal(run(caches[0]), run(caches[1])) and caches[0]._decode_ws is not None


def test_other_threads_run_while_the_host_route_launches():
    """With a switch interval that never ends, another Python thread gets on only when this one gives the interpreter's lock away:
    at each allocation and launch, as around ctypes' calls."""
    import sys
    import threading
    import time
    x = torch.randn(4, 128, device="cuda").half()
    host.quantize_rows(x, 1.0)
    turns, stop, started, interval = [0], threading.Event(), threading.Event(), sys.getswitchinterval()

    def other():
        started.set()
        while not stop.is_set():
            turns[0] += 1
            time.sleep(0)

    thread = threading.Thread(target=other, daemon=True)
    sys.setswitchinterval(1e4)
    try:
        thread.start()
        assert started.wait(30)
        before = turns[0]
        kept = [host.quantize_rows(x, 1.0) for _ in range(200)]               # (freeing a tensor may give the lock away too)
        assert turns[0] - before >= len(kept)
    finally:
        stop.set()
        sys.setswitchinterval(interval)
        thread.join(30)


def test_a_flag_without_a_truth_value_raises_its_own_error():
    """As the general route does, with nothing stored: not a launch followed by a SystemError."""
    c = kv.MultiLayerPagedKVCache4Bit(1, 16, 16, "cuda", 1, 2, 128)
    c.length = 1
    c.pages.zero_()
    tables = c.get_cache_specs_for_flash_infer(None)
    x = torch.randn(1, 2, 128, device="cuda").half()
    with pytest.raises(RuntimeError, match="[Bb]oolean value"):
        kv.quantize_append_kv_i4(**tables, k=x, v=x, seqlen_indptr=None, layer_idx=0, hadamard=torch.ones(2))
    assert int(c.pages.max()) == 0


def _decode_caches(n, length=2048, heads=4):
    """Caches that hold the same prompt, and tensors of some decode steps; steps of this length are split over workgroups."""
    g = torch.Generator(device="cuda").manual_seed(5)
    rnd = lambda t: torch.randn(1, t, heads, 128, generator=g, device="cuda").half()
    k0, v0, steps = rnd(length), rnd(length), [[rnd(1) for _ in range(3)] for _ in range(4)]
    caches = [kv.MultiLayerPagedKVCache4Bit(1, 16, length + 52, "cuda", 1, heads, 128) for _ in range(n)]
    for c in caches:
        c.pages.zero_(), c.scales.zero_()
        c.update(k0, v0, 0)
    assert kv._decode_workspace_bytes(1, heads, length + 1, 0) > 0
    return caches, steps


class _Spy:
    """The host module, with a record of the workspaces that decode steps were launched with."""

    def __init__(self):
        self.workspaces = []

    def __getattr__(self, name):
        return getattr(host, name)

    def decode_step(self, *args):
        self.workspaces.append(args[12])
        return host.decode_step(*args)


@pytest.fixture
def spy(monkeypatch):
    monkeypatch.setattr(_lib, "host", _Spy())
    return _lib.host


def test_decode_workspaces_of_two_streams_are_two(spy):
    """A workspace holds partial states and arrival counters; launches of different streams may overlap, so they share none, and
    what an overlap would leave in one stream's counters does not reach another stream's steps."""
    (a, b), steps = _decode_caches(2)
    streams, got = [torch.cuda.Stream() for _ in range(2)], []
    torch.cuda.synchronize()
    for i, s in enumerate(steps):
        with torch.cuda.stream(streams[1 - i % 2]):
            call = a.update(s[0], s[1], 0)
        torch.cuda.synchronize()
        with torch.cuda.stream(streams[i % 2]):                        # (the stream of the call counts, not update's)
            got.append(call(s[2]))
        torch.cuda.synchronize()
        if i == 1:
            spy.workspaces[1][:16] = 1                                 # (the fourth step, on that stream, is not looked at)
    ws = list(spy.workspaces)
    want = [b.update(s[0], s[1], 0)(s[2]) for s in steps[:3]]
    assert all(torch.equal(x, y) for x, y in zip(got, want))
    assert ws[0] is ws[2] and ws[1] is ws[3] and ws[0].data_ptr() != ws[1].data_ptr()
    for _ in range(2 * kv._MAX_WORKSPACES):
        with torch.cuda.stream(torch.cuda.Stream()):
            a.length -= 1
            a.update(steps[0][0], steps[0][1], 0)(steps[0][2])
    torch.cuda.synchronize()
    assert len(a._workspaces) <= kv._MAX_WORKSPACES


def test_a_captured_decode_step_has_its_own_workspace(spy):
    """Replays may overlap eager steps of any stream: a graph uses no workspace of an eager step or of another graph, one for all
    the layers of a capture, and zeroes its counters itself."""
    (a, b), steps = _decode_caches(2)
    run = lambda c, s: c.update(s[0], s[1], 0)(s[2])

    def captured(s):
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            a.length -= 1
            out = [run(a, s)]
            a.length -= 1                                              # (a second layer, as far as the workspace goes)
            out.append(run(a, s))
        return graph, out

    assert torch.equal(run(a, steps[0]), run(b, steps[0]))
    one, out = captured(steps[1])
    two, _ = captured(steps[1])
    eager, _, ws, same, other = spy.workspaces[:5]
    assert ws is same and len({t.data_ptr() for t in (eager, ws, other)}) == 3
    eager[:16] = 1                                                     # a step of another stream in flight
    b.length -= 1
    want = run(b, steps[1])
    for _ in range(3):
        ws[:16] = 1                                                    # whatever its memory held
        one.replay()
        torch.cuda.synchronize()
        assert torch.equal(out[0], want) and torch.equal(out[1], want)


def test_page_tables_made_under_capture_are_that_graphs_own():
    """They are filled by replays only: an eager step at that length that comes first makes its own, and the graph reads none of an
    eager step, whose memory goes back when the cache grows."""
    (a, b), steps = _decode_caches(2)
    tables = lambda c: [c.get_cache_specs_for_flash_infer(None)[n] for n in ("kv_indptr", "kv_indices", "last_page_offset")]
    eager = tables(a)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        inside, again = tables(a), tables(a)
        a.length += 1
        longer = tables(a)
        out = a._stub.forward(steps[0][2], 4, a.get_cache_specs_for_flash_infer(None), 0, a.length)
        a.length -= 1
    assert all(x is y for x, y in zip(inside, again)) and not any(x is y for x, y in zip(inside, eager))
    a.length += 1
    for x, y in zip(tables(a), longer):                                # no replay yet
        assert x is not y
    b.length += 1
    assert all(torch.equal(x, y) for x, y in zip(tables(a), tables(b)))
    want = b._stub.forward(steps[0][2], 4, b.get_cache_specs_for_flash_infer(None), 0, b.length)
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want) and all(torch.equal(x, y) for x, y in zip(longer, tables(b)))


@pytest.mark.parametrize("m,n,k", [(128, 4096, 11008), (256, 4096, 11008), (48, 5120, 13824), (96, 512, 8192)])
def test_linear_allocates_the_scratch_that_its_plan_uses(m, n, k, general_route):
    """The slabs of a K split are allocated where K is split, and not where the library would take room for them but has no use for
    it (128 x 11008 -> 4096: 10 MiB); on both routes, alone and behind the quantiser."""
    import ctypes
    L, used = _lib.lib(), ctypes.c_size_t()
    L.qr_linear_plan(m, n, k, L.qr_workspace_bytes(m, n, k), ctypes.byref(used))
    x, w, sw = torch.randn(m, k, device="cuda").half(), torch.zeros(n, k // 2, dtype=torch.uint8, device="cuda"), torch.ones(n, 1, device="cuda").half()
    q, s = quarot_amd.quantize_rows(x)

    def taken(call):
        torch.cuda.synchronize()
        before = torch.cuda.memory_allocated()
        torch.cuda.reset_peak_memory_stats()
        call()
        return torch.cuda.max_memory_allocated() - before

    def both():
        yield taken(lambda: quarot_amd.linear_i4(q, s, w, sw)), 0
        yield taken(lambda: quarot_amd.quantized_linear(x, w, sw)), m * k // 2 + 2 * m
    for route in ("native", "general"):
        for got, codes in both():
            least = 2 * m * n + used.value + codes
            assert least <= got < least + 2 ** 21, (route, got, least)         # (the allocator leaves up to 1 MiB of a block unused)
        general_route()
