"""The entry point that allocates nothing (qr_linear_i4_f16_static): through the C ABI, against
qr_linear_i4_f16_ws with a caller-provided workspace, bit for bit, on calls in a row that share the
library's built-in scratch buffer (the later ones with smaller inputs), plus the size limit."""
import ctypes

import numpy as np
import pytest
import torch

from oracle import quarot_oracle as o
from quarot_amd import _lib

pytestmark = pytest.mark.gpu
F16 = np.float16


def gpu(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")


@pytest.fixture(scope="module", autouse=True)
def first_call_on_the_device():
    """The documented first call, which looks the buffer up: it loads the code object that holds the buffer where no other kernel of that
    object has run yet (this file alone), and with it the buffer's memory."""
    a, w, sa, sw, _ = [gpu(t) for t in operands(64, 256, 16384, 0)]
    y = torch.empty(64, 256, dtype=torch.float16, device="cuda:0")
    assert _lib.lib().qr_linear_i4_f16_static(a.data_ptr(), sa.data_ptr(), w.data_ptr(), sw.data_ptr(), None, 64, 256, 16384, y.data_ptr(),
                                              torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()


def operands(m, n, k, seed):
    rng = np.random.default_rng(seed)
    a = o.pack_i4(rng.integers(-8, 8, (m, k)))
    w = o.pack_i4(rng.integers(-8, 8, (n, k)))
    sa = (np.abs(rng.standard_normal(m)) * 0.2 + 0.01).astype(F16)
    sw = (np.abs(rng.standard_normal(n)) * 0.01 + 0.001).astype(F16)
    bias = rng.standard_normal(n).astype(F16)
    return a, w, sa, sw, bias


def run_both(L, m, n, k, seed, with_bias):
    a, w, sa, sw, bias = operands(m, n, k, seed)
    ga, gw, gsa, gsw, gb = gpu(a), gpu(w), gpu(sa), gpu(sw), gpu(bias)
    bptr = gb.data_ptr() if with_bias else None
    st = torch.cuda.current_stream().cuda_stream
    ws_bytes = L.qr_workspace_bytes(m, n, k)
    ws = torch.empty(max(ws_bytes, 16), dtype=torch.uint8, device=ga.device)
    y_ws = torch.full((m, n), float("nan"), dtype=torch.float16, device=ga.device)
    y_st = torch.full((m, n), float("nan"), dtype=torch.float16, device=ga.device)
    assert L.qr_linear_i4_f16_ws(ga.data_ptr(), gsa.data_ptr(), gw.data_ptr(), gsw.data_ptr(), bptr, m, n, k,
                                 y_ws.data_ptr(), ws.data_ptr() if ws_bytes else None, ws_bytes, st) == 0
    free_before = torch.cuda.mem_get_info()[0]
    rc = L.qr_linear_i4_f16_static(ga.data_ptr(), gsa.data_ptr(), gw.data_ptr(), gsw.data_ptr(), bptr, m, n, k,
                                   y_st.data_ptr(), st)
    assert rc == 0, L.qr_strerror(rc)
    torch.cuda.synchronize()
    assert torch.cuda.mem_get_info()[0] == free_before          # the call took no device memory
    assert torch.equal(y_st, y_ws), (m, n, k)
    want = o.linear4bit(a, sa, w, sw, bias if with_bias else None)
    assert np.array_equal(y_st.cpu().numpy().view(np.uint16), want.view(np.uint16)), (m, n, k)
    return ws_bytes


def test_static_scratch_entry_point_matches_the_workspace_form_on_consecutive_calls():
    L = _lib.lib()
    # a split-K shape, then smaller ones that reuse (part of) the same scratch with its old contents,
    # then a shape that needs no scratch, then the first one again
    used = [run_both(L, 256, 4096, 11008, 1, False),
            run_both(L, 130, 520, 4160, 2, True),
            run_both(L, 96, 512, 8192, 3, False),
            run_both(L, 37, 300, 1024, 4, True),
            run_both(L, 2048, 4096, 512, 5, False),
            run_both(L, 256, 4096, 11008, 6, True)]
    assert used[0] > 0 and used[1] > 0 and used[2] > 0 and used[3] == 0 and used[4] == 0
    assert max(used) <= 32 << 20


def test_static_scratch_limit_and_argument_errors():
    L = _lib.lib()
    one = ctypes.c_void_p(256)
    big = None
    for shape in ((768, 3072, 65536), (192, 12288, 130944)):
        if L.qr_workspace_bytes(*shape) > (32 << 20):
            big = shape
            break
    assert big is not None
    assert L.qr_linear_i4_f16_static(one, one, one, one, None, *big, one, None) == -7     # nothing is launched
    assert b"scratch" in L.qr_strerror(-7)
    assert L.qr_linear_i4_f16_static(one, one, one, one, None, 128, 4096, 100, one, None) == -2
    assert L.qr_linear_i4_f16_static(one, None, one, one, None, 128, 4096, 4096, one, None) == -1
    assert L.qr_linear_i4_f16_static(one, one, one, one, None, 0, 4096, 4096, None, None) == 0


@pytest.mark.parametrize("m,n,k,launches", [(8, 4096, 28672, 1), (16, 4096, 28672, 1), (24, 5120, 13824, 1), (39, 4096, 28672, 1),
                                            (48, 5120, 13824, 1), (64, 4096, 16320, 1), (40, 4096, 16384, 2), (64, 8192, 28672, 2)])
def test_static_scratch_is_left_alone_by_decode_batches_below_40_tokens_or_16384_columns(m, n, k, launches):
    """Calls of those sizes may overlap: they must not share the library's buffer.  A call that uses it is two launches (slices, then
    their sum), one that does not is one; the launches are counted in a captured graph.  Results are the oracle's either way."""
    L, used = _lib.lib(), ctypes.c_size_t()
    L.qr_linear_plan(m, n, k, L.qr_workspace_bytes(m, n, k), ctypes.byref(used))
    assert used.value > 0                                              # (with a workspace of its own it would be sliced)
    a, w, sa, sw, _ = operands(m, n, k, m + n)
    ga, gw, gsa, gsw = gpu(a), gpu(w), gpu(sa), gpu(sw)
    y = torch.empty(m, n, dtype=torch.float16, device="cuda:0")
    call = lambda: L.qr_linear_i4_f16_static(ga.data_ptr(), gsa.data_ptr(), gw.data_ptr(), gsw.data_ptr(), None, m, n, k, y.data_ptr(),
                                             torch.cuda.current_stream().cuda_stream)
    assert call() == 0
    cols = np.arange(0, n, 61)
    want = o.linear4bit(a, sa, w[cols], sw[cols], None)
    assert np.array_equal(y[:, cols].cpu().numpy().view(np.uint16), want.view(np.uint16))
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph):
        assert call() == 0
    path = next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64" in line)
    count = ctypes.c_size_t()
    assert ctypes.CDLL(path).hipGraphGetNodes(ctypes.c_void_p(graph.raw_cuda_graph()), None, ctypes.byref(count)) == 0
    assert count.value == launches
