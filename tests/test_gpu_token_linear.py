"""One or two tokens behind a Hadamard of 64 or 128 values and a table of order 33 and more: qr_quantized_linear_f16 runs the front
and the dot products in one kernel in which every workgroup transforms the rows itself.  Its output must carry the bits of
the two-launch chain (same codes, same scale, same sums, same epilogue)."""
import ctypes
import math

import numpy as np
import pytest
import torch

import quarot_amd
from quarot_amd import _lib
from oracle import quarot_oracle as o

pytestmark = pytest.mark.gpu


def _chain(x, w, sw, b, hadK, K, clip):
    p = quarot_amd.hadamard_quantize(x, hadK, K, clip_ratio=clip)
    return quarot_amd.linear_i4(p.quantized_x, p.scales_x, w, sw, b)


def _weights(n, N, bias, gen):
    w = torch.randint(0, 256, (N, n // 2), dtype=torch.uint8, device="cuda", generator=gen)
    sw = (torch.rand(N, 1, device="cuda", generator=gen) * 0.01 + 0.001).half()
    return w, sw, torch.randn(N, device="cuda", generator=gen).half() if bias else None


@pytest.mark.parametrize("M", [1, 2, 3])
# 64 x 172 (sign words and table), 64 x 156 / 140 / 108, 128 x 108 / 60 / 52 / 40 / 36; a power of two and a short table stay with the chain
@pytest.mark.parametrize("n", [11008, 9984, 8960, 6912, 13824, 7680, 6656, 5120, 4608, 4096, 1792])
def test_one_token_behind_a_short_factor_in_one_launch(n, M):
    gen = torch.Generator(device="cuda").manual_seed(n + M)
    table, K = quarot_amd.functional.hadamard.get_hadK(n)
    hadK = table.to("cuda").half() if table is not None else None
    for N, bias, clip in [(1, False, 1.0), (17, True, 0.9), (4096, False, 1.0), (4097, True, 1.0), (9001, True, 0.8)]:
        w, sw, b = _weights(n, N, bias, gen)
        x = torch.randn(M, n, device="cuda", generator=gen)
        x[:, torch.randperm(n, generator=gen, device="cuda")[:n // 100]] *= 20
        x[M - 1] *= 0.21
        x = x.half()
        got = quarot_amd.quantized_linear(x, w, sw, b, hadK, K, clip_ratio=clip)
        assert got.shape == (M, N) and torch.equal(got, _chain(x, w, sw, b, hadK, K, clip)), N
        if N == 17:                                         # the oracle's layer on the kernel's own transformed row
            xq, xs = o.quantizer(quarot_amd.nn.OnlineHadamard(n).cuda()(x).cpu().numpy(), clip)
            ref = o.linear4bit(xq, xs, w.cpu().numpy(), sw.cpu().numpy(), b.cpu().numpy())
            assert np.array_equal(got.cpu().numpy().view(np.uint16), ref.view(np.uint16))
    w, sw, _ = _weights(n, 333, False, gen)
    for value, scale in [(0.0, 0.0), (float("inf"), 1.0), (float("nan"), 1.0), (1.0, 20000.0), (1.0, 1e-6)]:
        x = torch.randn(M, n, device="cuda", generator=gen) * (scale if value == 1.0 else 1.0)
        x = x.clamp(-60000, 60000).half()
        x[M - 1] = 0 if value == 0.0 else x[M - 1]
        x[M - 1, 5] = value if value != 1.0 else x[M - 1, 5]
        got, want = quarot_amd.quantized_linear(x, w, sw, None, hadK, K), _chain(x, w, sw, None, hadK, K, 1.0)
        assert torch.equal(got.view(torch.int16), want.view(torch.int16)), (value, scale)


def test_output_that_is_not_8_byte_aligned_is_refused():
    gen = torch.Generator(device="cuda").manual_seed(1)
    n, N = 11008, 40
    table, K = quarot_amd.functional.hadamard.get_hadK(n)
    hadK = table.to("cuda").half()
    w, sw, _ = _weights(n, N, False, gen)
    x = torch.randn(1, n, device="cuda", generator=gen).half()
    lib, size = _lib.lib(), _lib.lib().qr_quantized_linear_workspace_bytes(1, N, n)
    work, y = torch.empty(size, dtype=torch.uint8, device="cuda"), torch.full((N + 8,), 7, dtype=torch.float16, device="cuda")
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    call = lambda out: lib.qr_quantized_linear_f16(p(x), 1, n, K, p(hadK), 0, 1 / math.sqrt(n), 1.0, p(w), p(sw), None, N, p(out), p(work), size, None)
    assert call(y[1:]) == call(y[2:]) == -4                 # QR_E_ALIGN
    assert bool((y == 7).all())
    assert call(y[4:]) == 0 and bool((y[:4] == 7).all()) and bool((y[4 + N:] == 7).all())
