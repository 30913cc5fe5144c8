"""One decode step of the paged int4 cache in one launch (qr_kv_quant_append_batch_decode_f16_i4): the pages must hold
what quantise-and-append stores (bit for bit), the output must be the attention over that cache (oracle, rtol / atol
1e-3) and agree with the two-launch form."""
import numpy as np
import pytest
import torch

from oracle import quarot_oracle as o
from quarot_amd import _lib
from quarot_amd.transformers import kv_cache as kv
from test_gpu_paged_kv import ATOL, F16, RTOL, bits, close, gpu, paged_case, synth_kv

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hadamard", [True, False])
@pytest.mark.parametrize("page_size,lens,heads", [(16, [1, 16, 17, 100, 700], 5), (64, [64, 1000, 129], 3), (5, [11, 1, 64], 4),
                                                  (16, [4100, 33], 8), (2048, [2048, 2047], 2)])
def test_append_and_attention_in_one_launch(page_size, lens, heads, hadamard):
    rng = np.random.default_rng(page_size + len(lens) + heads)
    layer = 1
    data, param, indptr, indices, last = paged_case(rng, heads, page_size, lens)
    B = len(lens)
    k, v = synth_kv(rng, B, heads), synth_kv(rng, B, heads)
    # special vectors: an infinity, a NaN, all zeros, a constant, the fp16 extremes
    k[0, 0, 5] = np.inf
    v[0, 1, 7] = np.nan
    k[1, 0, :] = 0
    v[1, 0, :] = F16(3.25)
    if B > 2:
        k[2, 1, 3], k[2, 1, 4] = 65504, -65504
        v[2, 0, :] = F16(1e-7)
    q = (rng.standard_normal((B, heads, 128)) * 2).astype(F16)
    tabs = (gpu(indptr), gpu(indices), gpu(last))
    # two launches
    gd2, gp2 = gpu(data), gpu(param)
    kv.quantize_append_kv_i4(gd2, gp2, *tabs, gpu(k), gpu(v), None, layer, hadamard=hadamard)
    two = torch.full((B, heads, 128), float("nan"), dtype=torch.float16, device="cuda:0")
    kv.batch_decode_i4(two, gpu(q), gd2, gp2, *tabs, layer, q_hadamard=True)
    want = o.paged_batch_decode(o.kv_hadamard(q), gd2.cpu().numpy(), gp2.cpu().numpy(), indptr, indices, last, layer)
    for hint in (0, max(lens)):
        gd1, gp1 = gpu(data), gpu(param)
        one = torch.full_like(two, float("nan"))
        kv.batch_decode_i4(one, gpu(q), gd1, gp1, *tabs, layer, max_seq_len=hint, q_hadamard=True, append=(gpu(k), gpu(v), hadamard))
        assert torch.equal(gd1, gd2), (page_size, hint)
        assert torch.equal(gp1.view(torch.int16), gp2.view(torch.int16))
        g1, g2 = one.cpu().numpy(), two.cpu().numpy()
        finite = np.isfinite(want)
        assert np.array_equal(np.isnan(g1), np.isnan(g2))
        assert close(g1[finite], want[finite]) and close(g1[finite], g2[finite])
    # without the query's Hadamard, through the C entry point
    L = _lib.lib()
    gd1, gp1 = gpu(data), gpu(param)
    gq, gk, gv = gpu(o.kv_hadamard(q)), gpu(k), gpu(v)
    one = torch.full_like(two, float("nan"))
    rc = L.qr_kv_quant_append_batch_decode_f16_i4(one.data_ptr(), gq.data_ptr(), 0, gk.data_ptr(), gv.data_ptr(), 1 if hadamard else 0,
                                                  gd1.data_ptr(), gp1.data_ptr(), tabs[0].data_ptr(), tabs[1].data_ptr(), tabs[2].data_ptr(),
                                                  gd1.shape[0], 2, layer, heads, page_size, 128, B, 0, None, 0,
                                                  torch.cuda.current_stream().cuda_stream)
    assert rc == 0 and torch.equal(gd1, gd2)
    finite = np.isfinite(want)
    assert close(one.cpu().numpy()[finite], want[finite])
    assert L.qr_kv_quant_append_batch_decode_f16_i4(one.data_ptr(), gq.data_ptr(), 0, None, gv.data_ptr(), 1, gd1.data_ptr(), gp1.data_ptr(),
                                                    tabs[0].data_ptr(), tabs[1].data_ptr(), tabs[2].data_ptr(), gd1.shape[0], 2, layer, heads,
                                                    page_size, 128, B, 0, None, 0, None) == -1
    assert L.qr_kv_quant_append_batch_decode_f16_i4(one.data_ptr(), gq.data_ptr(), 2, gk.data_ptr(), gv.data_ptr(), 1, gd1.data_ptr(),
                                                    gp1.data_ptr(), tabs[0].data_ptr(), tabs[1].data_ptr(), tabs[2].data_ptr(), gd1.shape[0],
                                                    2, layer, heads, page_size, 128, B, 0, None, 0, None) == -5


@pytest.mark.parametrize("hadamard", [True, False])
def test_the_new_tokens_codes_come_from_every_lane_of_its_wave(hadamard):
    """Keys and values that tell the positions of a vector apart (one value in turn at each of the 128), vectors of both zeros, of ranges around
    the smallest normal scale and below, and of infinities and NaNs in one place each: pages as quantise-and-append stores them."""
    rng = np.random.default_rng(3)
    heads, B, page_size = 16, 24, 16
    vecs = rng.standard_normal((B * heads, 128)).astype(F16)
    for i in range(128):
        vecs[i], vecs[i, i] = rng.standard_normal(128) * 0.05, 4.0 + i / 64
        vecs[128 + i] = (rng.standard_normal(128) * 2.0 ** -(8 + i / 8)).astype(F16)
    vecs[256:272] = np.where(rng.random((16, 128)) < 0.5, F16(0.0), F16(-0.0))
    vecs[272:288, 0] = 0
    vecs[272:288, 1:] = np.abs(vecs[272:288, 1:]) * F16(-1) ** (np.arange(16) % 2)[:, None].astype(F16)
    for i, special in enumerate([np.inf, -np.inf, np.nan, 65504]):
        for j in range(8):
            vecs[288 + 8 * i + j, 17 * j + 5] = special
    k = vecs.reshape(B, heads, 128)
    v = vecs[::-1].copy().reshape(B, heads, 128)
    lens = [int(n) for n in rng.integers(1, 70, B)]
    data, param, indptr, indices, last = paged_case(rng, heads, page_size, lens, layers=1)
    tabs, q = (gpu(indptr), gpu(indices), gpu(last)), gpu((rng.standard_normal((B, heads, 128)) * 2).astype(F16))
    gd2, gp2 = gpu(data), gpu(param)
    kv.quantize_append_kv_i4(gd2, gp2, *tabs, gpu(k), gpu(v), None, 0, hadamard=hadamard)
    for hint in (0, max(lens), 2000):                        # workgroups of different sizes, split or not
        gd1, gp1, out = gpu(data), gpu(param), torch.empty_like(q)
        kv.batch_decode_i4(out, q, gd1, gp1, *tabs, 0, max_seq_len=hint, q_hadamard=True, append=(gpu(k), gpu(v), hadamard))
        assert torch.equal(gd1, gd2), hint
        assert torch.equal(gp1.view(torch.int16), gp2.view(torch.int16)), hint


@pytest.mark.parametrize("page_size", [16, 48, 128])
def test_walks_of_more_chunks_than_a_wave_has_lanes(page_size):
    """16 waves without a split: from 16384 positions on a wave walks 64 chunks of 16 and more, whose page numbers it fetches anew; pages of
    one, three and eight chunks, one page number outside the pool among them (its positions do not count)."""
    rng = np.random.default_rng(page_size)
    heads, lens = 2, [16384, 16385, 18100, 40]
    data, param, indptr, indices, last = paged_case(rng, heads, page_size, lens, layers=1)
    q = (rng.standard_normal((len(lens), heads, 128)) * 2).astype(F16)
    tabs = (gpu(indptr), gpu(indices), gpu(last))
    k, v = synth_kv(rng, len(lens), heads), synth_kv(rng, len(lens), heads)
    gd, gp = gpu(data), gpu(param)
    one, two = torch.empty((len(lens), heads, 128), dtype=torch.float16, device="cuda:0"), torch.empty((len(lens), heads, 128), dtype=torch.float16, device="cuda:0")
    kv.batch_decode_i4(one, gpu(q), gd, gp, *tabs, 0, q_hadamard=True, append=(gpu(k), gpu(v), True))
    want = o.paged_batch_decode(o.kv_hadamard(q), gd.cpu().numpy(), gp.cpu().numpy(), indptr, indices, last, 0)
    assert close(one.cpu().numpy(), want)
    # without the middle page of the third sequence: the same as with its positions' keys infinitely far
    gone = int(indptr[2] + (indptr[3] - indptr[2]) // 2)
    holed = indices.copy()
    holed[gone] = data.shape[0]
    kv.batch_decode_i4(one, gpu(q), gd, gp, gpu(indptr), gpu(holed), gpu(last), 0, q_hadamard=True)
    kv.batch_decode_i4(two, gpu(q), gd, gp, *tabs, 0, q_hadamard=True)
    keep = [0, 1, 3]
    assert torch.equal(one[keep], two[keep]) and not torch.equal(one[2], two[2])
    dense = indices[indptr[2]:indptr[3]].tolist()
    dense.remove(int(indices[gone]))
    short = o.paged_batch_decode(o.kv_hadamard(q)[2:3], gd.cpu().numpy(), gp.cpu().numpy(), np.array([0, len(dense)], dtype=indptr.dtype),
                                 np.array(dense, dtype=indices.dtype), last[2:3], 0)
    assert close(one[2:3].cpu().numpy(), short)


def test_cache_class_holds_the_token_for_the_attention_call_and_never_shows_a_stale_cache():
    """update() of a decode step hands the token to the attention call; reading the pages, asking for the tables or
    updating again before that call stores it first; a second call of the returned callable is plain attention."""
    dev = torch.device("cuda:0")
    B, P, S, H = 3, 16, 70, 4
    g = torch.Generator(device=dev).manual_seed(1)
    rnd = lambda *shape: torch.randn(*shape, generator=g, device=dev).half()
    k0, v0 = rnd(B, S, H, 128), rnd(B, S, H, 128)
    steps = [(rnd(B, 1, H, 128), rnd(B, 1, H, 128), rnd(B, 1, H, 128)) for _ in range(4)]

    def fresh():
        c = kv.MultiLayerPagedKVCache4Bit(B, P, S + 8, dev, 1, H, 128)
        c.pages.zero_()                                      # (the pool is uninitialised memory: make untouched slots comparable)
        c.scales.zero_()
        c.update(k0, v0, 0, {})
        return c

    # reference: every step as two launches (the token stored before the attention call)
    ref, outs = fresh(), []
    for k1, v1, q1 in steps:
        f = ref.update(k1, v1, 0, {})
        ref.pages                                            # (looking at the pages stores the held token)
        assert not ref._pending
        outs.append(f(q1))
    # one launch per step
    c = fresh()
    for i, (k1, v1, q1) in enumerate(steps):
        f = c.update(k1, v1, 0, {})
        assert 0 in c._pending
        y = f(q1)
        assert not c._pending
        assert close(y.cpu().numpy(), outs[i].cpu().numpy())
        y2 = f(q1)                                            # again: plain attention over the same cache
        assert close(y2.cpu().numpy(), outs[i].cpu().numpy())
    assert torch.equal(c.pages, ref.pages) and torch.equal(c.scales.view(torch.int16), ref.scales.view(torch.int16))
    # the callable never called: the next update stores the token first
    c2 = fresh()
    for k1, v1, q1 in steps:
        c2.update(k1, v1, 0, {})
    assert torch.equal(c2.pages, ref.pages) and torch.equal(c2.scales.view(torch.int16), ref.scales.view(torch.int16))
    # asking for the tables stores it as well
    c3 = fresh()
    c3.update(*steps[0][:2], 0, {})
    specs = c3.get_cache_specs_for_flash_infer(None)
    assert not c3._pending
    c4 = fresh()
    c4.update(*steps[0][:2], 0, {})(steps[0][2])
    assert torch.equal(specs["kv_data"], c4.pages)


@pytest.mark.parametrize("page_size", [16, 5])
@pytest.mark.parametrize("B,heads", [(40, 32), (12, 24)])
def test_append_and_attention_with_many_sequence_head_pairs(B, heads, page_size):
    """Batches with 288 and 1280 (sequence, head) pairs: the entry point then forms workgroups of eight and of four
    waves; pages and outputs as in the test above."""
    rng = np.random.default_rng(B + heads + page_size)
    lens = [int(v) for v in rng.integers(1, 90, B)]
    data, param, indptr, indices, last = paged_case(rng, heads, page_size, lens, layers=1)
    k, v = synth_kv(rng, B, heads), synth_kv(rng, B, heads)
    q = (rng.standard_normal((B, heads, 128)) * 2).astype(F16)
    tabs = (gpu(indptr), gpu(indices), gpu(last))
    gd2, gp2 = gpu(data), gpu(param)
    kv.quantize_append_kv_i4(gd2, gp2, *tabs, gpu(k), gpu(v), None, 0, hadamard=True)
    two = torch.empty((B, heads, 128), dtype=torch.float16, device="cuda:0")
    kv.batch_decode_i4(two, gpu(q), gd2, gp2, *tabs, 0, q_hadamard=True)
    want = o.paged_batch_decode(o.kv_hadamard(q), gd2.cpu().numpy(), gp2.cpu().numpy(), indptr, indices, last, 0)
    gd1, gp1 = gpu(data), gpu(param)
    one = torch.full_like(two, float("nan"))
    kv.batch_decode_i4(one, gpu(q), gd1, gp1, *tabs, 0, q_hadamard=True, append=(gpu(k), gpu(v), True))
    assert torch.equal(gd1, gd2) and torch.equal(gp1.view(torch.int16), gp2.view(torch.int16))
    assert close(one.cpu().numpy(), want) and close(one.cpu().numpy(), two.cpu().numpy())


def test_one_launch_decode_step_replays_from_a_hip_graph_and_rejects_wrong_shapes():
    """The step's one launch captured into a HIP graph: replays with fresh keys, values and queries copied into the
    static buffers, eager work and synchronisation in between, store the same pages and give the same outputs as the
    eager two-launch step.  The Python mirror refuses new-token tensors of the wrong shape, dtype or layout."""
    rng = np.random.default_rng(21)
    heads, P, lens = 8, 16, [300, 17, 64]
    B = len(lens)
    data, param, indptr, indices, last = paged_case(rng, heads, P, lens, layers=1)
    tabs = (gpu(indptr), gpu(indices), gpu(last))
    gd1, gp1 = gpu(data), gpu(param)
    sk, sv, sq = (torch.zeros((B, heads, 128), dtype=torch.float16, device="cuda:0") for _ in range(3))
    out = torch.empty_like(sq)
    step = lambda: kv.batch_decode_i4(out, sq, gd1, gp1, *tabs, 0, q_hadamard=True, append=(sk, sv, True))
    step()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step()
    for i in range(4):
        k, v = gpu(synth_kv(rng, B, heads)), gpu(synth_kv(rng, B, heads))
        q = gpu((rng.standard_normal((B, heads, 128)) * 2).astype(F16))
        gd2, gp2 = gpu(data), gpu(param)
        kv.quantize_append_kv_i4(gd2, gp2, *tabs, k, v, None, 0, hadamard=True)          # eager work between the replays
        two = torch.empty_like(out)
        kv.batch_decode_i4(two, q, gd2, gp2, *tabs, 0, q_hadamard=True)
        torch.cuda.synchronize()
        sk.copy_(k); sv.copy_(v); sq.copy_(q)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(gd1, gd2) and torch.equal(gp1.view(torch.int16), gp2.view(torch.int16)), f"replay {i}"
        assert close(out.cpu().numpy(), two.cpu().numpy()), f"replay {i}"
    q = gpu(rng.standard_normal((B, heads, 128)).astype(F16))
    good = gpu(synth_kv(rng, B, heads))
    for bad in (good[:, :, :64], good.float(), good[:2].contiguous(), good.view(B, heads * 128), good.transpose(0, 1)):
        with pytest.raises(RuntimeError):
            kv.batch_decode_i4(out, q, gd1, gp1, *tabs, 0, q_hadamard=True, append=(bad, good, True))
        with pytest.raises(RuntimeError):
            kv.batch_decode_i4(out, q, gd1, gp1, *tabs, 0, q_hadamard=True, append=(good, bad, True))


@pytest.mark.parametrize("page_size,lens,heads", [(16, [2048], 32), (16, [5000, 16], 8), (24, [700, 1], 4), (128, [16000], 2)])
def test_split_sequences_merged_by_the_last_workgroup_of_the_same_launch(page_size, lens, heads):
    """A step whose sequences are split over several workgroups, with a zeroed workspace: outputs as the unsplit launch and
    the one with a separate merge give, on every call (the counters are back at zero after each), also after a shorter
    bound has used the same workspace with another split, and when the launch is replayed from a graph."""
    rng = np.random.default_rng(page_size + heads)
    data, param, indptr, indices, last = paged_case(rng, heads, page_size, lens, layers=1)
    B, L = len(lens), _lib.lib()
    tabs = (gpu(indptr), gpu(indices), gpu(last))
    gd, gp = gpu(data), gpu(param)
    bound = max(lens)
    need = max(L.qr_batch_decode_workspace_bytes(B, heads, n) for n in (bound, bound // 3 + 1))
    assert L.qr_batch_decode_workspace_bytes(B, heads, bound) > 0
    ws = torch.zeros(need, dtype=torch.uint8, device="cuda:0")
    k, v = gpu(synth_kv(rng, B, heads)), gpu(synth_kv(rng, B, heads))
    sq = torch.empty((B, heads, 128), dtype=torch.float16, device="cuda:0")
    out, ref, two = torch.empty_like(sq), torch.empty_like(sq), torch.empty_like(sq)
    step = lambda y, hint, **kw: kv.batch_decode_i4(y, sq, gd, gp, *tabs, 0, max_seq_len=hint, q_hadamard=True, append=(k, v, True), **kw)
    graph = None
    for i in range(5):
        sq.copy_(gpu((rng.standard_normal((B, heads, 128)) * 2).astype(F16)))
        step(ref, 0)
        step(two, bound)
        if i == 2:
            step(out, bound // 3 + 1, workspace=ws, counters_zero=True)       # (a bound only chooses the split)
            assert close(out.cpu().numpy(), ref.cpu().numpy())
        out.fill_(float("nan"))
        if i < 3:
            step(out, bound, workspace=ws, counters_zero=True)
        else:
            if graph is None:
                graph = torch.cuda.CUDAGraph()
                with torch.cuda.graph(graph):
                    step(out, bound, workspace=ws, counters_zero=True)
            graph.replay()
        torch.cuda.synchronize()
        assert close(out.cpu().numpy(), ref.cpu().numpy()) and close(two.cpu().numpy(), ref.cpu().numpy())
        assert int(ws[:4 * B * heads].sum()) == 0


@pytest.mark.parametrize("B,S,heads", [(4, 17, 32), (4, 64, 32), (16, 320, 32), (64, 1000, 8), (2, 2048, 40), (1, 2048, 32)])
def test_decode_attention_is_as_exact_in_every_dimension(B, S, heads):
    """Against float64 over the dequantised cache.  The kernel multiplies codes with a bias or-ed in, 1024 in the even
    dimensions and 64 in the odd ones; its fp32 sums are rounded at the biased magnitude, so an even dimension may lose up to
    sixteen times as much before the fp16 rounding.  What is left of that must not show: the share of outputs that are not the
    float64 result's nearest fp16 value is what the odd dimensions have (8 to 14 %, from the logits), within four standard
    deviations of two counts and a fifth of it."""
    rng = np.random.default_rng(B + S + heads)
    cache = kv.MultiLayerPagedKVCache4Bit(B, 16, S + 1, "cuda:0", 1, heads, 128, hadamard_dtype=None)
    cache.pages.zero_(), cache.scales.zero_()
    cache.update(*(gpu(synth_kv(rng, B * (S - 1), heads)).view(B, S - 1, heads, 128) for _ in range(2)), 0)
    q, k, v = (gpu(synth_kv(rng, B, heads)).view(B, 1, heads, 128) for _ in range(3))
    out = cache.update(k, v, 0)(q).view(B, heads, 128).double()
    pages, n = cache.pages[:, 0], (S + 15) // 16
    codes = torch.stack([pages & 15, pages >> 4], -1).flatten(-2).double()
    values = codes * cache.scales[:, 0, ..., :1].double() - cache.scales[:, 0, ..., 1:].double()      # [page, K or V, head, entry, 128]
    want = torch.empty_like(out)
    for b in range(B):
        kv2 = values[torch.arange(n, device="cuda:0") * B + b].permute(1, 2, 0, 3, 4).reshape(2, heads, n * 16, 128)[:, :, :S]
        logits = (kv2[0] * q[b, 0].double().unsqueeze(1)).sum(-1) / 128 ** 0.5
        want[b] = (torch.softmax(logits, -1).unsqueeze(-1) * kv2[1]).sum(1)
    off = out != want.half().double()
    even, odd = float(off[..., 0::2].double().mean()), float(off[..., 1::2].double().mean())
    assert odd < 0.2 and even <= 1.2 * odd + 4 * (2 * odd / (B * heads * 64)) ** 0.5, (even, odd)
    assert float((out - want).norm() / want.norm()) < 3e-4              # fp16 rounding alone: 2.1e-4


@pytest.mark.parametrize("hadamard_dtype", [torch.float16, None])
def test_a_step_whose_attention_call_raises_keeps_its_token(hadamard_dtype):
    """update() has accepted the step's key and value; a query that the attention call refuses must not lose them: the pages hold
    the token afterwards, and the call can be made again."""
    rng = np.random.default_rng(4)
    k0, v0, k, v, q = (gpu(synth_kv(rng, n, 3)).view(1, n, 3, 128) for n in (5, 5, 1, 1, 1))
    caches = [kv.MultiLayerPagedKVCache4Bit(1, 4, 8, "cuda:0", 1, 3, 128, hadamard_dtype=hadamard_dtype) for _ in range(3)]
    calls = []
    for c in caches:
        c.pages.zero_(), c.scales.zero_()
        c.update(k0, v0, 0)
        calls.append(c.update(k, v, 0))
    for bad in (q[:, :, :2].contiguous(), q[..., :64].contiguous(), q.double()):
        for call in calls[:2]:
            with pytest.raises(Exception):
                call(bad)
    assert torch.equal(calls[0](q), calls[2](q))
    for c in caches[:2]:                                                # after the repeated call, and without one
        assert torch.equal(c.pages, caches[2].pages) and torch.equal(c.scales, caches[2].scales)


@pytest.mark.parametrize("page_size,heads,B", [(16, 4, 2), (32, 8, 1), (5, 3, 2)])
def test_a_step_that_opens_a_page_reads_none_of_what_its_memory_held(page_size, heads, B):
    """The pool is uninitialised memory.  Where the new token is the first of its page, that page holds nothing valid while the
    other waves walk over the cache; what they fetch from it -- parameters that are NaNs or infinities here -- must not meet
    the sums, not even with a probability of zero."""
    rng = np.random.default_rng(page_size)
    most = 64 * page_size
    prompt = [gpu(synth_kv(rng, B * most, heads)).view(B, most, heads, 128) for _ in range(2)]
    q, k, v = (gpu(synth_kv(rng, B, heads)).view(B, 1, heads, 128) for _ in range(3))
    cache = kv.MultiLayerPagedKVCache4Bit(B, page_size, most + page_size, "cuda:0", 1, heads, 128)
    cache.update(*prompt, 0)
    pages, scales = cache.pages.clone(), cache.scales.clone()
    for length in range(page_size, most + 1, page_size):
        outs = []
        for left in (0.0, float("nan"), float("inf"), -float("inf")):
            cache.pages.copy_(pages), cache.scales.copy_(scales)
            cache.length = length
            cache.scales[length // page_size * B:] = left
            outs.append(cache.update(k, v, 0)(q))
        assert bool(torch.isfinite(outs[0]).all())
        assert all(torch.equal(y, outs[0]) for y in outs[1:]), length


def test_a_query_without_its_head_axis_is_refused():
    """[batch, 1, 128] where [batch, 1, heads, 128] is due: also where the cache has one head and the elements would fit."""
    cache = kv.MultiLayerPagedKVCache4Bit(2, 16, 16, "cuda:0", 1, 1, 128)
    k, v, q = (torch.randn(2, 1, 1, 128, device="cuda:0").half() for _ in range(3))
    cache.update(k, v, 0)
    call = cache.update(k, v, 0)
    with pytest.raises(ValueError):
        call(q[:, :, 0])
    assert call(q).shape == q.shape
