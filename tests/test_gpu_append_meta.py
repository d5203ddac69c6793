"""Appends whose page lists sit at the edges of what travels in a kernel's arguments (256 and 896 ints; past
that a batch goes through a staging buffer, a single append by copies), one call per sequence and batched,
and on more streams than are tracked: stored bytes bit-exact, decode within tolerance, device table and
lengths as the host's.
"""

from __future__ import annotations

import numpy as np
import pytest

import pa_amd
from helpers import D, TOL, d2h, run_cache_case

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("gpu_device")]


@pytest.mark.parametrize("batched", [False, True], ids=["per_slot", "batched"])
@pytest.mark.parametrize("fp8", [False, True], ids=["fp16", "fp8"])
@pytest.mark.parametrize("lens", [[83], [84], [297], [298], [41, 42], [148, 147], [1000, 3]], ids=str)
def test_meta_sizes(fp8, batched, lens):
    """With one token per page a sequence of n new tokens takes 3 n + 5 ints of metadata (a batch of two
    10 + 3 (n0 + n1)): 254, 257, 896, 899, 259, 895 and 3019."""
    err, _, _ = run_cache_case(fp8, 8, 2, 1, lens, shuffle_seed=5, batched=batched)
    assert err <= TOL


@pytest.mark.parametrize("n,prefix", [(112, 0), (113, 0), (149, 1), (150, 1), (128, 3)], ids=str)
def test_decode_step_meta_sizes(n, prefix):
    """One token to each of n sequences: 8 n ints of metadata where each begins a page (896 and 904), 6 n where none
    does (894 and 900); the last with every sequence at the end of a page, so that 128 new entries go along (1024)."""
    import torch
    P, hkv = (1, 2) if prefix == 0 else (3 if prefix == 3 else 4, 2)
    cache = pa_amd.PagedKVCache(2 * n + 5, P, hkv, D, n, 4)
    cache.shuffle_free_pages(3)
    slots = [cache.admit() for _ in range(n)]
    x = torch.randn((n * max(prefix, 1), hkv, D), dtype=torch.float16, device="cuda")
    y = torch.randn((n, hkv, D), dtype=torch.float16, device="cuda")
    if prefix:
        assert cache.append_batch(slots, [prefix] * n, x, x, 0)
    assert cache.append_batch(slots, [1] * n, y, x, 0)
    p = cache.params()
    assert list(d2h(int(p.seq_lens), 4 * n, np.int32)) == [prefix + 1] * n
    table = d2h(int(p.block_table), 16 * n, np.int32).reshape(n, 4)
    k = d2h(int(p.k_cache), (2 * n + 5) * hkv * P * D * 2, np.uint16).reshape(-1, hkv, P, D)
    want = y.view(torch.int16).cpu().numpy().view(np.uint16)
    for i, s in enumerate(slots):
        pages = cache.block_table(s)
        assert list(table[s, :len(pages)]) == list(pages) and len(pages) == prefix // P + 1
        assert np.array_equal(k[pages[prefix // P], :, prefix % P], want[i])
    cache.close()


def test_appends_on_many_streams_then_release():
    """Ten streams append to a sequence each (more than the cache tracks at once); device lengths and tables are
    the host's, and a released slot's length is zero on the device."""
    import torch
    n, P, hkv = 10, 4, 2
    cache = pa_amd.PagedKVCache(400, P, hkv, D, n, 40)
    g = torch.Generator(device="cuda").manual_seed(1)
    slots = [cache.admit() for _ in range(n)]
    streams = [torch.cuda.Stream() for _ in range(n)]
    x = torch.randn((50, hkv, D), dtype=torch.float16, device="cuda", generator=g)
    torch.cuda.synchronize()
    for i, (s, st) in enumerate(zip(slots, streams)):
        assert cache.append_batch([s], [20 + i], x, x, st)
    cache.release(slots[3])
    torch.cuda.synchronize()
    p = cache.params()
    lens = d2h(p.seq_lens, 4 * n, np.int32)
    assert list(lens) == [0 if i == 3 else 20 + i for i in range(n)]
    table = d2h(p.block_table, 4 * n * 40, np.int32).reshape(n, 40)
    for i, s in enumerate(slots):
        t = cache.block_table(s)
        assert list(table[i, :len(t)]) == list(t)
    cache.close()


def test_releases_on_the_null_stream_then_appends_on_another():
    """Releases queued on the null stream (behind a long kernel there) and slots re-admitted at once, their
    appends on a side stream: the new lengths stand, on the device too."""
    import torch
    P, hkv = 4, 2
    cache = pa_amd.PagedKVCache(64, P, hkv, D, 3, 20)
    x = torch.randn((50, hkv, D), dtype=torch.float16, device="cuda")
    for i in range(3):
        assert cache.append_batch([cache.admit()], [10 + i], x, x, 0)
    big = torch.randn((4096, 4096), device="cuda")
    torch.cuda.synchronize()
    for _ in range(20):
        big = big @ big
        big = big / big.norm()
    cache.release(0)
    cache.release(2)
    side = torch.cuda.Stream()
    a, b = cache.admit(), cache.admit()
    assert (a, b) == (0, 2)
    assert cache.append_batch([a, b], [7, 9], x, x, side)
    torch.cuda.synchronize()
    assert list(d2h(cache.params().seq_lens, 12, np.int32)) == [7, 11, 9]
    cache.release(1)   # now with another stream seen: zero when the call returns
    assert list(d2h(cache.params().seq_lens, 12, np.int32)) == [7, 0, 9]
    cache.close()


def test_uploads_beyond_the_staging_buffers_and_in_a_graph():
    """More plan uploads than staging buffers queued without a wait, each decode under its own plan; and an
    upload captured into a graph with its decode, replayed between eager uploads of other plans."""
    import torch
    from helpers import paged_inputs
    lens_of = [[64 * (i + 1), 5, 300 + i] for i in range(20)]
    q, k, v, table, ks, vs = paged_inputs(3, [2000] * 3, 8, 2, 16, False, seed=3)
    dplan = pa_amd.DevicePlan()

    def decode(lens, out, stream=None, plan=None):
        dplan.upload(plan or pa_amd.make_plan(pa_amd.FP16, lens, 8, 2, D), 4, D, stream)
        p = pa_amd.DecodeParams()
        p.q, p.k_cache, p.v_cache, p.block_table = q.data_ptr(), k.data_ptr(), v.data_ptr(), table.data_ptr()
        p.out, p.block_table_stride = out.data_ptr(), table.size(1)
        p.batch, p.num_q_heads, p.num_kv_heads, p.head_dim, p.page_size = 3, 8, 2, D, 16
        p.sm_scale, p.k_scale, p.v_scale = pa_amd.sm_scale(D), ks, vs
        dplan.bind(p)
        pa_amd.paged_decode(pa_amd.FP16, p, stream)

    largest = torch.empty_like(q)
    decode([2000] * 3, largest)                      # sizes the plan's device arrays
    plans = [pa_amd.make_plan(pa_amd.FP16, lens, 8, 2, D) for lens in lens_of]
    alone = []
    for lens in lens_of:
        alone.append(torch.empty_like(q))
        decode(lens, alone[-1])
        torch.cuda.synchronize()
    outs = [torch.empty_like(q) for _ in lens_of]
    for lens, o, pl in zip(lens_of, outs, plans):
        decode(lens, o, plan=pl)
    torch.cuda.synchronize()
    assert all(torch.equal(a, o) for a, o in zip(alone, outs))
    side, graph, out = torch.cuda.Stream(), torch.cuda.CUDAGraph(), torch.empty_like(q)
    with torch.cuda.stream(side):
        with torch.cuda.graph(graph, stream=side):
            decode(lens_of[7], out, torch.cuda.current_stream(), plans[7])
        for rep in range(3):
            out.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, alone[7])
            for i in range(12):
                decode(lens_of[i], outs[i], side, plans[i])
            torch.cuda.synchronize()
            assert all(torch.equal(alone[i], outs[i]) for i in range(12))


def test_uploads_behind_long_work():
    """More uploads than staging buffers on a stream that is busy for tens of milliseconds: the call waits, asking
    the stream, and every decode runs under its own plan."""
    import torch
    from helpers import paged_inputs
    lens_of = [[40 * (i + 1), 5, 300 + i] for i in range(12)]
    q, k, v, table, ks, vs = paged_inputs(3, [600] * 3, 8, 2, 16, False, seed=3)
    side, dplan = torch.cuda.Stream(), pa_amd.DevicePlan()
    plans = [pa_amd.make_plan(pa_amd.FP16, lens, 8, 2, D) for lens in lens_of]
    big = torch.randn((8192, 8192), device="cuda")

    def decode(i, out):
        dplan.upload(plans[i], 4, D, side)
        p = pa_amd.DecodeParams()
        p.q, p.k_cache, p.v_cache, p.block_table = q.data_ptr(), k.data_ptr(), v.data_ptr(), table.data_ptr()
        p.out, p.block_table_stride = out.data_ptr(), table.size(1)
        p.batch, p.num_q_heads, p.num_kv_heads, p.head_dim, p.page_size = 3, 8, 2, D, 16
        p.sm_scale, p.k_scale, p.v_scale = pa_amd.sm_scale(D), ks, vs
        dplan.bind(p)
        pa_amd.paged_decode(pa_amd.FP16, p, side)

    alone = [torch.empty_like(q) for _ in lens_of]
    outs = [torch.empty_like(q) for _ in lens_of]
    torch.cuda.synchronize()
    for i, o in enumerate(alone):
        decode(i, o)
        torch.cuda.synchronize()
    with torch.cuda.stream(side):
        for _ in range(6):
            big = big @ big
            big = big / big.norm()
        for i, o in enumerate(outs):
            decode(i, o)
    torch.cuda.synchronize()
    assert all(torch.equal(a, o) for a, o in zip(alone, outs))


@pytest.mark.parametrize("n", [7, 400], ids=["in_arguments", "staged"])
def test_captured_append_after_a_release_on_the_null_stream(n):
    """A release queued on the null stream, then an append to the same slot captured on another: the wait for the
    release leaves the capture whole, and every replay stores the tokens then in the inputs, with the page list of
    its own batch, whatever appends ran in between (400 one-token pages are 1205 ints of metadata: past the kernel's
    arguments). Releases after it find no event that only a graph has."""
    import torch
    hkv, rows = 2, 2000
    cache = pa_amd.PagedKVCache(rows, 1, hkv, D, 8, 420)
    x, y = (torch.randn((420, hkv, D), dtype=torch.float16, device="cuda") for _ in range(2))
    first = cache.admit()
    assert cache.append_batch([first], [3], x, x, 0)
    assert cache.append_batch([cache.admit()], [400], x, x, 0)   # staging buffers are made outside captures
    graph, tokens, side = torch.cuda.CUDAGraph(), x.clone(), torch.cuda.Stream()
    with torch.cuda.graph(graph, stream=side):
        cache.release(first)
        slot = cache.admit()
        assert slot == first
        assert cache.append_batch([slot], [n], tokens, tokens, torch.cuda.current_stream())
    p = cache.params()
    pages = cache.block_table(slot)
    assert cache.seq_len(slot) == n and len(pages) == n

    def kept():
        from helpers import d2h
        k = d2h(int(p.k_cache), rows * hkv * D * 2, np.uint16).reshape(rows, hkv, D)
        return k[list(pages)]

    for rep in range(3):
        tokens.copy_(x if rep % 2 else y)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(kept(), tokens[:n].view(torch.int16).cpu().numpy().view(np.uint16))
        assert int(d2h(p.seq_lens, 4 * 8, np.int32)[slot]) == n
        other = cache.admit()          # eager appends of other shapes between the replays
        assert cache.append_batch([other], [390 + rep], y, y, side)
        torch.cuda.synchronize()
        assert int(d2h(p.seq_lens, 4 * 8, np.int32)[other]) == 390 + rep
        cache.release(other)
        assert int(d2h(p.seq_lens, 4 * 8, np.int32)[other]) == 0
    cache.close()
