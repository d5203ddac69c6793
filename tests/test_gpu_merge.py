"""The split kernel's merges where a block holds many split rows, a run of more
than eight slots, or two rows that it is the last block of: against the merge
kernel on the same plan and the fp32 oracle, and bitwise equal from run to run.
"""

from __future__ import annotations

import ctypes

import numpy as np
import pytest

import oracle
import pa_amd
from helpers import D, TOL, paged_inputs

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("gpu_device")]


def _check(fp8, lens, group, hkv, handle, mode, page=16, repeats=6):
    import torch
    hq = hkv * group
    dt = pa_amd.FP8_E4M3 if fp8 else pa_amd.FP16
    q, k, v, table, ks, vs = paged_inputs(len(lens), lens, hq, hkv, page, fp8, seed=7 * group + len(lens))
    dplan = pa_amd.DevicePlan()
    pa_amd._lib.call("pa_device_plan_upload", dplan._h, handle, group, D, None)
    outs = []
    for rep in range(repeats + 1):
        p = pa_amd.DecodeParams()
        p.q, p.k_cache, p.v_cache, p.block_table = q.data_ptr(), k.data_ptr(), v.data_ptr(), table.data_ptr()
        out = torch.full_like(q, float("nan"))
        p.out = out.data_ptr()
        p.block_table_stride = table.size(1)
        p.batch, p.num_q_heads, p.num_kv_heads, p.head_dim, p.page_size = len(lens), hq, hkv, D, page
        p.sm_scale, p.k_scale, p.v_scale = pa_amd.sm_scale(D), ks, vs
        dplan.bind(p)
        assert p.block_merge == mode and p.needs_merge == (mode == 3)
        if rep == repeats:
            p.block_merge, p.needs_merge = 0, 1   # the merge kernel on the same plan
        pa_amd.paged_decode(dt, p)
        torch.cuda.synchronize()
        outs.append(out)
    for o in outs[1:repeats]:
        assert torch.equal(outs[0].view(torch.int16), o.view(torch.int16))
    kb = k.view(torch.uint8).cpu().numpy() if fp8 else k.view(torch.int16).cpu().numpy().view(np.uint16)
    vb = v.view(torch.uint8).cpu().numpy() if fp8 else v.view(torch.int16).cpu().numpy().view(np.uint16)
    ref = oracle.paged_decode(dt, q.view(torch.int16).cpu().numpy().view(np.uint16), kb, vb, table.cpu().numpy(),
                              np.asarray(lens, np.int32), hq, hkv, D, page, ks, vs, threads=16)
    for o in (outs[0], outs[-1]):
        assert float(np.max(np.abs(o.float().cpu().numpy() - ref))) < TOL
    # Both merges average the same fp32 partials; two fp16 roundings of values below 4 differ by at most 2^-9.
    assert float((outs[0].float() - outs[-1].float()).abs().max()) <= 2.0 ** -9


def _plan(fp8, lens, group, hkv, ctas):
    return pa_amd.make_plan(pa_amd.FP8_E4M3 if fp8 else pa_amd.FP16, lens, hkv * group, hkv, D, ctas)


@pytest.mark.parametrize("group", [1, 2, 4, 8])
@pytest.mark.parametrize("fp8", [False, True], ids=["fp16", "fp8"])
def test_many_split_rows_in_a_block(fp8, group):
    """Rows of 2 to 5 tiles over units of 3: most blocks hold 5 to 9 runs, the first and last of them
    continuing in the neighbouring blocks, so a block is often the last of two rows at once."""
    tile = 32 if fp8 else 16
    rng = np.random.default_rng(3)
    lens = [int(x) for x in rng.integers(tile + 1, 5 * tile, size=40)]
    total = sum(-(-n // tile) for n in lens) * 8
    plan = _plan(fp8, lens, group, 8, -(-total // 3))
    _check(fp8, lens, group, 8, plan.handle.value, 2)


@pytest.mark.parametrize("lens,ctas", [([100], 28), ([129], 36), ([16 * 17] * 3, 204), ([528], 0),
                                       ([5000, 1, 700, 16, 17], 96)],
                         ids=["7_tiles", "9_tiles", "17_tiles", "33_tiles", "mixed"])
def test_short_rows_across_blocks(lens, ctas):
    """Rows that straddle two or three blocks because their tiles are no multiple of a block's units."""
    plan = _plan(False, lens, 4, 8, ctas)
    _check(False, lens, 4, 8, plan.handle.value, 2)


def _device_plan_arrays(p, items):
    from helpers import d2h
    cta = d2h(int(p.cta_seg_begin), 4 * (p.num_ctas + 1), np.int32)
    item = d2h(int(p.item_seg_begin), 4 * (items + 1), np.int32)
    return cta, item, d2h(int(p.segments), 16 * int(cta[-1]), np.int32).reshape(-1, 4)


def test_decode_static_refuses_the_same_plans():
    """A plan whose partials exceed the static workspace keeps its rows across blocks, and is refused there."""
    import torch
    lens = [17 + (i * 37) % 48 for i in range(1024)]
    q, k, v, table, ks, vs = paged_inputs(len(lens), lens, 64, 8, 16, False, seed=5)
    plan = _plan(False, lens, 8, 8, 0)
    assert plan.merge_mode == 2 and len(plan.segments) * 8 * (D + 1) * 4 > 32 << 20
    dplan = pa_amd.DevicePlan()
    dplan.upload(plan, 8, D)
    p = pa_amd.DecodeParams()
    dplan.bind(p)
    out = torch.empty_like(q)
    p.q, p.k_cache, p.v_cache, p.block_table = q.data_ptr(), k.data_ptr(), v.data_ptr(), table.data_ptr()
    p.out, p.block_table_stride = out.data_ptr(), table.size(1)
    p.batch, p.num_q_heads, p.num_kv_heads, p.head_dim, p.page_size = len(lens), 64, 8, D, 16
    p.sm_scale, p.k_scale, p.v_scale = pa_amd.sm_scale(D), ks, vs
    assert p.block_merge == 2
    lib = pa_amd._lib.load()
    assert lib.pa_decode_static(pa_amd.FP16, ctypes.byref(p), p.num_segments, None) == pa_amd._lib.PA_ERR_LENGTH


@pytest.mark.parametrize("lens,fp8,group,hkv", [
    ([48] * 165, False, 4, 8),
    ([192] * 203, True, 4, 8),
    ([1344] * 248, True, 4, 8),
    ([112] * 385, False, 4, 4),
    ([200] * 32, False, 4, 8),
    ([200], False, 8, 8),
    ([33, 17, 48], True, 1, 8),
], ids=["165x48", "203x192_fp8", "248x1344_fp8", "385x112", "32x200", "row", "ragged"])
def test_decode_static_takes_grouped_plans(lens, fp8, group, hkv):
    """Plans whose host copy has split rows, grouped inside blocks or not: the allocation-free entry point takes
    them and gives what the plain one gives, and the oracle."""
    import torch
    hq, dt = hkv * group, pa_amd.FP8_E4M3 if fp8 else pa_amd.FP16
    q, k, v, table, ks, vs = paged_inputs(len(lens), lens, hq, hkv, 16, fp8, seed=len(lens))
    plan = _plan(fp8, lens, group, hkv, 0)
    dplan = pa_amd.DevicePlan()
    dplan.upload(plan, group, D)
    outs = []
    for static in (False, True):
        p = pa_amd.DecodeParams()
        out = torch.full_like(q, float("nan"))
        p.q, p.k_cache, p.v_cache, p.block_table = q.data_ptr(), k.data_ptr(), v.data_ptr(), table.data_ptr()
        p.out, p.block_table_stride = out.data_ptr(), table.size(1)
        p.batch, p.num_q_heads, p.num_kv_heads, p.head_dim, p.page_size = len(lens), hq, hkv, D, 16
        p.sm_scale, p.k_scale, p.v_scale = pa_amd.sm_scale(D), ks, vs
        dplan.bind(p)
        assert p.num_segments == len(plan.segments)
        if static:
            pa_amd._lib.call("pa_decode_static", dt, ctypes.byref(p), p.num_segments, None)
        else:
            pa_amd.paged_decode(dt, p)
        torch.cuda.synchronize()
        outs.append(out)
    assert torch.equal(outs[0].view(torch.int16), outs[1].view(torch.int16))
    kb = k.view(torch.uint8).cpu().numpy() if fp8 else k.view(torch.int16).cpu().numpy().view(np.uint16)
    vb = v.view(torch.uint8).cpu().numpy() if fp8 else v.view(torch.int16).cpu().numpy().view(np.uint16)
    ref = oracle.paged_decode(dt, q.view(torch.int16).cpu().numpy().view(np.uint16), kb, vb, table.cpu().numpy(),
                              np.asarray(lens, np.int32), hq, hkv, D, 16, ks, vs, threads=16)
    assert float(np.max(np.abs(outs[1].float().cpu().numpy() - ref))) < TOL


@pytest.mark.parametrize("lens,fp8,group,hkv", [
    ([200], False, 4, 8),                          # one item per block, fewer blocks than the chip has
    ([33], False, 2, 8),                           # three tiles per item
    ([200] * 32, False, 4, 8),                     # as many items as blocks
    ([1100] * 32, True, 8, 8),
    ([10, 33, 300, 1, 64, 250, 17, 129], True, 1, 8),
    ([200] * 64, False, 4, 8),                     # two items per block
    ([1, 9, 33, 20, 16, 31, 2, 40, 17] * 6, False, 8, 8),           # many short items per block
    ([95, 161, 128] * 40, True, 4, 4),
], ids=["row", "three_tiles", "full", "g8", "ragged", "packed", "short", "fp8_packed"])
def test_items_kept_inside_blocks(lens, fp8, group, hkv):
    """Plans of make_plan's own grid whose items would straddle blocks run on other units: every block of 8 units
    holds whole items, an item's segments lie in consecutive units, a unit's split ones are its first and last, and
    the decode matches the oracle and the merge kernel. The segments stay the plan's own (block_merge 1), or, where
    those are single tiles, runs of two or three of them (block_merge 4)."""
    plan = _plan(fp8, lens, group, hkv, 0)
    assert plan.merge_mode == 2
    tile, host, items = 32 if fp8 else 16, np.asarray(plan.segments), len(lens) * hkv
    single = bool(np.all(host[:, 3] - host[:, 2] <= tile))
    dplan = pa_amd.DevicePlan()
    dplan.upload(plan, group, D)
    p = pa_amd.DecodeParams()
    dplan.bind(p)
    assert p.block_merge == (4 if single else 1)
    assert p.num_segments == len(host) and p.num_ctas % 8 == 0
    cta, item, seg = _device_plan_arrays(p, items)
    if single:
        assert np.all(seg[:, 3] - seg[:, 2] <= 3 * tile)
    else:
        assert np.array_equal(seg, host)
    assert cta[0] == 0 and cta[-1] == len(seg) and np.all(np.diff(cta) >= 0)
    unit = np.repeat(np.arange(p.num_ctas), np.diff(cta))
    split = np.repeat(np.diff(item) > 1, np.diff(item))
    for i in range(items):
        rows = seg[item[i]:item[i + 1]]
        assert len(rows) and np.all(rows[:, 0] == i // hkv) and np.all(rows[:, 1] == i % hkv)
        assert rows[0, 2] == 0 and rows[-1, 3] == lens[i // hkv] and np.array_equal(rows[1:, 2], rows[:-1, 3])
        assert np.all(rows[:, 2] % tile == 0)
        u = unit[item[i]:item[i + 1]]
        assert u[0] // 8 == u[-1] // 8 and np.array_equal(u, np.arange(u[0], u[0] + len(u)))
    for u in range(p.num_ctas):
        assert not split[cta[u] + 1:cta[u + 1] - 1].any()
    _check(fp8, lens, group, hkv, plan.handle.value, p.block_merge, repeats=2)


@pytest.mark.parametrize("lens,fp8,group,hkv", [
    ([200], False, 4, 8),                          # 13 tiles in 8 units
    ([199, 250, 33], True, 8, 8),
    ([200] * 32, False, 4, 8),
    ([1, 9, 33, 20, 16, 31, 2, 40, 17] * 6, False, 2, 8),
], ids=["row", "ragged", "full", "short"])
def test_grouping_keeps_the_partials(lens, fp8, group, hkv):
    """Inside blocks or across them, the decode averages the same partials. With partials equal bit for bit, two
    fp32 averages of at most 16 of them (weights in [0, 1], values below 4.5) differ by at most 16 * 2^-24 * 4.5,
    so two fp16 results differ by one rounding at most, and only where the average lies that near to the middle of
    two fp16 values: 2 * 4.3e-6 of the spacing 2^-13 of values above 1/8, under 2^-3 of the results at worst."""
    import torch
    hq, dt = hkv * group, pa_amd.FP8_E4M3 if fp8 else pa_amd.FP16
    q, k, v, table, ks, vs = paged_inputs(len(lens), lens, hq, hkv, 16, fp8, seed=11)
    plan = _plan(fp8, lens, group, hkv, 0)
    # The same units behind an empty one: no cut that make_plan gives, so it runs as it is.
    cta = np.concatenate([[0], plan.cta_seg_begin]).astype(np.int32)
    seg, item = np.ascontiguousarray(plan.segments), np.ascontiguousarray(plan.item_seg_begin)
    h = ctypes.c_void_p()
    pa_amd._lib.call("pa_plan_create", len(cta) - 1, plan.tile, seg.ctypes.data, len(seg), cta.ctypes.data,
                     item.ctypes.data, len(item) - 1, hkv, ctypes.byref(h))
    outs = []
    try:
        for handle, modes in ((plan.handle.value, (1, 4)), (h.value, (2,))):
            dplan = pa_amd.DevicePlan()
            pa_amd._lib.call("pa_device_plan_upload", dplan._h, handle, group, D, None)
            p = pa_amd.DecodeParams()
            out = torch.empty_like(q)
            p.q, p.k_cache, p.v_cache, p.block_table = q.data_ptr(), k.data_ptr(), v.data_ptr(), table.data_ptr()
            p.out, p.block_table_stride = out.data_ptr(), table.size(1)
            p.batch, p.num_q_heads, p.num_kv_heads, p.head_dim, p.page_size = len(lens), hq, hkv, D, 16
            p.sm_scale, p.k_scale, p.v_scale = pa_amd.sm_scale(D), ks, vs
            dplan.bind(p)
            assert p.block_merge in modes
            pa_amd.paged_decode(dt, p)
            torch.cuda.synchronize()
            outs.append(out.float())
    finally:
        pa_amd._lib.load().pa_plan_destroy(h.value)
    apart = (outs[0] - outs[1]).abs()
    assert float(apart.max()) <= 2.0 ** -9
    assert float((apart > 0).float().mean()) < 2.0 ** -3


@pytest.mark.parametrize("factors", [[60.0, 0.1], [0.1, 60.0], [60.0, 30.0, 1.0, 0.0], [0.0]], ids=str)
def test_joined_tiles_far_apart(factors):
    """Tiles of one segment whose largest scores lie hundreds of powers of two apart, in either order, and tiles of
    equal scores: each is scored against its own maximum or, far below, counts nothing; finite, and as across blocks."""
    import torch
    lens, group, hkv, hq = [200], 4, 8, 32
    q, k, v, table, ks, vs = paged_inputs(1, lens, hq, hkv, 16, False, seed=23)
    for j, page in enumerate(table[0].tolist()[:13]):
        k[page] *= factors[j % len(factors)]
    plan = _plan(False, lens, group, hkv, 0)
    asked = _plan(False, lens, group, hkv, plan.num_ctas)   # the same cut, on its own units
    outs = []
    for pl, mode in ((plan, 4), (asked, 2)):
        dplan = pa_amd.DevicePlan()
        dplan.upload(pl, group, D)
        p = pa_amd.DecodeParams()
        out = torch.full_like(q, float("nan"))
        p.q, p.k_cache, p.v_cache, p.block_table = q.data_ptr(), k.data_ptr(), v.data_ptr(), table.data_ptr()
        p.out, p.block_table_stride = out.data_ptr(), table.size(1)
        p.batch, p.num_q_heads, p.num_kv_heads, p.head_dim, p.page_size = 1, hq, hkv, D, 16
        p.sm_scale, p.k_scale, p.v_scale = pa_amd.sm_scale(D), ks, vs
        dplan.bind(p)
        assert p.block_merge == mode
        pa_amd.paged_decode(pa_amd.FP16, p)
        torch.cuda.synchronize()
        outs.append(out.float())
    assert torch.isfinite(outs[0]).all()
    # Two fp16 roundings of fp32 averages of the same partials, of values below 4.5.
    assert float((outs[0] - outs[1]).abs().max()) <= 2.0 ** -8
    kb, vb = (x.view(torch.int16).cpu().numpy().view(np.uint16) for x in (k, v))
    ref = oracle.paged_decode(pa_amd.FP16, q.view(torch.int16).cpu().numpy().view(np.uint16), kb, vb,
                              table.cpu().numpy(), np.asarray(lens, np.int32), hq, hkv, D, 16, ks, vs, threads=16)
    # Scores of several hundred carry the rounding of their fp32 sums (2^-24 of sums below 2^13: 2^-11 in the
    # exponent, so 2^-11 of a weight) besides what the ordinary cases have.
    assert float(np.max(np.abs(outs[0].cpu().numpy() - ref))) < TOL + 4.5 * 2.0 ** -11


def test_another_grid_is_left_as_it_is():
    """A caller's grid, and rows that are cheaper across blocks, keep the host plan's arrays."""
    for lens, ctas in (([200] * 32, 512), ([500], 0), ([300, 1000, 450, 700] * 8, 0),
                       ([100, 150, 200, 130, 170, 110, 190, 120] * 16, 0),
                       ([48], 24), ([200], 104), ([200] * 32, 2048)):   # as many tiles per unit as without a grid
        plan = _plan(False, lens, 4, 8, ctas)
        assert plan.merge_mode == 2
        dplan = pa_amd.DevicePlan()
        dplan.upload(plan, 4, D)
        p = pa_amd.DecodeParams()
        dplan.bind(p)
        assert p.block_merge == 2 and p.num_ctas == plan.num_ctas
        cta, item, seg = _device_plan_arrays(p, len(lens) * 8)
        assert np.array_equal(seg, plan.segments) and np.array_equal(cta, plan.cta_seg_begin)
        assert np.array_equal(item, plan.item_seg_begin)


@pytest.mark.parametrize("group", [1, 4, 8])
def test_run_of_sixteen_slots(group):
    """A caller's plan that gives every unit of a block two segments of one row: 16 slots in one run."""
    segs = np.array([[0, 0, 16 * i, 16 * i + 16] for i in range(16)] + [[1, 0, 0, 16], [1, 0, 16, 29]], np.int32)
    cta = np.array([0, 2, 4, 6, 8, 10, 12, 14, 16, 17, 18], np.int32)
    item = np.array([0, 16, 18], np.int32)
    h = ctypes.c_void_p()
    pa_amd._lib.call("pa_plan_create", 10, 16, segs.ctypes.data, len(segs), cta.ctypes.data, item.ctypes.data, 2, 1,
                     ctypes.byref(h))
    try:
        _check(False, [256, 29], group, 1, h.value, 1)
    finally:
        pa_amd._lib.load().pa_plan_destroy(h.value)


@pytest.mark.parametrize("lens,ctas,group,hkv", [
    ([4096], 0, 4, 8),                          # one tile per unit, 32 blocks per row
    ([131072], 0, 1, 1),                        # one query head, 256 blocks
    ([131072 - 7], 0, 8, 1),
    ([30000, 17, 1, 1100, 9000], 0, 2, 8),      # rows inside a block, over a few, over many
    ([2048, 2048], 0, 8, 8),                    # 16 blocks
    ([700, 5000], 700, 4, 2),
], ids=["one_tile", "one_head", "g8", "ragged", "two_rows", "few_units"])
@pytest.mark.parametrize("fp8", [False, True], ids=["fp16", "fp8"])
def test_block_partials_for_the_merge_kernel(fp8, lens, ctas, group, hkv):
    """Rows over more than 8 blocks: the blocks merge their own part first."""
    if fp8:
        lens = [2 * n for n in lens]            # the tile is twice as long: the same units
    plan = _plan(fp8, lens, group, hkv, ctas)
    assert plan.merge_mode == 0
    _check(fp8, lens, group, hkv, plan.handle.value, 3, repeats=3)
