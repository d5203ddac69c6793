"""Appends whose page lists sit at the edges of what travels in a kernel's arguments (256 and 896 ints; past
that through a staging buffer), one call per sequence and batched, and on more streams than are tracked:
stored bytes bit-exact, decode within tolerance, device table and lengths as the host's.
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
