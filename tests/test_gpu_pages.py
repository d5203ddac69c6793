"""Page sizes that are no powers of two: the same tokens in pages of P decode bitwise the same as in pages
of 16, on the path that looks a page up once per 1 KiB part (multiples of 8, and of 4 for fp16) and on the
per-lane path (every other size), at lengths around the edges of pages, parts and steps.
"""

from __future__ import annotations

import pytest

import pa_amd
from helpers import D

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("gpu_device")]


def _paged(x, P, perm):
    """[B][L][Hkv][D] -> pool [pages][Hkv][P][D], row b's page i at perm[b * per_row + i]."""
    import torch
    B, L, H, _ = x.shape
    per = -(-L // P)
    pad = torch.zeros((B, per * P, H, D), dtype=x.dtype, device=x.device)
    pad[:, :L] = x
    pages = pad.view(B, per, P, H, D).permute(0, 1, 3, 2, 4).reshape(B * per, H, P, D)
    pool = torch.empty_like(pages)
    pool[perm.long()] = pages
    return pool.contiguous()


@pytest.mark.parametrize("fp8", [False, True], ids=["fp16", "fp8"])
@pytest.mark.parametrize("P", [3, 5, 12, 20, 24, 40, 56, 100, 1000, 2112])
def test_odd_page_sizes_match_pages_of_16(fp8, P):
    import torch
    B, L, hkv, hq = 7, 2400, 2, 8
    lens = [1, P - 1, P, P + 1, 2399, 33, 17 * P + 9]
    lens = [min(max(n, 1), L) for n in lens]
    g = torch.Generator(device="cuda").manual_seed(P)
    x = [torch.randn((B, L, hkv, D), dtype=torch.float16, device="cuda", generator=g) for _ in range(2)]
    if fp8:
        x = [(t.float() * 80).to(torch.float8_e4m3fn).view(torch.uint8) for t in x]
    q = torch.randn((B, hq, D), dtype=torch.float16, device="cuda", generator=g)
    lt = torch.tensor(lens, dtype=torch.int32)
    outs = []
    for page in (16, P):
        per = -(-L // page)
        perm = torch.randperm(B * per, device="cuda", generator=g).to(torch.int32)
        k, v = (_paged(t, page, perm) for t in x)
        dec = pa_amd.Decoder(hq, hkv, D, page, fp8)
        dec.plan(lt)
        outs.append(dec.run(q, k, v, perm.view(B, per).contiguous(), lt.cuda(), 1 / 80, 1 / 80))
    torch.cuda.synchronize()
    assert torch.isfinite(outs[0]).all()
    assert torch.equal(outs[0].view(torch.int16), outs[1].view(torch.int16))
