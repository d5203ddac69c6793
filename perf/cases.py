"""The decode path's work as its users call it: what is timed, on which inputs, and what the answer is.

Three kinds of case, told apart by `kind`:

  decode  one attention layer's decode step through `Decoder.run` over a paged cache, planned once
          beforehand (a serving step plans once and runs every layer with that plan)
  step    one step of a small serving loop through `PagedKVCache`: requests join a resident batch, their
          prompts are appended, the batch is planned and decoded, the joined requests leave again
  append  a prompt's tokens written (fp16 copy or E4M3 quantize) into scattered pages through
          `append_quantize`

Sequence lengths come from the case alone (`lens_of`), values from the seed.
"""

from __future__ import annotations

import math
import pathlib
import random
import sys

import torch

ROOT = pathlib.Path(__file__).resolve().parent.parent
if str(ROOT / "paged-attention_amd") not in sys.path:
    sys.path.insert(0, str(ROOT / "paged-attention_amd"))

import pa_amd  # noqa: E402

D = 128   # head_dim, the only one the path supports
DEV = "cuda"


def _decode(name, fp8, batch, lo, hi, hq, hkv, page):
    return {"name": name, "kind": "decode", "fp8": fp8, "batch": batch, "lo": lo, "hi": hi, "hq": hq, "hkv": hkv,
            "page": page, "len_seed": 4}


def listed():
    return [
        # The smallest step: one short chat turn. Launch and lookup latency only.
        _decode("decode 1x200 fp16", False, 1, 200, 200, 32, 8, 16),
        # A few short sequences: every sequence is cut over several blocks, latency-bound.
        _decode("decode 4x1024 fp16", False, 4, 1024, 1024, 32, 8, 16),
        # The ordinary batch of a busy server at moderate context, quantized cache.
        _decode("decode 32x1024 fp8", True, 32, 1024, 1024, 32, 8, 16),
        # The headline batch at long context, fp16 and FP8.
        _decode("decode 32x8192 fp16", False, 32, 8192, 8192, 32, 8, 16),
        _decode("decode 64x8192 fp8", True, 64, 8192, 8192, 32, 8, 16),
        # Continuous batching in earnest: every length different; the largest case.
        _decode("decode 128 ragged fp16", False, 128, 128, 16384, 32, 8, 16),
        # One long document, quantized: each sequence is cut over the whole chip.
        _decode("decode 1x131072 fp8", True, 1, 131072, 131072, 32, 8, 16),
        # One GPU's share of the headline batch under 8-way head sharding: one kv head.
        _decode("decode 32x8192 fp16 1 kv head", False, 32, 8192, 8192, 4, 1, 16),
        # Odd everything: ragged rows down to a single token, a page size that is no power of two,
        # a group of 8 query heads per kv head.
        _decode("decode 37 ragged fp8 page 24", True, 37, 1, 3001, 64, 8, 24),
        # A serving step: two requests with their prompts join 30 resident sequences.
        {"name": "step 30+2 fp16", "kind": "step", "fp8": False, "batch": 30, "lo": 100, "hi": 2000, "join": 2,
         "join_len": 333, "batched": True, "hq": 32, "hkv": 8, "page": 16, "len_seed": 5},
        # Prompts going into the cache: a long one quantized, a short one copied at an odd offset.
        {"name": "append 8192 fp8", "kind": "append", "fp8": True, "n": 8192, "start": 0, "hkv": 8, "page": 16},
        {"name": "append 500 fp16", "kind": "append", "fp8": False, "n": 500, "start": 37, "hkv": 8, "page": 16},
    ]


def _log_int(rng: random.Random, lo: int, hi: int) -> int:
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng: random.Random) -> dict:
    fp8 = rng.random() < 0.5
    kind = rng.choices(["decode", "step", "append"], [7, 2, 2])[0]
    page = rng.choice([1, 4, 8, 16, 16, 16, 16, 24, 32, 64, 128])
    if kind == "append":
        return {"kind": kind, "fp8": fp8, "n": _log_int(rng, 1, 16384), "start": rng.randrange(0, 200),
                "hkv": rng.choice([1, 2, 8]), "page": page}
    hq, hkv = rng.choice([(32, 8), (32, 8), (64, 8), (16, 8), (8, 8), (4, 1), (8, 1)])
    if kind == "step":
        hi = _log_int(rng, 16, 4000)
        return {"kind": kind, "fp8": fp8, "batch": _log_int(rng, 1, 64), "lo": max(1, hi // 8), "hi": hi,
                "join": rng.randrange(1, 5), "join_len": _log_int(rng, 1, 2000), "batched": rng.random() < 0.6,
                "hq": hq, "hkv": hkv, "page": page, "len_seed": rng.randrange(1000)}
    batch = _log_int(rng, 1, 128)
    # At most half of the largest listed case's tokens (some page sizes stream slower).
    most = min(131072, 500000 // batch)
    hi = _log_int(rng, 16, most)
    lo = hi if rng.random() < 0.4 else max(1, hi // rng.choice([2, 8, 1000]))
    return {"kind": kind, "fp8": fp8, "batch": batch, "lo": lo, "hi": hi, "hq": hq, "hkv": hkv, "page": page,
            "len_seed": rng.randrange(1000)}


def lens_of(case: dict) -> list[int]:
    r = random.Random(case["len_seed"])
    return [r.randint(case["lo"], case["hi"]) for _ in range(case["batch"])]


def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _normal(shape, g) -> torch.Tensor:
    return torch.empty(shape, dtype=torch.float16, device=DEV).normal_(generator=g)


def _fill(pool: torch.Tensor, g, scale: float) -> None:
    """N(0,1) values into a pool, as fp16 or as E4M3 of value / scale, a few pages at a time."""
    flat = pool.view(-1)
    chunk = 1 << 27
    for i in range(0, flat.numel(), chunk):
        part = flat[i:i + chunk]
        if pool.dtype == torch.float16:
            part.normal_(generator=g)
        else:
            x = _normal(part.shape, g).float().div_(scale).clamp_(-448.0, 448.0)
            part.copy_(x.to(torch.float8_e4m3fn).view(torch.uint8))


SCALE = 6.0 / 448.0   # about the largest of some 10^8 normal values / 448


def _decode_inputs(case: dict, seed: int) -> dict:
    lens, P = lens_of(case), case["page"]
    pages = [-(-n // P) for n in lens]
    g = _gen(seed)
    total = sum(pages) + 3
    k, v = pa_amd.alloc_kv_pools(total, case["hkv"], P, D, case["fp8"])
    scale = SCALE if case["fp8"] else 1.0
    _fill(k, g, scale)
    _fill(v, g, scale)
    perm = torch.randperm(total, device=DEV, generator=g).to(torch.int32)
    # Row b's pages are the next pages[b] of the permutation; short rows' spare columns stay 0.
    first = torch.tensor([0] + pages[:-1]).cumsum(0).to(DEV)
    count = torch.tensor(pages, device=DEV)
    col = torch.arange(max(pages), device=DEV)
    at = (first[:, None] + col[None, :]).clamp_(max=total - 1)
    table = torch.where(col[None, :] < count[:, None], perm[at], torch.zeros((), dtype=torch.int32, device=DEV))
    q = _normal((len(lens), case["hq"], D), g)
    return {"lens": lens, "k": k, "v": v, "table": table.contiguous(), "q": q, "scale": scale}


def _step_inputs(case: dict, seed: int) -> dict:
    g = _gen(seed)
    lens = lens_of(case)
    joined = [case["join_len"]] * case["join"]
    return {"lens": lens, "joined": joined, "resident": [_normal((2, n, case["hkv"], D), g) for n in lens],
            "k": _normal((sum(joined), case["hkv"], D), g), "v": _normal((sum(joined), case["hkv"], D), g),
            "q": _normal((len(lens) + len(joined), case["hq"], D), g)}


def _append_inputs(case: dict, seed: int) -> dict:
    g = _gen(seed)
    shape = (case["n"], case["hkv"], D)
    pages = -(-(case["start"] + case["n"]) // case["page"])
    return {"k": _normal(shape, g), "v": _normal(shape, g),
            "table": torch.randperm(pages, device=DEV, generator=g).to(torch.int32), "pages": pages}


def prepare(case: dict, seed: int) -> dict:
    hkv, P, fp8 = case["hkv"], case["page"], case["fp8"]
    if case["kind"] == "append":
        s = _append_inputs(case, seed)
        shape = (s["pages"], hkv, P, D)
        dt = torch.uint8 if fp8 else torch.float16
        s["kc"], s["vc"] = torch.zeros(shape, dtype=dt, device=DEV), torch.zeros(shape, dtype=dt, device=DEV)
    elif case["kind"] == "step":
        s = _step_inputs(case, seed)
        need = [-(-n // P) for n in s["lens"] + s["joined"]]
        cache = pa_amd.PagedKVCache(sum(need) + 3, P, hkv, D, len(need), max(need),
                                    pa_amd.FP8_E4M3 if fp8 else pa_amd.FP16, SCALE, SCALE)
        cache.shuffle_free_pages(seed & 0x7FFFFFFF)
        s["slots"] = [cache.admit() for _ in s["lens"]]
        for slot, kv in zip(s["slots"], s.pop("resident")):
            cache.append(slot, kv[0], kv[1], kv.shape[1])
        s["cache"], s["out"] = cache, torch.empty_like(s["q"])
    else:
        s = _decode_inputs(case, seed)
        lens = torch.tensor(s["lens"], dtype=torch.int32)
        s["dec"] = pa_amd.Decoder(case["hq"], hkv, D, P, fp8)
        s["dec"].plan(lens)
        s["lens_dev"] = lens.to(DEV)
    s["case"] = case
    return s


def run(s: dict):
    case = s["case"]
    if case["kind"] == "decode":
        return s["dec"].run(s["q"], s["k"], s["v"], s["table"], s["lens_dev"], s["scale"], s["scale"])
    if case["kind"] == "append":
        inv = 1.0 / SCALE
        pa_amd.append_quantize(pa_amd.FP8_E4M3 if case["fp8"] else pa_amd.FP16, s["k"], s["v"], s["kc"], s["vc"],
                               s["table"], case["start"], case["n"], case["hkv"], D, case["page"], inv, inv)
        return s["kc"], s["vc"]
    cache = s["cache"]
    new = [cache.admit() for _ in s["joined"]]
    if case["batched"]:
        cache.append_batch(new, s["joined"], s["k"], s["v"])
    else:
        at = 0
        for slot, n in zip(new, s["joined"]):
            cache.append(slot, s["k"][at:at + n], s["v"][at:at + n], n)
            at += n
    cache.plan(s["slots"] + new, case["hq"])
    cache.run(s["q"], s["out"])
    for slot in new:
        cache.release(slot)
    return s["out"]


def work(case: dict) -> dict:
    eb, hkv = (1 if case["fp8"] else 2), case["hkv"]
    if case["kind"] == "append":
        return {"bytes": 2 * case["n"] * hkv * D * (2 + eb) + 4 * -(-case["n"] // case["page"]), "flops": 0}
    joined = [case["join_len"]] * case["join"] if case["kind"] == "step" else []
    lens, new = lens_of(case) + joined, sum(joined)
    # K and V read once, q in and the result out, one table entry a page; a step's new tokens are read
    # in fp16 and written besides.
    kv = 2 * sum(lens) * hkv * D * eb + 4 * sum(-(-n // case["page"]) for n in lens)
    return {"bytes": kv + 4 * len(lens) * case["hq"] * D + 2 * new * hkv * D * (2 + eb),
            "flops": 4 * sum(lens) * case["hq"] * D}


def tolerance(case: dict):
    # Bytes and copies are exact. Decode outputs are rounded to fp16 (2^-12 of each value on average), and the
    # kernels weigh V with probabilities rounded to fp16; 2.4e-4 to 2.9e-4 measured against 64 bits.
    return "exact" if case["kind"] == "append" else {"rel": 1.2e-3, "max": 0.02}


def _attend(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor) -> torch.Tensor:
    """One row in 64 bits: q [Hq, D], k and v [L, Hkv, D] -> [Hq, D]."""
    hkv = k.shape[1]
    qg = q.double().view(hkv, -1, D)
    kt = k.double().permute(1, 2, 0).contiguous()
    vt = v.double().permute(1, 0, 2).contiguous()
    w = torch.softmax(torch.matmul(qg, kt) / math.sqrt(D), dim=-1)
    return torch.matmul(w, vt).reshape(-1, D)


def _value(x: torch.Tensor, scale: float) -> torch.Tensor:
    return x.double() if x.dtype == torch.float16 else x.view(torch.float8_e4m3fn).to(torch.float16).double() * scale


def exact(case: dict, seed: int):
    if case["kind"] == "append":
        return None   # bytes, compared as such
    P, hkv = case["page"], case["hkv"]
    if case["kind"] == "step":
        s = _step_inputs(case, seed)
        inv = torch.tensor(1.0 / SCALE, dtype=torch.float32, device=DEV)

        def kept(x):   # what the cache holds of x
            if not case["fp8"]:
                return x
            e = (x.float() * inv).clamp_(-448.0, 448.0).to(torch.float8_e4m3fn).view(torch.uint8)
            return _value(e, SCALE)
        at, rows = 0, [(kv[0], kv[1]) for kv in s["resident"]]
        for n in s["joined"]:
            rows.append((s["k"][at:at + n], s["v"][at:at + n]))
            at += n
        return torch.stack([_attend(s["q"][b], kept(k), kept(v)) for b, (k, v) in enumerate(rows)])
    s = _decode_inputs(case, seed)
    out = []
    for b, n in enumerate(s["lens"]):
        pages = s["table"][b, :-(-n // P)].long()
        k, v = (_value(x[pages].permute(0, 2, 1, 3).reshape(-1, hkv, D)[:n], s["scale"]) for x in (s["k"], s["v"]))
        out.append(_attend(s["q"][b], k, v))
    return torch.stack(out)
