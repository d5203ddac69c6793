// C-ABI host layer, part 1: the persistent planner, the device plan and the
// kernel entry points (decode, append, gather, stream reads) over the gfx950
// kernels in pa_decode.hip and pa_cache.hip. Every exported function catches
// exceptions and returns a pa_status (pa_decode.h maps them to the
// reference's errors).

#include "pa_host.hpp"

#include <algorithm>
#include <climits>
#include <string>
#include <vector>

namespace {

using namespace pa::host;

int group_of(int num_q_heads, int num_kv_heads) {
    if (num_kv_heads <= 0 || num_q_heads <= 0 || num_q_heads % num_kv_heads != 0)
        throw std::invalid_argument("num_q_heads must be a multiple of num_kv_heads");
    return num_q_heads / num_kv_heads;
}

void check_shape(int dtype, int head_dim, int group) {
    check_dtype(dtype);
    if (head_dim != pa::kHeadDim) throw std::invalid_argument("unsupported head_dim " + std::to_string(head_dim));
    if (group != 1 && group != 2 && group != 4 && group != 8)
        throw std::invalid_argument("unsupported GQA group size " + std::to_string(group));
}

int device_cus() {
    int dev = 0, cus = 0;
    pa::hip_check(hipGetDevice(&dev), "hipGetDevice");
    pa::hip_check(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev), "hipDeviceGetAttribute");
    return cus;
}

int wave_ctas_impl(int dtype, int head_dim, int group) {
    check_shape(dtype, head_dim, group);
    return device_cus() * pa::kernel_units_per_cu(dtype, group);
}

// Segments of one item whose partial rows the kernels address with 32-bit
// offsets (8 heads x 128 floats each).
constexpr int kMaxItemSegments = 1 << 19;

// The persistent cut (decode.cu:65-108): all (row, kv head) items are laid out
// in order as runs of `tile`-token tiles; the total is split into equal
// contiguous ranges of `per` tiles, one per work unit, and every maximal run of
// one item inside a range becomes a segment.
void cut(pa_plan& plan, int tile, const int32_t* lens, int batch, int hkv, int requested) {
    if (tile <= 0) throw std::invalid_argument("make_plan: tile must be positive");
    if (batch < 0 || hkv <= 0) throw std::invalid_argument("make_plan: bad batch or kv head count");
    if (batch > 0 && !lens) throw std::invalid_argument("make_plan: seq_lens is null");
    if (requested <= 0) throw std::invalid_argument("make_plan: num_ctas must be positive");
    // Emptied (its arrays' memory stays for the next cut), also when a length
    // is refused.
    plan.segments.clear();
    plan.cta_seg_begin.clear();
    plan.item_seg_begin.clear();
    plan.shape    = {};
    plan.num_ctas = 0;
    plan.tile     = tile;
    plan.items    = batch * hkv;
    plan.per      = 0;
    plan.own_grid = false;

    long total = 0;
    for (int b = 0; b < batch; ++b) {
        if (lens[b] <= 0) throw std::invalid_argument("make_plan: every sequence needs at least one token");
        total += (static_cast<long>(lens[b]) + tile - 1) / tile * hkv;
    }
    plan.item_seg_begin.assign(static_cast<size_t>(plan.items) + 1, 0);
    plan.cta_seg_begin.assign(1, 0);
    if (total == 0) return;
    const long per = (total + requested - 1) / requested;
    plan.per      = static_cast<int>(std::min<long>(per, INT_MAX));
    plan.num_ctas = static_cast<int>((total + per - 1) / per);
    plan.cta_seg_begin.resize(static_cast<size_t>(plan.num_ctas) + 1);
    // Every unit boundary adds at most one segment to the items' own.
    plan.segments.resize(4 * (static_cast<size_t>(plan.num_ctas) + static_cast<size_t>(plan.items)));
    pa_split_shape& sh = plan.shape;
    sh.item_unit.resize(static_cast<size_t>(plan.items));

    int32_t* seg  = plan.segments.data();
    int32_t  nseg = 0;
    int      item = 0, u = 0;   // u: the current unit
    long     left = per;        // tiles the current unit still takes
    for (int b = 0; b < batch; ++b) {
        const long tiles = (static_cast<long>(lens[b]) + tile - 1) / tile;
        for (int h = 0; h < hkv; ++h, ++item) {
            const int32_t first = nseg;
            plan.item_seg_begin[static_cast<size_t>(item)] = first;
            if (left == 0) {
                plan.cta_seg_begin[static_cast<size_t>(++u)] = nseg;
                left = per;
            }
            sh.item_unit[static_cast<size_t>(item)] = u;
            for (long done = 0; done < tiles;) {
                if (left == 0) {
                    plan.cta_seg_begin[static_cast<size_t>(++u)] = nseg;
                    left = per;
                }
                const long take = std::min(left, tiles - done);
                seg[0] = b;
                seg[1] = h;
                seg[2] = static_cast<int32_t>(done * tile);
                seg[3] = static_cast<int32_t>(std::min((done + take) * tile, static_cast<long>(lens[b])));
                seg += 4;
                ++nseg;
                done += take;
                left -= take;
            }
            // What split_shape would find: a unit takes one run of an item, and
            // an item's runs lie in consecutive units.
            const int n = nseg - first;
            sh.max_segments = std::max(sh.max_segments, n);
            if (n > 1) {
                const int nb = u / pa::kBlockUnits - sh.item_unit[static_cast<size_t>(item)] / pa::kBlockUnits + 1;
                sh.split      = true;
                sh.max_blocks = std::max(sh.max_blocks, nb);
                if (nb > 1) sh.in_block = false;
                if (n >= kMaxItemSegments) sh.consecutive = false;
            }
        }
    }
    plan.item_seg_begin[static_cast<size_t>(plan.items)] = nseg;
    plan.cta_seg_begin[static_cast<size_t>(plan.num_ctas)] = nseg;
    plan.segments.resize(4 * static_cast<size_t>(nseg));
}

}  // namespace

namespace pa::host {

thread_local std::string g_last_error;

void check_dtype(int dtype) {
    if (dtype != PA_KV_FP16 && dtype != PA_KV_FP8_E4M3)
        throw std::invalid_argument("unknown kv dtype " + std::to_string(dtype));
}
// The shape of any plan, from its arrays (make_plan's cut fills its own).
pa_split_shape split_shape(const pa_plan& plan) {
    pa_split_shape sh;
    const size_t nseg = plan.segments.size() / 4;
    sh.split = nseg > static_cast<size_t>(plan.items);
    std::vector<int32_t> unit_of(nseg, 0);
    for (int u = 0; u < plan.num_ctas; ++u)
        for (int sg = plan.cta_seg_begin[u]; sg < plan.cta_seg_begin[u + 1]; ++sg)
            unit_of[static_cast<size_t>(sg)] = u;
    sh.item_unit.resize(static_cast<size_t>(plan.items));
    for (int i = 0; i < plan.items; ++i) {
        const int a = plan.item_seg_begin[i], z = plan.item_seg_begin[i + 1];
        const int u0 = unit_of[static_cast<size_t>(a)];
        sh.item_unit[static_cast<size_t>(i)] = u0;
        sh.max_segments = std::max(sh.max_segments, z - a);
        if (z - a <= 1) continue;
        const int nb = unit_of[static_cast<size_t>(z - 1)] / pa::kBlockUnits - u0 / pa::kBlockUnits + 1;
        sh.max_blocks = std::max(sh.max_blocks, nb);
        if (nb > 1) sh.in_block = false;
        if (z - a >= kMaxItemSegments) sh.consecutive = false;
        for (int sg = a; sg < z; ++sg) {
            const int u = unit_of[static_cast<size_t>(sg)];
            if (sg != plan.cta_seg_begin[u] && sg != plan.cta_seg_begin[u + 1] - 1) sh.slots = false;
            if (u != u0 + (sg - a)) sh.consecutive = false;
        }
    }
    return sh;
}
// Tiles per unit of a plan that cuts its items, whole and in order, into equal
// ranges of tiles (the last unit may hold fewer), as make_plan does; 0 for others.
int equal_cut(const pa_plan& plan) {
    auto tiles = [&](int sg) {
        const int32_t* s = &plan.segments[4 * static_cast<size_t>(sg)];
        return (s[3] - s[2] + plan.tile - 1) / plan.tile;
    };
    long per = 0;
    for (int u = 0; u < plan.num_ctas; ++u) {
        long n = 0;
        for (int sg = plan.cta_seg_begin[u]; sg < plan.cta_seg_begin[u + 1]; ++sg) n += tiles(sg);
        if (u == 0) per = n;
        if (n <= 0 || n > per || (n < per && u + 1 < plan.num_ctas)) return 0;
    }
    for (int i = 0; i < plan.items; ++i) {
        int at = 0;
        for (int sg = plan.item_seg_begin[i]; sg < plan.item_seg_begin[i + 1]; ++sg) {
            const int32_t* s = &plan.segments[4 * static_cast<size_t>(sg)];
            const bool last = sg + 1 == plan.item_seg_begin[i + 1];
            if (s[2] != at || (!last && s[3] % plan.tile != 0)) return 0;
            at = s[3];
        }
    }
    return static_cast<int>(std::min<long>(per, INT_MAX));
}
// The split kernel's combine of a spanning item runs on one CU and reads one
// partial per block. Up to 8 blocks per item that is as fast as a merge launch
// or faster; past 8 the split kernel leaves one partial per block and the merge
// kernel, which spreads every item over many CUs, combines those (one MI355X,
// us per step, combine in the split kernel against this: 16 blocks per item,
// 2 x 2048 fp16 9.9 / 8.7, 2 x 16384 FP8 16.9 / 16.2; 32 blocks, 1 x 131072 FP8
// 47.4 / 45.8, 1 x 16384 fp16 19.0 / 15.7).
constexpr int kChainMaxBlocks = 8;
// One query head per kv head leaves partials of 512 bytes per segment: merging
// them per block first costs what it saves (1 x 131072 FP8 44.6 without, 45.2
// with; 1 x 16384 fp16 14.7 / 15.1; 2 x 16384 FP8 level) until an item has
// hundreds of segments (one kv head, 1 x 131072 fp16, 256 blocks: 18.2 / 15.6).
constexpr int kOneHeadMinBlocks = 64;
int merge_mode_of(const pa_split_shape& sh, int max_blocks) {
    // The split kernel keeps a unit's split segments in two LDS slots: they
    // must be the unit's first and last segments (true of every make_plan cut).
    if (!sh.split || !sh.slots) return 0;
    if (sh.in_block) return 1;
    // Merged across blocks: a block finds an item's other blocks from the unit
    // of the item's first segment, which needs the item's k-th segment in unit
    // u0 + k.
#if PA_CHAIN_MERGE
    if (sh.consecutive && sh.max_blocks <= max_blocks) return 2;
#endif
    return 0;
}
int plan_merge_mode(const pa_plan& plan) { return merge_mode_of(plan.shape, kChainMaxBlocks); }
void make_plan_impl(pa_plan& plan, int dtype, const int32_t* lens, int batch, int hq, int hkv, int hd,
                    int num_ctas) {
    const int group = group_of(hq, hkv);
    check_shape(dtype, hd, group);
    const int tile = pa::kernel_tile_tokens(dtype, group);
    const bool own = num_ctas <= 0;
    if (own) num_ctas = wave_ctas_impl(dtype, hd, group);
    cut(plan, tile, lens, batch, hkv, num_ctas);
    plan.own_grid = own;
}

namespace {
// Time a block takes per tile (8 KiB of K and V) with `blocks` of them running,
// in us: one CU alone streams 67 GB/s, 256 together 27 GB/s each, and between
// the two the measured time is linear (rows of 500 tokens, fp16, one block per
// (row, kv head): 8 blocks 67 GB/s per CU, 32 52, 128 36).
double tile_us(double blocks) { return 0.122 + 0.00071 * blocks; }
// Tiles of one item joined in a segment at most (block_merge 4).
constexpr int kMaxJoined = 3;
// What merging across blocks adds after a block's last wave, in us: the partial
// row stored, the arrival, the combine (FP8's blocks hold more rows).
constexpr double kSpanUs16 = 1.2, kSpanUs32 = 2.0;   // fp16, FP8 (16- and 32-token tiles)

// make_plan's equal cut leaves most items across two or more blocks unless their
// tiles happen to be whole blocks. Where that costs more than uneven units do,
// its segments run on other units, so that no item spans blocks: whole items per
// block (one each where there are no more items than blocks), a unit's segments
// consecutive, at most `limit` tiles of them (the smallest that fits) and only the
// first and last of them split ones (the kernel's two LDS slots).
// A segment's probabilities are rounded to 16 bits against its own running
// maximum, so the segments stay the plan's own, in units of their own: longer
// ones would lose precision. Where the plan's are single tiles, a unit's tiles of
// one item are joined, and the kernel takes each against its own maximum
// (block_merge 4): the same probabilities, bit for bit. (Joined without that, one
// row of 200 lay 2.65e-4 from 64 bits instead of 2.46e-4.)
// The estimates of both: the plan's blocks are equal; uneven ones run together for
// the average block and the rest of the largest at less than half of them. Same
// box, us per decode, 50 in a graph, across blocks -> inside: joined tiles, fp16
// 1 x 33 6.0 -> 4.1, 1 x 200 6.4 -> 5.6, 16 x 200 7.6 -> 6.2, FP8 16 x 200 7.6 ->
// 5.9, 1 x 400 7.1 -> 6.7; the plan's segments, fp16 32 x 200 9.2 -> 6.6, 64 x 200
// 12.9 -> 10.1, FP8 120 rows of 95 to 161 10.1 -> 8.1, 32 x 1100 14.7 -> 14.5. Left
// across blocks by the estimate, for longer segments inside would cost precision
// and uneven units time: fp16 32 x 1000, 32 x 5000, 128 rows of 100 to 200, FP8 32 x
// 2000 (22.3, 97, 16.4 and 23.0 when segments were cut anew; 24.7, 102, 17.9, 25.5).
// Only for a plan whose grid make_plan chose (`units`; own_grid): another grid is the
// caller's, also where it has as many tiles per unit. The host plan stays as it is.
// False: not grouped, `out` holds nothing of use.
bool group_in_blocks(const pa_plan& plan, int units, pa_plan& out) {
    const int items = plan.items, max_blocks = units / pa::kBlockUnits;
    if (!plan.own_grid || items <= 0 || max_blocks <= 0 || plan.per <= 0) return false;
    const int shift = __builtin_ctz(static_cast<unsigned>(plan.tile));   // the kernels' tiles are powers of two
    auto tiles = [&](int sg) {
        const int32_t* s = &plan.segments[4 * static_cast<size_t>(sg)];
        return (s[3] - s[2] + plan.tile - 1) >> shift;
    };
    std::vector<int32_t> item_tiles(static_cast<size_t>(items));
    long longest = 0, total = 0;
    for (int i = 0; i < items; ++i) {
        const int     len = plan.segments[4 * static_cast<size_t>(plan.item_seg_begin[i + 1]) - 1];
        const int32_t t   = (len + plan.tile - 1) >> shift;
        item_tiles[static_cast<size_t>(i)] = t;
        longest = std::max<long>(longest, t);
        total += t;
    }
    if (plan.per != (total + units - 1) / units) return false;
    const double across = static_cast<double>(pa::kBlockUnits) * plan.per * tile_us(plan.num_ctas / 8.0) +
                          (plan.tile == 16 ? kSpanUs16 : kSpanUs32);
    auto inside = [&](int limit, int blocks) {
        const double mean    = static_cast<double>(total) / blocks;
        const double largest = static_cast<double>(std::max<long>(longest, static_cast<long>(pa::kBlockUnits) * limit));
        return mean * tile_us(blocks) + (largest - mean) * tile_us(0.4 * blocks);
    };
    const bool one_each = items <= max_blocks;
    const bool join     = plan.per == 1;
    // Units as prefixes of the plan's segments: the last entry is the open one,
    // with `load` tiles in `count` segments, the last of a split item or not.
    auto& cta = out.cta_seg_begin;
    int  limit = plan.per, load = 0, count = 0;
    bool last_split = false;
    auto block_begins = [&] { return count == 0 && (cta.size() - 1) % pa::kBlockUnits == 0; };
    auto close_block = [&](int sg) {
        do cta.push_back(sg);
        while ((cta.size() - 1) % pa::kBlockUnits != 0);
        load = count = 0;
    };
    auto place = [&](int i) {   // false: the block has no unit left for item i
        const int first = plan.item_seg_begin[i], end = plan.item_seg_begin[i + 1];
        for (int sg = first; sg < end; ++sg) {
            const int  t    = tiles(sg);
            const bool more = sg > first && count > 0;   // the unit's last segment is the item's too
            if (count > 0 && (load + t > limit || (more ? !join : count > 1 && last_split))) {
                if (cta.size() % pa::kBlockUnits == 0) return false;
                cta.push_back(sg);
                load = count = 0;
            } else if (more) {
                --count;   // joined
            }
            load += t;
            ++count;
            last_split = end - first > 1;
        }
        return true;
    };
    // Whole items per block up to `cap` tiles (at least one). False as soon as the
    // units left could not hold the tiles left.
    auto fill = [&](long cap) {
        cta.assign(1, 0);
        load = count = 0;
        long block = 0, left = total;
        for (int i = 0; i < items; ++i) {
            const size_t at = cta.size();
            const bool begins = block_begins();
            const int  t = item_tiles[static_cast<size_t>(i)];
            if (begins) block = 0;
            left -= t;
            if (!begins && block + t > cap) {
                close_block(plan.item_seg_begin[i]);
            } else if (place(i)) {
                block += t;
                continue;
            } else if (begins) {
                return false;
            } else {
                cta.resize(at);
                close_block(plan.item_seg_begin[i]);
            }
            if (static_cast<long>(cta.size()) - 1 + (left + t + limit - 1) / limit > units || !place(i)) return false;
            block = t;
        }
        return true;
    };
    // The smallest cap, to 1/32, under which runs of items need no more blocks than
    // there are: full blocks beside idle CUs are slower (432 items of 1 to 3 tiles
    // 5.1 us, spread 4.4).
    auto spread = [&] {
        if (one_each) return 1l;
        for (long cap = std::max(longest, (total + max_blocks - 1) / max_blocks);; cap += cap / 32 + 1) {
            int  blocks = 0;
            long left   = 0;
            for (const int32_t t : item_tiles) {
                if (t > left) ++blocks, left = cap;
                left -= t;
            }
            if (blocks <= max_blocks) return cap;
        }
    };
    long cap = 0;
    for (;; limit += limit / 8 + 1) {
        if ((join && limit > kMaxJoined) || inside(limit, one_each ? items : max_blocks) >= across) return false;
        if (cap == 0) cap = spread();
        if (fill(cap)) break;
    }
    close_block(plan.item_seg_begin[items]);   // its last entry ends the last unit
    out.num_ctas = static_cast<int>(cta.size()) - 1;
    if (inside(limit, out.num_ctas / pa::kBlockUnits) >= across) return false;
    out.shape = {};
    out.segments.clear();
    out.segments.reserve(plan.segments.size());
    out.item_seg_begin.assign(static_cast<size_t>(items) + 1, 0);
    for (int u = 0, item = 0, sg = 0, begin = 0; u < out.num_ctas; ++u) {
        const int end = cta[static_cast<size_t>(u) + 1];
        for (cta[static_cast<size_t>(u)] = begin; sg < end; ++sg) {
            const bool first = sg == plan.item_seg_begin[item + 1];
            if (first) out.item_seg_begin[static_cast<size_t>(++item)] = begin;
            const int32_t* s = &plan.segments[4 * static_cast<size_t>(sg)];
            if (!first && join && begin > cta[static_cast<size_t>(u)]) {
                out.segments.back() = s[3];
            } else {
                out.segments.insert(out.segments.end(), s, s + 4);
                ++begin;
            }
            const int n = begin - out.item_seg_begin[static_cast<size_t>(item)];
            out.shape.max_segments = std::max(out.shape.max_segments, n);
        }
    }
    cta.back() = out.item_seg_begin.back() = static_cast<int32_t>(out.segments.size() / 4);
    return true;
}
}  // namespace
namespace {
// Whether the copy kernel of the buffer's last use has read it.
bool stage_read(const pa_stage& st) {
    for (size_t i = 0; i < st.marks; ++i)
        if (__atomic_load_n(st.host + st.cap + i, __ATOMIC_ACQUIRE) != st.mark) return false;
    return true;
}
// What the queue of that copy is at (pa::host::wait_read's status).
hipError_t queue_status(hipStream_t s) {
    // A query ends the capture of a stream that is being captured.
    hipStreamCaptureMode   mode = hipStreamCaptureModeRelaxed;
    hipStreamCaptureStatus cs   = hipStreamCaptureStatusNone;
    hipError_t e = hipThreadExchangeStreamCaptureMode(&mode);
    if (e != hipSuccess) return e;
    e = hipStreamIsCapturing(s, &cs);
    if (e == hipSuccess) e = cs == hipStreamCaptureStatusNone ? hipStreamQuery(s) : hipErrorNotReady;
    // The caller's stream may be gone; its work is not.
    if (e == hipErrorContextIsDestroyed || e == hipErrorInvalidHandle) e = hipDeviceSynchronize();
    if (e == hipErrorStreamCaptureImplicit || e == hipErrorStreamCaptureUnsupported) e = hipErrorNotReady;
    if (e == hipErrorNotReady) (void)hipGetLastError();   // an answer, not an error of the next launch
    const hipError_t back = hipThreadExchangeStreamCaptureMode(&mode);
    return back == hipSuccess ? e : back;
}
hipError_t wait_stage(const pa_stage& st) {
    return wait_read([&] { return stage_read(st); }, [&] { return queue_status(st.queue); });
}
bool stage_idle(const pa_stage& st) {
    if (!stage_read(st)) return false;
    if (!st.done) return true;
    const hipError_t q = hipEventQuery(st.done);
    if (q != hipErrorNotReady) pa::hip_check(q, "hipEventQuery staging");
    return q == hipSuccess;
}
}  // namespace
pa_stage& take_stage(pa_stage_pool& sp, size_t need, bool with_device) {
    const size_t n = sp.bufs.size();
    size_t pick = n, used = 0, oldest = n;
    for (size_t k = 0; k < n && pick == n; ++k) {
        const size_t i = (sp.next + k) % n;
        if (sp.bufs[i].captured) continue;
        ++used;
        if (oldest == n) oldest = i;
        if (stage_idle(sp.bufs[i])) pick = i;
    }
    if (pick == n) {
        if (used < pa_stage_pool::kMaxStages) {
            sp.bufs.emplace_back();
        } else {
            pick = oldest;   // every buffer in flight
            pa::hip_check(wait_stage(sp.bufs[pick]), "staging copy");
            if (sp.bufs[pick].done)
                pa::hip_check(hipEventSynchronize(sp.bufs[pick].done), "hipEventSynchronize staging");
        }
    }
    sp.next = (pick + 1) % sp.bufs.size();
    pa_stage& st = sp.bufs[pick];
    if (st.cap < need || (with_device && !st.dev)) {
        const size_t cap = (std::max<size_t>(need + need / 2, 4096) + 3) & ~size_t{3};   // whole 16 bytes
        const size_t all = cap + pa::stage_copy_blocks(cap);
        (void)hipHostFree(st.host);
        (void)hipFree(st.dev);
        st.host  = nullptr;
        st.dev   = nullptr;
        st.cap   = 0;
        st.marks = 0;
        pa::hip_check(hipHostMalloc(reinterpret_cast<void**>(&st.host), all * sizeof(int32_t),
                                    hipHostMallocMapped | hipHostMallocCoherent),
                      "hipHostMalloc staging");
        pa::hip_check(hipHostGetDevicePointer(reinterpret_cast<void**>(&st.host_dev), st.host, 0),
                      "hipHostGetDevicePointer staging");
        std::fill(st.host + cap, st.host + all, 0);
        st.mark = 0;
        if (with_device)
            pa::hip_check(hipMalloc(reinterpret_cast<void**>(&st.dev), cap * sizeof(int32_t)), "hipMalloc staging");
        st.cap = cap;
    }
    return st;
}
bool capturing(hipStream_t s) {
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    if (s) pa::hip_check(hipStreamIsCapturing(s, &cs), "hipStreamIsCapturing");
    return cs != hipStreamCaptureStatusNone;
}
void release_stage(pa_stage& st, hipStream_t s) {
    if (capturing(s)) {
        st.captured = true;
        return;
    }
    if (!st.done) pa::hip_check(hipEventCreateWithFlags(&st.done, hipEventDisableTiming), "hipEventCreate");
    pa::hip_check(hipEventRecord(st.done, s), "hipEventRecord staging");
}
void copy_stage(pa_stage& st, int32_t* dev, size_t n, hipStream_t s) {
    if (capturing(s)) {   // the graph's replays read it
        pa::hip_check(pa::launch_stage_copy(st.host_dev, dev, n, nullptr, 0, s), "staging copy kernel launch");
        st.captured = true;
        return;
    }
    st.mark  = st.mark == INT32_MAX ? 1 : st.mark + 1;
    st.marks = pa::stage_copy_blocks(n);
    st.queue = s;
    const hipError_t e = pa::launch_stage_copy(st.host_dev, dev, n, st.host_dev + st.cap, st.mark, s);
    if (e != hipSuccess) st.marks = 0;   // nothing was queued
    pa::hip_check(e, "staging copy kernel launch");
}
void free_stages(pa_stage_pool& sp) {
    for (pa_stage& st : sp.bufs) {
        (void)wait_stage(st);
        if (st.done) (void)hipEventSynchronize(st.done);
        (void)hipHostFree(st.host);
        (void)hipFree(st.dev);
        if (st.done) (void)hipEventDestroy(st.done);
    }
    sp = pa_stage_pool{};
}
void device_plan_upload(pa_device_plan& dp, const pa_plan& plan, int group, int head_dim, hipStream_t s,
                        const int32_t* extra, size_t n_extra) {
    if (group <= 0 || head_dim <= 0) throw std::invalid_argument("upload: bad group or head_dim");
    if (n_extra && !extra) throw std::invalid_argument("upload: extra ints are null");
    scratch_prepare();
    const size_t nseg = plan.segments.size() / 4;
    // The kernels read a 16-token group from one page run (page sizes >= 16) or
    // one 1 KiB part from one page: a segment may only start on a group boundary.
    for (size_t i = 0; i < nseg; ++i)
        if (plan.segments[4 * i + 2] % pa::kGroupTokens != 0)
            throw std::invalid_argument("upload: segment starts must be multiples of 16 tokens");
    const bool kernel_tile = plan.tile == pa::kernel_tile_tokens(PA_KV_FP16, group) ||
                             plan.tile == pa::kernel_tile_tokens(PA_KV_FP8_E4M3, group);
    // Grouped only where pa_decode_static's array holds the plan's partials: a
    // plan merged in LDS needs none of it, and what that call refuses does not
    // depend on the grouping.
    const size_t rows  = nseg * static_cast<size_t>(group);
    const size_t need  = rows * (static_cast<size_t>(head_dim) + 1);
    const bool   fits  = need * sizeof(float) <= scratch_bytes();
    const bool   inside = fits && kernel_tile && plan.per > 0 && plan_merge_mode(plan) == 2 &&
                        group_in_blocks(plan, device_cus() * pa::kernel_units_per_cu(PA_KV_FP16, group), dp.blocks);
    const pa_plan& run = inside ? dp.blocks : plan;   // what the device gets
    // One block: segments | cta_seg_begin | item_seg_begin | extra | merge
    // counters, each part starting on a 16-byte boundary (the kernels read
    // segments as int4).
    auto round4 = [](size_t n) { return (n + 3) & ~size_t{3}; };
    const size_t o_cta   = round4(run.segments.size());
    const size_t o_item  = o_cta + round4(run.cta_seg_begin.size());
    const size_t o_extra = o_item + round4(run.item_seg_begin.size());
    const size_t o_ctr   = o_extra + round4(n_extra);   // merge counters, uploaded as zeros
    const pa_split_shape& shape = run.shape;
    const int  in_kernel = !inside ? merge_mode_of(shape, kChainMaxBlocks) : plan.per == 1 ? 4 : 1;
    // Past kChainMaxBlocks: block partials for the merge kernel (block_merge 3),
    // where the split kernel can find an item's part of a block. Same box, us per
    // step, every segment's partial / block partials: one row of 131072, one kv
    // head 20.8 / 16.1; 1 x 4096 fp16 10.0 / 8.9; 2 x 2048, 64 query heads 12.0 /
    // 9.4; 3 ragged rows to 30000 21.9 / 20.5; 1 x 131072 FP8 46.4 / 45.9.
    const bool blocks    = in_kernel == 0 && merge_mode_of(shape, INT_MAX) == 2 &&
                        (group > 1 || shape.max_blocks >= kOneHeadMinBlocks);
    const size_t o_unit  = o_ctr + pa::plan_item_units(plan.items, group);
    const size_t total   = blocks ? o_unit + round4(shape.item_unit.size()) : o_unit;
    if (total > dp.ints_cap) {
        // Growing frees the old block, which decodes queued before may still
        // read: wait for them first (growth only happens for a plan larger
        // than every earlier one).
        pa::hip_check(hipStreamSynchronize(s), "hipStreamSynchronize");
        pa::hip_check(hipFree(dp.ints), "hipFree");
        dp.ints = nullptr;
        dp.ints_cap = 0;
        const size_t cap = std::max<size_t>(total + total / 4, 1024);
        pa::hip_check(hipMalloc(reinterpret_cast<void**>(&dp.ints), cap * sizeof(int32_t)), "hipMalloc plan");
        dp.ints_cap = cap;
    }
    pa_stage& st = take_stage(dp.staging, total, false);
    std::copy(run.segments.begin(), run.segments.end(), st.host);
    std::copy(run.cta_seg_begin.begin(), run.cta_seg_begin.end(), st.host + o_cta);
    std::copy(run.item_seg_begin.begin(), run.item_seg_begin.end(), st.host + o_item);
    if (n_extra) std::copy(extra, extra + n_extra, st.host + o_extra);
    std::fill(st.host + o_ctr, st.host + o_unit, 0);
    if (blocks) std::copy(shape.item_unit.begin(), shape.item_unit.end(), st.host + o_unit);
    copy_stage(st, dp.ints, total, s);
    dp.segments       = dp.ints;
    dp.cta_seg_begin  = dp.ints + o_cta;
    dp.item_seg_begin = dp.ints + o_item;
    dp.extra          = n_extra ? dp.ints + o_extra : nullptr;
    dp.merge_counters = dp.ints + o_ctr;
    if (need > dp.part_cap) {
        pa::hip_check(hipStreamSynchronize(s), "hipStreamSynchronize");   // queued decodes may still use it
        pa::hip_check(hipFree(dp.partial_out), "hipFree");
        dp.partial_out = nullptr;
        pa::hip_check(hipMalloc(reinterpret_cast<void**>(&dp.partial_out), sizeof(float) * need), "hipMalloc");
        dp.part_cap = need;
    }
    dp.partial_lse = dp.partial_out ? dp.partial_out + rows * head_dim : nullptr;
    dp.num_ctas = run.num_ctas;
    dp.num_segments = static_cast<int>(nseg);
    dp.block_merge = blocks ? 3 : in_kernel;
    dp.needs_merge = blocks || (in_kernel == 0 && shape.split) ? 1 : 0;
    dp.max_item_segments = shape.max_segments;
}
void device_plan_bind(const pa_device_plan& dp, pa_decode_params& p) {
    p.segments       = dp.segments;
    p.cta_seg_begin  = dp.cta_seg_begin;
    p.item_seg_begin = dp.item_seg_begin;
    p.num_ctas       = dp.num_ctas;
    p.needs_merge    = dp.needs_merge;
    p.partial_out    = dp.partial_out;
    p.partial_lse    = dp.partial_lse;
    p.max_item_segments = dp.max_item_segments;
    p.block_merge       = dp.block_merge;
    p.num_segments      = dp.num_segments;
    p.merge_counters    = dp.merge_counters;
}
void device_plan_free(pa_device_plan& dp) {
    free_stages(dp.staging);
    (void)hipFree(dp.ints);
    (void)hipFree(dp.partial_out);
    dp = pa_device_plan{};
}
void decode_impl(int dtype, const pa_decode_params& p, hipStream_t s, bool split, bool merge) {
    if (split) pa::hip_check(pa::launch_decode_split(dtype, p, s), "decode split kernel launch");
    if (merge) pa::hip_check(pa::launch_decode_merge(dtype, p, s), "decode merge kernel launch");
}

}  // namespace pa::host

using namespace pa::host;

extern "C" {

const char* pa_last_error(void) { return g_last_error.c_str(); }

int pa_kv_dtype_bytes(int dtype) { return dtype == PA_KV_FP16 ? 2 : 1; }
const char* pa_kv_dtype_name(int dtype) { return dtype == PA_KV_FP16 ? "fp16" : "fp8_e4m3"; }

pa_status pa_tile_tokens(int dtype, int head_dim, int group, int* out) {
    return guarded([&] {
        check_shape(dtype, head_dim, group);
        if (!out) throw std::invalid_argument("out is null");
        *out = pa::kernel_tile_tokens(dtype, group);
    });
}

pa_status pa_wave_ctas(int dtype, int head_dim, int group, int* out) {
    return guarded([&] {
        if (!out) throw std::invalid_argument("out is null");
        *out = wave_ctas_impl(dtype, head_dim, group);
    });
}

pa_status pa_default_ctas(int dtype, int head_dim, int group, int* out) {
    // One full wave: every resident work unit gets one equal range.
    return pa_wave_ctas(dtype, head_dim, group, out);
}

pa_status pa_plan_build(int dtype, const int32_t* seq_lens, int batch, int num_q_heads, int num_kv_heads,
                        int head_dim, int num_ctas, pa_plan** out) {
    return guarded([&] {
        if (!out) throw std::invalid_argument("out is null");
        auto* plan = new pa_plan;
        try {
            make_plan_impl(*plan, dtype, seq_lens, batch, num_q_heads, num_kv_heads, head_dim, num_ctas);
        } catch (...) {
            delete plan;
            throw;
        }
        *out = plan;
    });
}

pa_status pa_plan_build_tiled(int tile, const int32_t* seq_lens, int batch, int num_kv_heads, int num_ctas,
                              pa_plan** out) {
    return guarded([&] {
        if (!out) throw std::invalid_argument("out is null");
        auto* plan = new pa_plan;
        try {
            cut(*plan, tile, seq_lens, batch, num_kv_heads, num_ctas);
        } catch (...) {
            delete plan;
            throw;
        }
        *out = plan;
    });
}

pa_status pa_plan_create(int num_ctas, int tile, const int32_t* segments, int num_segments,
                         const int32_t* cta_seg_begin, const int32_t* item_seg_begin, int num_items,
                         int num_kv_heads, pa_plan** out) {
    return guarded([&] {
        if (!out) throw std::invalid_argument("out is null");
        if (num_ctas < 0 || num_segments < 0 || num_items < 0 || tile <= 0 || num_kv_heads < 0)
            throw std::invalid_argument("plan: negative sizes or non-positive tile");
        if ((num_segments && !segments) || !cta_seg_begin || !item_seg_begin)
            throw std::invalid_argument("plan: null array");
        if (num_kv_heads == 0) {   // every (row, kv head) has a segment, so the heads are 0 .. max
            for (int i = 0; i < num_segments; ++i) num_kv_heads = std::max(num_kv_heads, segments[4 * i + 1] + 1);
            num_kv_heads = std::max(num_kv_heads, 1);
        }
        if (num_items % num_kv_heads != 0) throw std::invalid_argument("plan: items must be batch * num_kv_heads");
        auto prefix_ok = [&](const int32_t* a, int n) {
            if (a[0] != 0 || a[n] != num_segments) return false;
            for (int i = 0; i < n; ++i)
                if (a[i + 1] < a[i]) return false;
            return true;
        };
        if (!prefix_ok(cta_seg_begin, num_ctas) || !prefix_ok(item_seg_begin, num_items))
            throw std::invalid_argument("plan: segment prefix arrays must rise from 0 to num_segments");
        for (int i = 0; i < num_items; ++i)
            if (item_seg_begin[i + 1] == item_seg_begin[i])
                throw std::invalid_argument("plan: every (row, kv head) needs a segment");
        for (int i = 0; i < num_segments; ++i) {
            const int32_t* sg = segments + 4 * static_cast<size_t>(i);
            const long item = static_cast<long>(sg[0]) * num_kv_heads + sg[1];
            if (sg[0] < 0 || sg[1] < 0 || sg[1] >= num_kv_heads || item >= num_items)
                throw std::invalid_argument("plan: segment row / kv head out of range");
            if (sg[2] < 0 || sg[3] <= sg[2]) throw std::invalid_argument("plan: empty or negative segment");
            if (sg[2] % pa::kGroupTokens != 0)
                throw std::invalid_argument("plan: segment starts must be multiples of 16 tokens");
            if (i < item_seg_begin[item] || i >= item_seg_begin[item + 1])
                throw std::invalid_argument("plan: segment is not listed under its (row, kv head)");
        }
        auto* plan = new pa_plan;
        plan->num_ctas = num_ctas;
        plan->tile     = tile;
        plan->items    = num_items;
        plan->segments.assign(segments, segments + 4 * static_cast<size_t>(num_segments));
        plan->cta_seg_begin.assign(cta_seg_begin, cta_seg_begin + num_ctas + 1);
        plan->item_seg_begin.assign(item_seg_begin, item_seg_begin + num_items + 1);
        plan->shape    = split_shape(*plan);
        plan->per      = equal_cut(*plan);
        *out = plan;
    });
}

void pa_plan_destroy(pa_plan* plan) { delete plan; }
int  pa_plan_num_ctas(const pa_plan* plan) { return plan ? plan->num_ctas : 0; }
int  pa_plan_tile(const pa_plan* plan) { return plan ? plan->tile : 0; }
int  pa_plan_num_segments(const pa_plan* plan) { return plan ? static_cast<int>(plan->segments.size() / 4) : 0; }
int  pa_plan_num_items(const pa_plan* plan) { return plan ? plan->items : 0; }
int pa_plan_own_grid(const pa_plan* plan) { return plan && plan->own_grid ? 1 : 0; }
pa_status pa_plan_set_own_grid(pa_plan* plan, int own) {
    return guarded([&] {
        if (!plan) throw std::invalid_argument("plan is null");
        plan->own_grid = own != 0;
    });
}
pa_status pa_plan_merge_mode(const pa_plan* plan, int* out) {
    return guarded([&] {
        if (!plan || !out) throw std::invalid_argument("plan or out is null");
        *out = plan_merge_mode(*plan);
    });
}

pa_status pa_plan_copy(const pa_plan* plan, int32_t* segments, int32_t* cta_seg_begin, int32_t* item_seg_begin) {
    return guarded([&] {
        if (!plan) throw std::invalid_argument("plan is null");
        if (segments) std::copy(plan->segments.begin(), plan->segments.end(), segments);
        if (cta_seg_begin) std::copy(plan->cta_seg_begin.begin(), plan->cta_seg_begin.end(), cta_seg_begin);
        if (item_seg_begin) std::copy(plan->item_seg_begin.begin(), plan->item_seg_begin.end(), item_seg_begin);
    });
}

pa_status pa_device_plan_create(pa_device_plan** out) {
    return guarded([&] {
        if (!out) throw std::invalid_argument("out is null");
        *out = new pa_device_plan;
    });
}

void pa_device_plan_destroy(pa_device_plan* dp) {
    if (!dp) return;
    device_plan_free(*dp);
    delete dp;
}

pa_status pa_device_plan_upload(pa_device_plan* dp, const pa_plan* plan, int group, int head_dim, void* stream) {
    return guarded([&] {
        if (!dp || !plan) throw std::invalid_argument("device plan or plan is null");
        device_plan_upload(*dp, *plan, group, head_dim, as_stream(stream));
    });
}

pa_status pa_device_plan_bind(const pa_device_plan* dp, pa_decode_params* p) {
    return guarded([&] {
        if (!dp || !p) throw std::invalid_argument("device plan or params is null");
        device_plan_bind(*dp, *p);
    });
}

pa_status pa_decode(int dtype, const pa_decode_params* p, void* stream) {
    return guarded([&] {
        if (!p) throw std::invalid_argument("params is null");
        decode_impl(dtype, *p, as_stream(stream), true, true);
    });
}

pa_status pa_decode_split(int dtype, const pa_decode_params* p, void* stream) {
    return guarded([&] {
        if (!p) throw std::invalid_argument("params is null");
        decode_impl(dtype, *p, as_stream(stream), true, false);
    });
}

pa_status pa_decode_merge(int dtype, const pa_decode_params* p, void* stream) {
    return guarded([&] {
        if (!p) throw std::invalid_argument("params is null");
        decode_impl(dtype, *p, as_stream(stream), false, true);
    });
}

pa_status pa_append_quantize(int dtype, const uint16_t* k, const uint16_t* v, void* k_cache, void* v_cache,
                             const int32_t* block_table_row, int start_pos, int n, int num_kv_heads, int head_dim,
                             int page_size, float inv_k_scale, float inv_v_scale, void* stream) {
    return guarded([&] {
        check_dtype(dtype);
        if (head_dim != pa::kHeadDim) throw std::invalid_argument("unsupported head_dim " + std::to_string(head_dim));
        if (num_kv_heads <= 0 || page_size <= 0 || start_pos < 0 || n < 0)
            throw std::invalid_argument("append: bad sizes");
        // One thread per (token, kv head, 8-dim chunk), indexed in 32 bits.
        if (static_cast<long long>(n) * num_kv_heads * (pa::kHeadDim / 8) > INT_MAX)
            throw std::length_error("append: n * num_kv_heads * 16 exceeds INT_MAX");
        if (n > 0 && (!k || !v || !k_cache || !v_cache || !block_table_row))
            throw std::invalid_argument("append: null pointer");
        pa::hip_check(pa::launch_append(dtype, k, v, k_cache, v_cache, block_table_row, start_pos, n, num_kv_heads,
                                        page_size, inv_k_scale, inv_v_scale, as_stream(stream)),
                      "append kernel launch");
    });
}

pa_status pa_gather_kv(int dtype, const void* cache, const int32_t* block_table_row, int num_kv_heads, int head_dim,
                       int page_size, int kv_head, int len, void* out, void* stream) {
    return guarded([&] {
        check_dtype(dtype);
        if (head_dim != pa::kHeadDim) throw std::invalid_argument("unsupported head_dim " + std::to_string(head_dim));
        if (num_kv_heads <= 0 || page_size <= 0 || kv_head < 0 || kv_head >= num_kv_heads || len < 0)
            throw std::invalid_argument("gather: bad sizes");
        pa::hip_check(pa::launch_gather(dtype, cache, block_table_row, num_kv_heads, page_size, kv_head, len, out,
                                        as_stream(stream)),
                      "gather kernel launch");
    });
}

pa_status pa_stream_read(const void* buf, size_t bytes, int blocks, uint32_t* sink, void* stream) {
    return pa_stream_read_ex(buf, bytes, blocks, 256, 1, 0, sink, stream);
}

pa_status pa_stream_read_chunked(const void* buf, size_t bytes, int blocks, int threads, int unroll, uint32_t* sink,
                                 void* stream) {
    return guarded([&] {
        if (!buf || !sink) throw std::invalid_argument("stream_read_chunked: null pointer");
        pa::hip_check(pa::launch_stream_read_chunked(buf, bytes, blocks, threads, unroll, sink, as_stream(stream)),
                      "stream_read_chunked launch");
    });
}

pa_status pa_stream_read_ex(const void* buf, size_t bytes, int blocks, int threads, int unroll, int nontemporal,
                            uint32_t* sink, void* stream) {
    return guarded([&] {
        if (bytes % 16 != 0 || blocks <= 0 || !buf || !sink) throw std::invalid_argument("stream_read: bad arguments");
        pa::hip_check(pa::launch_stream_read(buf, bytes, blocks, threads, unroll, nontemporal != 0, sink,
                                             as_stream(stream)),
                      "read kernel launch");
    });
}

pa_status pa_f32_to_f16(const float* in, uint16_t* out, size_t n, void* stream) {
    return guarded([&] {
        if (n && (!in || !out)) throw std::invalid_argument("f32_to_f16: null pointer");
        pa::hip_check(pa::launch_convert(in, out, n, true, as_stream(stream)), "convert kernel launch");
    });
}

pa_status pa_f16_to_f32(const uint16_t* in, float* out, size_t n, void* stream) {
    return guarded([&] {
        if (n && (!in || !out)) throw std::invalid_argument("f16_to_f32: null pointer");
        pa::hip_check(pa::launch_convert(in, out, n, false, as_stream(stream)), "convert kernel launch");
    });
}

pa_status pa_fill_bytes(void* buf, size_t bytes, int value, void* stream) {
    return guarded([&] {
        if (bytes % 16 != 0 || (bytes && !buf)) throw std::invalid_argument("fill_bytes: bad arguments");
        pa::hip_check(pa::launch_fill_bytes(buf, bytes, value, as_stream(stream)), "fill kernel launch");
    });
}

}  // extern "C"
