// Host-only logic of the Q4_RDNA runtime (see q4rdna_host.h): nothing here
// calls the HIP runtime.
#include "q4rdna_host.h"

#include <algorithm>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <functional>
#include <map>
#include <queue>
#include <utility>

namespace q4rdna {
namespace host {
namespace {

int fail(std::string *error, int code, const char *fmt, ...) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    std::vsnprintf(buf, sizeof(buf), fmt, ap);
    va_end(ap);
    if (error) *error = buf;
    return code;
}

bool aligned(const void *p, uintptr_t a) { return (reinterpret_cast<uintptr_t>(p) & (a - 1)) == 0; }

uint64_t align256(uint64_t v) { return (v + 255) & ~uint64_t(255); }

}  // namespace

int parse_index(const uint8_t *image, uint64_t image_size, uint64_t file_size, FileHeader *header,
                std::vector<Entry> *entries, std::string *error) {
    if (image == nullptr) return fail(error, Q4RDNA_ERR_ARGUMENT, "sidecar image is NULL");
    if (image_size < sizeof(FileHeader) || file_size < sizeof(FileHeader))
        return fail(error, Q4RDNA_ERR_FORMAT, "invalid sidecar header: truncated");
    FileHeader h;
    std::memcpy(&h, image, sizeof(h));
    if (std::memcmp(h.magic, "Q4RDNA1", 8) != 0 || h.version != 1 || h.group != kGroup ||
        h.tile_rows != kTileRows || h.tile_bytes != kTileBytes)
        return fail(error, Q4RDNA_ERR_FORMAT, "invalid sidecar header");
    const uint64_t index_end = sizeof(FileHeader) + static_cast<uint64_t>(h.count) * sizeof(FileEntry);
    if (file_size < index_end) return fail(error, Q4RDNA_ERR_FORMAT, "truncated sidecar index");
    if (image_size < index_end)
        return fail(error, Q4RDNA_ERR_ARGUMENT, "image holds %llu bytes, the index ends at %llu",
                    static_cast<unsigned long long>(image_size), static_cast<unsigned long long>(index_end));
    std::vector<Entry> out;
    out.reserve(h.count);
    for (uint32_t i = 0; i < h.count; ++i) {
        FileEntry e;
        std::memcpy(&e, image + sizeof(FileHeader) + static_cast<uint64_t>(i) * sizeof(FileEntry), sizeof(e));
        // The data region's end, computed without wrapping: an entry must lie
        // inside [data_offset, data_offset + data_bytes).
        const bool inside = e.offset >= h.data_offset && e.offset - h.data_offset <= h.data_bytes &&
                            e.size <= h.data_bytes - (e.offset - h.data_offset);
        if (std::memchr(e.name, '\0', sizeof(e.name)) == nullptr || !inside || e.rows % kTileRows != 0 ||
            e.columns % kGroup != 0 || e.size != static_cast<uint64_t>(e.rows) * e.columns * 34 / kGroup)
            return fail(error, Q4RDNA_ERR_FORMAT, "invalid sidecar entry %u", i);
        out.push_back(Entry{std::string(e.name), e.rows, e.columns, e.offset, e.size});
    }
    if (h.data_offset > file_size || h.data_bytes > file_size - h.data_offset)
        return fail(error, Q4RDNA_ERR_FORMAT, "truncated sidecar data");
    if (header) *header = h;
    if (entries) *entries = std::move(out);
    return Q4RDNA_OK;
}

bool valid_shape(uint32_t rows, uint32_t cols) {
    return rows > 0 && cols > 0 && rows % kTileRows == 0 && cols % kGroup == 0;
}

// About 32 groups per workgroup (eight waves of four tiles, all in flight at
// once) and at most 8 chunks; more chunks only when the row tiles are so few
// that under a quarter of the CUs would get a workgroup, fewer when there would
// be more than six workgroups per CU.  Measured on MI355X (split sweep, with
// and without a SwiGLU gate): 4096x4096 best at 2, 1024x4096 at 2-4, 12288x4096
// at 2, 4096x12288 at 6, 2048x28672 at 7-8, 151936x4096 at 1-2.
static uint32_t coarse_split(uint32_t tiles, uint32_t groups, uint32_t cus) {
    uint32_t split = std::min<uint32_t>((groups + 31) / 32, 8);
    if (static_cast<uint64_t>(tiles) * split * 4 < cus)
        split = std::min((cus / 4 + tiles - 1) / tiles, std::max<uint32_t>(1, groups / 16));
    if (static_cast<uint64_t>(tiles) * split > 6ull * cus) split = 6 * cus / tiles;
    return std::max<uint32_t>(1, std::min(split, std::min(groups, kMaxSplit)));
}

// The finer of two splits where it is the faster one, of about 900 timings of
// both (8 to 3072 row tiles, 33 to 256 groups, with and without a gate, single
// launches and groups; us in the lines below are single launches, coarse /
// fine).
uint32_t policy_split(uint32_t rows, uint32_t cols, uint32_t cus, bool gate, LaunchKind kind) {
    const uint32_t tiles = rows / kTileRows, groups = cols / kGroup;
    const uint32_t coarse = coarse_split(tiles, groups, cus);
    // Several vectors: each chunk costs a meeting per vector (5120x5120, four
    // vectors: 9.9 us in three chunks, 11.1 in five; 28672x8192 47.6, 50.5).
    if (kind == LaunchKind::kVectors) return coarse;
    auto wgs = [&](uint32_t split) { return static_cast<uint64_t>(tiles) * split; };

    // Chunks of about 16 groups where they fill the waves, which hold 1, 2, 4
    // or 8 tiles, better than 32 (41 groups: three chunks of 14 instead of two
    // of 21), and in single launches with a gate, whose chunks are twice the
    // bytes, once that makes more than six workgroups per CU (12288x4096 with
    // a gate, six, measures 12.5 either way; 16384x4096 15.4 / 15.2, 22400x4096
    // 22.5 / 19.6).
    const uint32_t by32 = (groups + 31) / 32, by16 = (groups + 15) / 16;
    const bool finer = by16 <= 8 && (by16 < 2 * by32 || (gate && kind == LaunchKind::kSingle && wgs(by16) > 6ull * cus));
    const uint32_t fine = finer ? by16 : std::min<uint32_t>(by32, 8);
    // Long rows (chunks of more than 32 groups at eight chunks) stay at six
    // workgroups per CU.  So does what would pass 32 per CU: 65536x8192, 32 per
    // CU, 55.3 / 47.9, but nothing finer is tried beyond (65568x8192 in one
    // chunk 55.3, in two 50.3; 64000x5120 in one 36.8, in three 33.1).
    if (fine == coarse || groups > 32 * fine || wgs(fine) * 4 < cus || wgs(fine) > 32ull * cus) return coarse;

    // The groups of the CU with the most workgroups.
    auto fullest = [&](uint32_t split) { return (wgs(split) + cus - 1) / cus * ((groups + split - 1) / split); };
    if (coarse >= by32) {
        // 16 groups against 32.  Without a gate a launch of at most one
        // workgroup per CU is latency that more chunks only add to (3072x2624
        // 4.07 / 4.49); with more it depends on the fullest CU (5120x2624, 42
        // groups / 28, 4.88 / 4.64; 5120x4608, 48 / 60, 5.88 / 6.18), past two
        // chunks only a clear gain there shows (4096x4160, 44 / 39, 5.46 /
        // 5.66; 6144x4160, 66 / 52, 6.50 / 6.23), and from four per CU on the
        // finer chunks win (12288x5120 10.02 / 9.53), groups' where the fullest
        // CU has no more to do (12288x7168, 168 / 176, 11.90 / 12.43).
        if (!gate && wgs(by32) < 4ull * cus)
            return wgs(by32) > cus && (by32 == 2 ? fullest(fine) <= fullest(coarse)
                                                 : 100 * fullest(fine) < 87 * fullest(coarse))
                       ? fine : coarse;
        if (!gate && kind == LaunchKind::kGroup && by32 > 2 && fullest(fine) > fullest(coarse)) return coarse;
        // With a gate they win unless the fullest CU gets much more to do
        // (2720x4608, 24 / 30 groups, 6.49 / 6.65; 5120x4160, 44 / 52, 8.57 /
        // 8.91; 6144x6208, 75 / 84, 12.06 / 11.77).
        return !gate || by32 <= 2 || by16 == 2 * by32 || 8 * fullest(fine) <= 9 * fullest(coarse) ? fine : coarse;
    }
    // Tall matrices: up to 32 workgroups per CU of short chunks run ahead of
    // six of longer ones (28672x8192 27.5 / 23.5, 9216x16384 20.6 / 17.3;
    // 32768x2624 with a gate 24.9 / 19.7).  Coarse chunks of more than 64
    // groups, which only single launches run, go through the pipelined loop,
    // which pads nothing: against it 16-group chunks must fill their waves
    // (32768x4160, 13 of 16, 16.6 / 17.7; 32768x6208, 14, 23.1 / 23.4;
    // 49152x4608, 15, 25.3 / 25.5; 32768x5120, 16, 19.9 / 18.9), and 32-group
    // chunks with a gate (32768x8256, 26 of 32, 53.8 / 59.4; 12800x12352, 28,
    // 35.2 / 37.6; 12800x14400, 29, 42.6 / 41.6).
    // One chunk of a group with a gate, of up to 64 groups, is not cut into
    // 32-group ones (49152x4096 39.6 / 41.6).
    if (gate && !finer && groups <= 64 && coarse == 1) return coarse;
    if (kind == LaunchKind::kSingle && groups > 64 * coarse) {
        if (finer ? 100 * groups < 83 * 16 * fine : gate && 8 * groups < 7 * 32 * fine) return coarse;
    }
    return fine;
}

// Steps of 32 tiles of an item that makes `passes` passes over its groups.
// Single vectors: a step of a wave is a quad of four groups by two row tiles,
// the passes' quads are dealt to the workgroup's four waves, and the item
// takes as long as its fullest wave.  Batches: a wave's step is one group by
// eight row tiles, each pass's groups dealt from the first wave on.
static uint32_t steps_of(uint32_t batch, uint32_t groups, uint32_t passes) {
    const uint32_t quads = (groups + 3) / 4;
    return batch == 1 ? (passes * quads + 3) / 4 : passes * quads;
}

std::vector<uint32_t> item_costs(const PlanLayout &layout) {
    std::vector<uint32_t> cost(layout.items);
    for (uint32_t i = 0; i < layout.count; ++i) {
        const PlanDesc &p = layout.descs[i];
        const uint32_t g = p.cols / kGroup;
        for (uint32_t item = p.item_begin; item < layout.descs[i + 1].item_begin; ++item) {
            const uint32_t part = (item - p.item_begin) % p.per;
            const uint32_t chunk = part % p.chunks;
            const uint32_t chunk_g = std::min(g, (chunk + 1) * p.chunk_groups) - chunk * p.chunk_groups;
            const uint32_t passes = p.pair || (p.streams > 1 && p.per == 1) ? 2u : 1u;
            cost[item] = 32 * steps_of(layout.batch, chunk_g, passes) +
                         (layout.batch == 1 ? kItemEndTiles : kBatchItemEndTiles);
        }
    }
    return cost;
}

// Of the two workgroups a CU holds, the one dispatched first (b < CUs, as
// workgroups are dispatched in order) wins the CU's arbitration and streams
// faster: with equal loads on the Qwen3-8B stack, workgroups b >= CUs
// finished 20 us after the others (per-workgroup clock reads), so the CU ran
// its second workgroup alone at the end.  Workgroup b runs on XCD b % 8, and
// per-workgroup clock reads put some XCDs a few us ahead of others; the XCD
// weights are the mean relative time per unit of three boxes.
constexpr uint32_t kSecondSlotWeight = 1100;
constexpr uint32_t kXcdWeight[8] = {1029, 1023, 1027, 1015, 1028, 1019, 1028, 1023};

std::vector<uint32_t> workgroup_weights(uint32_t workgroups, uint32_t cus) {
    std::vector<uint32_t> weight(workgroups, 1024);
    for (uint32_t b = cus; b < workgroups; ++b) weight[b] = kSecondSlotWeight;
    for (uint32_t b = 0; b < workgroups; ++b) weight[b] = weight[b] * kXcdWeight[b % 8] / 1024;
    return weight;
}

// Items go in order, longest GEMV first, each to the workgroup that would
// finish it first; then moves and swaps of one item between the latest
// workgroup and an earlier one bring the latest forward while any does (each
// lowers the sorted vector of finish times, so this ends; it is capped
// besides).  On the Qwen3-8B stack (2,304 items of 192 groups x 64 rows, 9,792
// of 64 groups x 128 rows, 512 workgroups, equal weights) a round-robin deal
// leaves the most-loaded workgroup 53 units of 64 groups x 64 rows against a
// mean of 51.75; this one 52.
std::vector<uint32_t> deal_items(const std::vector<uint32_t> &cost, const std::vector<uint32_t> &weight) {
    const uint32_t workgroups = static_cast<uint32_t>(weight.size());
    std::vector<std::vector<uint32_t>> own(workgroups);
    std::vector<uint64_t> load(workgroups, 0);
    auto finish = [&](uint32_t b, uint64_t l) { return l * weight[b]; };
    // One heap of workgroups per distinct weight, least loaded on top.
    using Slot = std::pair<uint64_t, uint32_t>;
    using Heap = std::priority_queue<Slot, std::vector<Slot>, std::greater<Slot>>;
    std::map<uint32_t, Heap> lightest;
    for (uint32_t b = 0; b < workgroups; ++b) lightest[weight[b]].push({0, b});
    for (uint32_t i = 0; i < cost.size(); ++i) {
        Heap *best = nullptr;
        uint64_t best_t = UINT64_MAX;
        for (auto &kv : lightest) {
            const uint64_t t = (kv.second.top().first + cost[i]) * kv.first;
            if (t < best_t) best_t = t, best = &kv.second;
        }
        const uint32_t b = best->top().second;
        best->pop();
        own[b].push_back(i);
        load[b] += cost[i];
        best->push({load[b], b});
    }
    // One item of each distinct cost a workgroup holds (the candidates of a
    // move; which item of a cost moves does not change any load).
    auto kinds = [&](uint32_t b) {
        std::vector<uint32_t> k;
        for (uint32_t pos = 0; pos < own[b].size(); ++pos) {
            bool seen = false;
            for (uint32_t q : k) seen |= cost[own[b][q]] == cost[own[b][pos]];
            if (!seen) k.push_back(pos);
        }
        return k;
    };
    std::vector<uint32_t> by_time(workgroups);
    for (uint32_t round = 0; round < 4 * workgroups; ++round) {
        uint32_t a = 0;
        for (uint32_t b = 1; b < workgroups; ++b)
            if (finish(b, load[b]) > finish(a, load[a])) a = b;
        const uint64_t t_a = finish(a, load[a]);
        for (uint32_t b = 0; b < workgroups; ++b) by_time[b] = b;
        std::sort(by_time.begin(), by_time.end(),
                  [&](uint32_t x, uint32_t y) { return finish(x, load[x]) < finish(y, load[y]); });
        const std::vector<uint32_t> ka = kinds(a);
        uint64_t best_max = t_a;
        uint32_t best_b = 0, best_pa = 0, best_pb = 0;
        bool found = false;
        for (uint32_t b : by_time) {
            if (b == a || finish(b, load[b]) >= t_a) break;
            std::vector<uint32_t> kb = kinds(b);
            kb.push_back(UINT32_MAX);  // a move with nothing in return
            for (uint32_t pa : ka)
                for (uint32_t pb : kb) {
                    const uint64_t give = cost[own[a][pa]], take = pb == UINT32_MAX ? 0 : cost[own[b][pb]];
                    if (give <= take) continue;
                    const uint64_t m = std::max(finish(a, load[a] - (give - take)), finish(b, load[b] + (give - take)));
                    if (m < best_max) {
                        best_max = m;
                        best_b = b;
                        best_pa = pa;
                        best_pb = pb;
                        found = true;
                    }
                }
            if (found) break;
        }
        if (!found) break;
        const uint32_t item_a = own[a][best_pa];
        own[a].erase(own[a].begin() + best_pa);
        load[a] -= cost[item_a];
        if (best_pb != UINT32_MAX) {
            const uint32_t item_b = own[best_b][best_pb];
            own[best_b].erase(own[best_b].begin() + best_pb);
            load[best_b] -= cost[item_b];
            own[a].push_back(item_b);
            load[a] += cost[item_b];
        }
        own[best_b].push_back(item_a);
        load[best_b] += cost[item_a];
    }
    std::vector<uint32_t> deal(workgroups + 1 + cost.size());
    uint32_t k = 0;
    for (uint32_t b = 0; b < workgroups; ++b) {
        deal[b] = k;
        std::sort(own[b].begin(), own[b].end());
        for (uint32_t i : own[b]) deal[workgroups + 1 + k++] = i;
    }
    deal[workgroups] = k;
    return deal;
}

int layout_plan(const q4rdna_gemv_desc *descs, uint32_t count, uint32_t n, int device, uint32_t cus, PlanLayout *out,
                std::string *error) {
    if (out == nullptr || (descs == nullptr && count > 0))
        return fail(error, Q4RDNA_ERR_ARGUMENT, "NULL descriptors or layout");
    if (n < 1 || n > Q4RDNA_MAX_BATCH)
        return fail(error, Q4RDNA_ERR_ARGUMENT, "batch %u is outside 1..%d", n, Q4RDNA_MAX_BATCH);
    // Single vectors: 64-row blocks, kPrepBytes per group.  Batches: 256-row
    // blocks, one kBatchQuadBytesHost record per (group, quad of vectors).
    const uint32_t block_rows = n == 1 ? kBlockRows : kBatchBlockRows;
    const uint64_t prep_per_group = n == 1 ? kPrepBytes : static_cast<uint64_t>((n + 3) / 4) * kBatchQuadBytesHost;
    const uint32_t chunk_groups = n == 1 ? kChunkGroups : kBatchChunkGroups;
    for (uint32_t i = 0; i < count; ++i) {
        const q4rdna_gemv_desc &d = descs[i];
        if (d.weight.tiles == nullptr || d.x == nullptr || d.y == nullptr)
            return fail(error, Q4RDNA_ERR_ARGUMENT, "descriptor %u has a NULL pointer", i);
        if (!valid_shape(d.weight.rows, d.weight.columns) || !aligned(d.weight.tiles, 16) ||
            (d.gate_tiles != nullptr && !aligned(d.gate_tiles, 16)) || !aligned(d.x, 16) || !aligned(d.y, 4) ||
            (d.add != nullptr && !aligned(d.add, 4)))
            return fail(error, Q4RDNA_ERR_ARGUMENT, "descriptor %u: invalid shape or alignment", i);
        if (d.weight.device != device)
            return fail(error, Q4RDNA_ERR_ARGUMENT, "descriptor %u lives on device %d", i, d.weight.device);
    }
    // The GEMVs run concurrently: no y may overlap another descriptor's y,
    // x or add, and a descriptor's add is its own y or apart from it.  The
    // outputs are checked sorted by address (they must be disjoint), then
    // each input range against them by binary search.  A descriptor's x may
    // overlap its own y: the prepare launch reads every x before the sweep
    // writes any y.
    {
        struct Range {
            uintptr_t lo, hi;
            uint32_t owner;
        };
        std::vector<Range> ys(count);
        for (uint32_t i = 0; i < count; ++i) {
            const uintptr_t y0 = reinterpret_cast<uintptr_t>(descs[i].y);
            ys[i] = {y0, y0 + 4ull * n * descs[i].weight.rows, i};
        }
        std::sort(ys.begin(), ys.end(), [](const Range &a, const Range &b) { return a.lo < b.lo; });
        for (uint32_t i = 1; i < count; ++i)
            if (ys[i].lo < ys[i - 1].hi)
                return fail(error, Q4RDNA_ERR_ARGUMENT, "descriptors %u and %u: outputs overlap", ys[i - 1].owner,
                            ys[i].owner);
        // Every output that [lo, hi) meets, owner by owner.
        auto meets = [&](uintptr_t lo, uintptr_t hi, uint32_t self, bool is_add, const float *own_y) -> int {
            auto it = std::upper_bound(ys.begin(), ys.end(), lo, [](uintptr_t v, const Range &r) { return v < r.hi; });
            for (; it != ys.end() && it->lo < hi; ++it) {
                if (it->owner != self)
                    return fail(error, Q4RDNA_ERR_ARGUMENT, "descriptor %u: its %s overlaps descriptor %u's y", self,
                                is_add ? "add" : "x", it->owner);
                if (is_add && reinterpret_cast<uintptr_t>(own_y) != lo)
                    return fail(error, Q4RDNA_ERR_ARGUMENT, "descriptor %u: add overlaps y without being y", self);
            }
            return Q4RDNA_OK;
        };
        for (uint32_t i = 0; i < count; ++i) {
            const q4rdna_gemv_desc &d = descs[i];
            const uintptr_t x0 = reinterpret_cast<uintptr_t>(d.x);
            int rc = meets(x0, x0 + 4ull * n * d.weight.columns, i, false, d.y);
            if (rc == Q4RDNA_OK && d.add != nullptr) {
                const uintptr_t a0 = reinterpret_cast<uintptr_t>(d.add);
                rc = meets(a0, a0 + 4ull * n * d.weight.rows, i, true, d.y);
            }
            if (rc != Q4RDNA_OK) return rc;
        }
    }
    PlanLayout L;
    L.count = count;
    L.batch = n;
    // The GEMVs of a plan are independent, so the sweep may take them in any
    // order: GEMVs with longer items (wider K chunks) go first, so that the
    // end of the sweep, where workgroups run out of items, deals short ones.
    L.order.resize(count);
    for (uint32_t i = 0; i < count; ++i) L.order[i] = i;
    // Items are as large as the plan's work allows: `share` is the steps of a
    // workgroup if all ran the same number.
    const uint64_t workgroups = uint64_t(cus) * kPlanWorkgroupsPerCu;
    uint64_t steps = 0;
    for (uint32_t i = 0; i < count; ++i)
        steps += static_cast<uint64_t>((descs[i].weight.rows + block_rows - 1) / block_rows) *
                 steps_of(n, descs[i].weight.columns / kGroup, descs[i].gate_tiles != nullptr ? 2 : 1);
    const double share = static_cast<double>(steps) / static_cast<double>(workgroups);
    // Items well beyond a share are cut (a SwiGLU site into its streams; a
    // batch's rows also into K chunks of about a share): the other workgroups
    // are done before them, which costs more than the parts' meeting in
    // memory.  Batches, us per step at N = 2 / 8, whole items against these:
    // one Qwen3-8B layer (share 5.8) 78 / 94 against 33 / 44, four (share 23)
    // 104 / 105 against 88 / 96; cutting from 1.25 shares on took 118 instead
    // of 115 at an eighth of Qwen3-8B's widths (share 26) and N = 8.  A single
    // vector's K chunks are not cut: its sums do not depend on the plan.
    auto too_long = [&](uint32_t item) { return item > (n == 1 ? 2.0 : 1.6) * share; };
    auto chunk_of = [&](uint32_t i) {
        const uint32_t g = descs[i].weight.columns / kGroup;
        if (n == 1 || !too_long(steps_of(n, std::min(g, chunk_groups), 1))) return chunk_groups;
        const uint32_t least = share < 2.0 ? kMinBatchChunkGroups / 2 : kMinBatchChunkGroups;
        const uint32_t most = std::min(chunk_groups, std::max(least, 4 * static_cast<uint32_t>(share)));
        const uint32_t chunks = (g + most - 1) / most;
        return ((g + chunks - 1) / chunks + 3) / 4 * 4;
    };
    // A SwiGLU GEMV whose rows fit one chunk runs both weight streams in one
    // item per block (no split-K partials), single vectors and batches alike.
    // That saves the two streams' meeting in memory, about two steps' time;
    // beyond twice the share the item costs more than that (the other
    // workgroups are done before it) and the streams are items of their own.
    auto both_streams = [&](uint32_t i) {
        const uint32_t g = descs[i].weight.columns / kGroup;
        return descs[i].gate_tiles != nullptr && g <= chunk_of(i) && !too_long(steps_of(n, g, 2));
    };
    // A single-vector GEMV with no gate whose rows fit one 64-group step
    // block runs two 64-row blocks per item: half the item ends.  One block
    // costs nothing else, so two are taken only up to half a share: two
    // Qwen3-8B layers (share 11.5 steps) run in 37.4 us instead of 42.6, eight
    // layers of 1024 and 2816 columns (share 2.7) in 14.7 instead of 17.1; at
    // four Qwen3-8B layers both measure 67.8.
    auto pairs = [&](uint32_t i) {
        const uint32_t g = descs[i].weight.columns / kGroup;
        const uint32_t pair_steps = steps_of(n, g, 2);
        return n == 1 && descs[i].gate_tiles == nullptr && g <= kPairGroups &&
               (pair_steps <= 1 || pair_steps <= 0.5 * share);
    };
    auto item_groups = [&](uint32_t i) {
        return std::min(descs[i].weight.columns / kGroup, chunk_of(i)) * (both_streams(i) || pairs(i) ? 2u : 1u);
    };
    std::stable_sort(L.order.begin(), L.order.end(),
                     [&](uint32_t a, uint32_t b) { return item_groups(a) > item_groups(b); });
    L.descs.assign(static_cast<size_t>(count) + 1, PlanDesc{});
    L.prep_off.assign(count, 0);
    L.part_off.assign(count, 0);
    L.cnt_off.assign(count, 0);
    uint64_t items = 0, groups = 0, tail = 0;
    for (uint32_t i = 0; i < count; ++i) {
        const q4rdna_gemv_desc &d = descs[L.order[i]];
        const uint32_t g = d.weight.columns / kGroup;
        const uint32_t chunk = chunk_of(L.order[i]);
        const uint32_t chunks = (g + chunk - 1) / chunk;
        const bool pair = pairs(L.order[i]);
        const uint32_t item_rows = pair ? 2 * block_rows : block_rows;
        const uint32_t blocks = (d.weight.rows + item_rows - 1) / item_rows;
        const uint32_t streams = d.gate_tiles != nullptr ? 2u : 1u;
        PlanDesc &p = L.descs[i];
        p.w = d.weight.tiles;
        p.gate = d.gate_tiles;
        p.x = d.x;
        p.add = d.add;
        p.y = d.y;
        p.rows = d.weight.rows;
        p.cols = d.weight.columns;
        p.item_begin = static_cast<uint32_t>(items);
        p.group_begin = static_cast<uint32_t>(groups);
        p.chunks = chunks;
        p.streams = streams;
        p.per = both_streams(L.order[i]) || pair ? 1u : chunks * streams;
        p.pair = pair ? 1u : 0u;
        p.chunk_groups = chunk;
        L.prep_off[i] = groups * prep_per_group;
        if (p.per > 1) {
            L.part_off[i] = tail;
            tail = align256(tail + static_cast<uint64_t>(chunks) * streams * n * d.weight.rows * sizeof(float));
            L.cnt_off[i] = tail;
            tail += static_cast<uint64_t>(blocks) * sizeof(uint32_t);
        }
        tail = align256(tail);
        items += static_cast<uint64_t>(blocks) * p.per;
        groups += g;
        if (items > 0xffffffffull || groups * n > 0xffffffffull)
            return fail(error, Q4RDNA_ERR_ARGUMENT, "plan too large");
        L.both_streams |= p.streams > 1 && p.per == 1;
    }
    L.descs[count].item_begin = static_cast<uint32_t>(items);
    L.descs[count].group_begin = static_cast<uint32_t>(groups);
    L.items = static_cast<uint32_t>(items);
    L.groups = static_cast<uint32_t>(groups);
    // Group table of the prep launch: single vectors get each group's
    // activation address (one load, no descriptor lookup); batches the
    // descriptor index of each group.
    L.table_off = align256(groups * prep_per_group);
    L.table_bytes = groups * (n == 1 ? sizeof(uint64_t) : sizeof(uint32_t));
    L.workgroups = static_cast<uint32_t>(
        std::max<uint64_t>(1, std::min<uint64_t>(uint64_t(cus) * kPlanWorkgroupsPerCu, items)));
    // After the group table, the items' deal to the workgroups in the
    // kernels' form: the offsets (padded to an even count), then per item its
    // descriptor index and its index within the descriptor.
    const std::vector<uint32_t> lists = deal_items(item_costs(L), workgroup_weights(L.workgroups, cus));
    const uint32_t head = (L.workgroups + 2) & ~1u;
    L.deal.assign(head + 2 * items, 0);
    std::copy(lists.begin(), lists.begin() + L.workgroups + 1, L.deal.begin());
    std::vector<uint32_t> owner(items);
    for (uint32_t i = 0; i < count; ++i)
        for (uint32_t item = L.descs[i].item_begin; item < L.descs[i + 1].item_begin; ++item) owner[item] = i;
    for (uint64_t k = 0; k < items; ++k) {
        const uint32_t item = lists[L.workgroups + 1 + k];
        L.deal[head + 2 * k] = owner[item];
        L.deal[head + 2 * k + 1] = item - L.descs[owner[item]].item_begin;
    }
    L.deal_off = align256(L.table_off + L.table_bytes);
    L.tail_off = align256(L.deal_off + L.deal.size() * sizeof(uint32_t));
    L.scratch_bytes = L.tail_off + tail;
    L.table.assign(n == 1 ? groups : (groups + 1) / 2, 0);
    for (uint32_t i = 0; i < count; ++i)
        for (uint32_t g = L.descs[i].group_begin; g < L.descs[i + 1].group_begin; ++g) {
            if (n == 1)
                L.table[g] = reinterpret_cast<uint64_t>(L.descs[i].x + static_cast<size_t>(g - L.descs[i].group_begin) * kGroup);
            else
                reinterpret_cast<uint32_t *>(L.table.data())[g] = i;
        }
    *out = std::move(L);
    return Q4RDNA_OK;
}

}  // namespace host
}  // namespace q4rdna
