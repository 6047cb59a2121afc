// A decode step (no more tokens than sequences) in one launch: every workgroup finds its share of the keys for itself, folds it
// with the loop for few rows (paged_narrow.hip.h), and the last of a row's shares to be done merges them.
//
// A sequence's rows go sixteen to a unit (a token's query heads of a kv head, or a few tokens').  Units are shared out over
// `row_tiles` workgroups a kv head: shares of one length for all of them, so that a long sequence beside short ones does not set
// the time by itself, the length being what the paging vectors say there is over the workgroups that are left when every unit
// has one.  No merge kernel and no kernel in front that looks at the paging vectors: for few sequences the launches of those
// (and the gaps around them) were most of a step.
//
// What bounds it is a chain of round trips to memory: the paging vectors, the page ids, the first keys, and where a unit is
// shared out four more (its rows out, its word out, the words in, the rows in), which is why a unit of up to kStepWholeTiles is not.
// One token of 32 / 8 heads x 128, device time over 700 MB of caches: 100 keys 7.7 us, 800 13.5, 2000 14.5, 32000 31 (three launches:
// 12.4, 12.9, 13.6, 34); sixteen of 16 to 700 keys 14.7 (16.7).  The figures of whole calls stand at `decode_step_entries`.
#pragma once

#include "paged_locate.hip.h"
#include "paged_narrow.hip.h"

namespace {

constexpr int kStepChunks = kStepMostSequences / 64;
static_assert(kStepMostSequences % 64 == 0 && kStepRows == kNarrowRows, "limits");
constexpr unsigned int kStepMostShares = 64;     // of a unit
constexpr unsigned int kStepLeastTiles = 4;      // of 64 keys, to a share
// As many tiles as a unit may have that is not shared out.  Eleven or fourteen on eight waves, many steps in turn over 700 MB of
// caches: 32 / 8 heads x 128, one sequence of 800 keys 13.8 / 15.5 us, eight of 700 to 900 16.1 / 17.8; x 64 11.8 / 11.2, 13.8 / 13.8.
template <unsigned int WAVES>
constexpr unsigned int kStepWholeTiles = WAVES == 8 && kHeadDim > 64 ? 11 : 14;

// A unit's share: rows 16 row_tile .. of the sequence, tiles [first_tile, end_tile) of its keys; `shares` neighbouring entries,
// this one the `share`-th.
struct StepPlace {
    SequenceSpan span;
    unsigned int row_tile, share, shares, first_tile, end_tile;
};

template <int FORM, unsigned int WAVES>
SINGE_DEVICE bool place_step(const PagedAttentionArgs& a, unsigned int entry, StepPlace& place) {
    const unsigned int lane = threadIdx.x & 63u, groups = a.heads / a.kv_heads;
    const bool windowed = a.window >= 0;
    const unsigned int window = !windowed ? 0u : a.window > 0x7fffffffll ? 0x7fffffffu : static_cast<unsigned int>(a.window);
    SequenceSpan spans[kStepChunks];
    unsigned int units[kStepChunks], first_tile[kStepChunks], tiles[kStepChunks];
    bool any_bad = false;
    unsigned int mine_units = 0, mine_longest = 0;
    float mine_tiles = 0.0f;  // (for the length of the shares only, which allows for its rounding)
#pragma unroll
    for (int c = 0; c < kStepChunks; ++c) {
        units[c] = first_tile[c] = tiles[c] = 0;
        spans[c] = SequenceSpan{};
        if (64u * c >= a.sequences) continue;
        const unsigned int s = 64u * c + lane;
        if (s < a.sequences) {
            spans[c] = load_span<FORM>(s, a.query_offsets, a.page_offsets, a.last_page_lengths, nullptr, a.tokens, a.page_table, a.page_size);
            bool bad;
            units[c] = row_tiles_of<FORM, kNarrowRows>(a.query_offsets, nullptr, a.tokens, groups, s, bad);
            any_bad |= bad;
            const unsigned int queries = spans[c].queries, keys = spans[c].keys;
            if (queries != 0) {
                // (keys below `low` - window are hidden from every row of the sequence)
                const unsigned int low = (keys > queries ? keys - queries : 0u) + 1u;
                first_tile[c] = windowed && low > window ? (low - window) / kKeyTile : 0u;
                tiles[c] = (keys + kKeyTile - 1u) / kKeyTile - first_tile[c];
            }
            mine_units += units[c];
            mine_tiles += static_cast<float>(units[c]) * static_cast<float>(tiles[c]);
            mine_longest = mine_longest > tiles[c] ? mine_longest : tiles[c];
        }
    }
    unsigned int length = ~0u;
    if (!__any(any_bad) && a.share_done != nullptr) {
        auto add = [](auto x, auto y) { return x + y; };
        const unsigned int all_units = across_wave(mine_units, add), longest = across_wave(mine_longest, [](unsigned int x, unsigned int y) { return x > y ? x : y; });
        const float all_tiles = across_wave(mine_tiles, add);
        // Shares of `length` tiles are at most all tiles / length and one more a unit.
        if (a.row_tiles > all_units) {
            const float enough = 1.0001f * all_tiles / static_cast<float>(a.row_tiles - all_units) + 1.0f;
            length = enough < static_cast<float>(longest) ? static_cast<unsigned int>(enough) : longest;
            const unsigned int least = (longest + kStepMostShares - 1u) / kStepMostShares;
            length = length > least ? length : least;
            length = __builtin_amdgcn_readfirstlane(length > kStepLeastTiles ? length : kStepLeastTiles);
        }
    }
    unsigned int left = a.row_tiles;
#pragma unroll
    for (int c = 0; c < kStepChunks; ++c) {
        if (64u * c >= a.sequences) break;
        const unsigned int shares = tiles[c] <= (length > kStepWholeTiles<WAVES> ? length : kStepWholeTiles<WAVES>) ? 1u : (tiles[c] - 1u) / length + 1u;
        const unsigned int mine = units[c] * shares, through = sums_through_lane(mine), total = __builtin_amdgcn_readlane(through, 63);
        if (entry >= total) {
            entry -= total;
            left -= total;
            continue;
        }
        const unsigned int owner = static_cast<unsigned int>(__builtin_ctzll(__ballot(entry < through)));
        const unsigned int owner_through = __builtin_amdgcn_readlane(through, owner);
        if (owner_through > left) return false;  // (only behind offsets that make no sense: see bad_queries)
        const unsigned int within = entry - (owner_through - __builtin_amdgcn_readlane(mine, owner));
        place.shares = __builtin_amdgcn_readlane(shares, owner);
        place.row_tile = within / place.shares;
        place.share = within - place.row_tile * place.shares;
        auto owners = [&](unsigned int value) __attribute__((always_inline)) { return static_cast<unsigned int>(__builtin_amdgcn_readlane(value, owner)); };
        auto owners_wide = [&](long long value) __attribute__((always_inline)) {
            const unsigned long long bits = static_cast<unsigned long long>(value);
            return static_cast<long long>(static_cast<unsigned long long>(owners(static_cast<unsigned int>(bits >> 32))) << 32 | owners(static_cast<unsigned int>(bits)));
        };
        place.span.query_start = owners_wide(spans[c].query_start);
        place.span.page_start = owners_wide(spans[c].page_start);
        place.span.queries = owners(spans[c].queries);
        place.span.keys = owners(spans[c].keys);
        place.span.valid = owners(spans[c].valid ? 1u : 0u) != 0u;
        const unsigned int first = owners(first_tile[c]), end = first + owners(tiles[c]);
        // (cut evenly: a unit of fifteen tiles takes eight and seven, not fourteen and one with a merge behind them)
        const unsigned int each = (end - first + place.shares - 1u) / place.shares;
        place.first_tile = first + place.share * each;
        place.end_tile = end - place.first_tile < each ? end : place.first_tile + each;
        return true;
    }
    return false;
}

// Words that workgroups on other XCDs read or have written: past the caches that the XCDs do not share.
SINGE_DEVICE void shared_store(void* address, unsigned long long bits) {
    __hip_atomic_store(static_cast<unsigned long long*>(address), bits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
SINGE_DEVICE unsigned long long shared_load(const void* address) {
    return __hip_atomic_load(static_cast<const unsigned long long*>(address), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
SINGE_DEVICE unsigned long long two_floats(float low, float high) {
    return static_cast<unsigned long long>(__builtin_bit_cast(unsigned int, high)) << 32 | __builtin_bit_cast(unsigned int, low);
}

// Until this wave's own are where the others see them.
SINGE_DEVICE void shared_stores_landed() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

template <int FORM, class Half, unsigned int WAVES>
SINGE_DEVICE void decode_step_body(const PagedAttentionArgs& a, unsigned char* lds) {
    constexpr unsigned int kThreads = 64u * WAVES;
    const unsigned int groups = a.heads / a.kv_heads, tid = threadIdx.x;
    if (blockIdx.x >= a.kv_heads * a.row_tiles) {
        clear_unowned_tokens<FORM, kThreads, kNarrowRows>(reinterpret_cast<unsigned int*>(lds), kThreads * (blockIdx.x - a.kv_heads * a.row_tiles), a.query_offsets,
                                                     a.page_offsets, a.last_page_lengths, a.tokens, a.sequences, a.page_table, a.page_size, groups,
                                                     a.row_tiles, a.output, a.heads * kHeadDim * 2u, a.lse, a.heads, a.status);
        return;
    }
    const unsigned int entry = blockIdx.x / a.kv_heads, kv_head = blockIdx.x - entry * a.kv_heads;
    StepPlace place;
    if (!place_step<FORM, WAVES>(a, entry, place)) return;
    const SequenceSpan& span = place.span;
    if (!span.valid) {
        if (tid == 0) report_index_error(a.status);
        return;
    }
    const unsigned int packed = span.queries * groups, first_row = place.row_tile * kNarrowRows;
    if (first_row >= packed) return;
    const unsigned int rows = packed - first_row < kNarrowRows ? packed - first_row : kNarrowRows;
    const bool shared = place.shares > 1u;
    // The keys of the share that the unit's rows see: from the sixteen that hold the first one inside the window of its first
    // row, up to its last row's position.
    auto position_of = [&](unsigned int row) __attribute__((always_inline)) {
        const long long position = static_cast<long long>(span.keys) - static_cast<long long>(span.queries) + row / groups;
        return position < 0 ? 0u : static_cast<unsigned int>(position);
    };
    unsigned int key_begin = place.first_tile * kKeyTile, key_end = place.end_tile * kKeyTile < span.keys ? place.end_tile * kKeyTile : span.keys;
    if (a.causal != 0) {
        const unsigned int reach = position_of(first_row + rows - 1u) + 1u;
        key_end = key_end < reach ? key_end : reach;
    }
    if (a.window >= 0) {
        const unsigned int window = a.window > 0x7fffffffll ? 0x7fffffffu : static_cast<unsigned int>(a.window), low = position_of(first_row) + 1u;
        const unsigned int seen = low > window ? (low - window) & ~(kNarrowKeys - 1u) : 0u;
        key_begin = key_begin > seen ? key_begin : seen;
    }
    // A share leaves its rows normalised, with a log-sum-exp each, in its own place of the scratch.
    constexpr unsigned int kShareFloats = kNarrowRows * kHeadDim;
    float* const partial = a.partial_out + static_cast<size_t>(blockIdx.x) * kShareFloats;
    float* const partial_lse = a.partial_lse + static_cast<size_t>(blockIdx.x) * (2u * kNarrowRows);
    auto flat_of = [&](unsigned int row) __attribute__((always_inline)) {
        const unsigned int r = first_row + row;
        return (static_cast<size_t>(span.query_start) + r / groups) * a.heads + kv_head * groups + r % groups;
    };
    auto finish = [&](unsigned int row, unsigned int quad, const float4& merged, float lse2) __attribute__((always_inline)) {
        if (shared) {
            shared_store(partial + row * kHeadDim + 4u * quad, two_floats(merged.x, merged.y));
            shared_store(partial + row * kHeadDim + 4u * quad + 2u, two_floats(merged.z, merged.w));
            if (quad == 0) shared_store(partial_lse + 2u * row, two_floats(lse2, 0.0f));
        } else {
            const size_t flat = flat_of(row);
            *reinterpret_cast<uint2*>(a.output + flat * kHeadDim + 4u * quad) =
                make_uint2(pack_pair(Half{}, merged.x, merged.y), pack_pair(Half{}, merged.z, merged.w));
            if (a.lse != nullptr && quad == 0) a.lse[flat] = lse2;
        }
    };
    narrow_rows<false, FORM, true, WAVES, Half>(a, lds, span, kv_head, first_row, rows, key_begin, key_end, finish);
    if (!shared) return;

    // Everything a share leaves is where the others see it before its word says so, and its word before it looks at theirs: of
    // a unit's workgroups at least the one whose word came last sees all of them.  (Another that does too writes the same rows.)
    // The words hold the launch's own number, which nothing left in the scratch by an earlier use does, and are cleared by who
    // has seen them, so that a captured launch finds none of its own when it is played again.
    shared_stores_landed();
    __syncthreads();
    const unsigned int first_block = blockIdx.x - place.share * a.kv_heads;  // of the unit's first share; the others a.kv_heads on
    if (tid < 64u) {
        if (tid == 0) shared_store(a.share_done + blockIdx.x, a.launch_number);
        shared_stores_landed();
        const bool done = tid >= place.shares || shared_load(a.share_done + first_block + tid * a.kv_heads) == a.launch_number;
        if (tid == 0) reinterpret_cast<unsigned int*>(lds)[0] = 0u;
        if (__all(done) && tid == 0) reinterpret_cast<unsigned int*>(lds)[0] = 1u;
    }
    __syncthreads();
    if (reinterpret_cast<unsigned int*>(lds)[0] == 0u) return;
    // Each share's rows weigh 2^(lse - largest) over the sum of those.  A row's values are asked for before the weights are
    // worked out, sixteen shares a thread, and where the rows leave threads over, several take turns at a row's shares.  What a
    // share that sees no key of the row holds is not used (its weight is kNoWeight, and past the last share too); a log-sum-exp
    // that is NaN makes the row NaN.
    constexpr unsigned int kQuads = kHeadDim / 4u, kAtOnce = 16;
    constexpr float kNoWeight = -1.0f;
    float* const weights = reinterpret_cast<float*>(lds) + 4;               // [rows][kStepMostShares]
    float* const row_lse = weights + kNarrowRows * kStepMostShares;         // [rows]
    float4* const sums = reinterpret_cast<float4*>(row_lse + kNarrowRows);  // [kThreads]
    const unsigned int wave = tid >> 6, lane = tid & 63u, shares = place.shares, items = rows * kQuads;
    const unsigned int turns = items >= kThreads ? 1u : kThreads / items, turn = items >= kThreads ? 0u : tid / items;
    const size_t stride = static_cast<size_t>(a.kv_heads) * kShareFloats;
    const float* const first_partial = a.partial_out + static_cast<size_t>(first_block) * kShareFloats;
    unsigned long long low[kAtOnce], high[kAtOnce];
    auto ask = [&](unsigned int item, unsigned int from_share) __attribute__((always_inline)) {
#pragma unroll
        for (unsigned int i = 0; i < kAtOnce; ++i) {
            const unsigned int s = from_share + i * turns;
            if (s < shares) {
                const float* share = first_partial + s * stride + (item / kQuads) * kHeadDim + 4u * (item % kQuads);
                low[i] = shared_load(share);
                high[i] = shared_load(share + 2);
            }
        }
    };
    auto fold = [&](float4& merged, unsigned int item, unsigned int from_share) __attribute__((always_inline)) {
#pragma unroll
        for (unsigned int i = 0; i < kAtOnce; ++i) {
            const unsigned int s = from_share + i * turns;
            const float w = s < shares ? weights[(item / kQuads) * kStepMostShares + s] : kNoWeight;
            auto part = [&](unsigned long long bits) __attribute__((always_inline)) { return __builtin_bit_cast(float, static_cast<unsigned int>(bits)); };
            merged.x = w == kNoWeight ? merged.x : fmaf(w, part(low[i]), merged.x);
            merged.y = w == kNoWeight ? merged.y : fmaf(w, part(low[i] >> 32), merged.y);
            merged.z = w == kNoWeight ? merged.z : fmaf(w, part(high[i]), merged.z);
            merged.w = w == kNoWeight ? merged.w : fmaf(w, part(high[i] >> 32), merged.w);
        }
    };
    const bool working = turn < turns;
    const unsigned int first_item = items >= kThreads ? tid : tid - turn * items;
    if (working) ask(first_item, turn);
    for (unsigned int row = wave; row < rows; row += WAVES) {
        const float mine = lane < shares ? __builtin_bit_cast(float, static_cast<unsigned int>(shared_load(
                                               a.partial_lse + static_cast<size_t>(first_block + lane * a.kv_heads) * (2u * kNarrowRows) + 2u * row)))
                                         : -INFINITY;
        const float largest = across_wave(mine, [](float x, float y) { return fmaxf(x, y); });
        const float weight = mine == -INFINITY ? 0.0f : fast_exp2(mine - largest);
        const float total = across_wave(weight, [](float x, float y) { return x + y; });
        weights[row * kStepMostShares + lane] = mine == -INFINITY ? kNoWeight : weight * (1.0f / total);
        if (lane == 0) row_lse[row] = total == 0.0f ? -INFINITY : largest + fast_log2(total);
    }
    __syncthreads();
    for (unsigned int item = first_item; item < items; item += kThreads) {
        float4 merged = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (working) {
            if (item != first_item) ask(item, turn);
            fold(merged, item, turn);
            for (unsigned int s = turn + kAtOnce * turns; s < shares; s += kAtOnce * turns) {
                ask(item, s);
                fold(merged, item, s);
            }
        }
        if (turns == 1u && !working) break;
        if (turns > 1u) {
            sums[tid] = merged;
            __syncthreads();
            if (tid >= items) break;
            for (unsigned int t = 1; t < turns; ++t) {
                const float4 other = sums[tid + t * items];
                merged.x += other.x;
                merged.y += other.y;
                merged.z += other.z;
                merged.w += other.w;
            }
        }
        const size_t flat = flat_of(item / kQuads);
        *reinterpret_cast<uint2*>(a.output + flat * kHeadDim + 4u * (item % kQuads)) =
            make_uint2(pack_pair(Half{}, merged.x, merged.y), pack_pair(Half{}, merged.z, merged.w));
        if (a.lse != nullptr && item % kQuads == 0) a.lse[flat] = row_lse[item / kQuads];
    }
    if (tid < shares) shared_store(a.share_done + first_block + tid * a.kv_heads, 0ull);
}

}  // namespace
