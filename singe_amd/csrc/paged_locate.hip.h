// Which (sequence, kv head, row tile, key split) a workgroup of the paged attention kernels works on.
#pragma once

#include "kernel_args.h"
#include "paging.hip.h"

namespace {

// The kernels' argument block where it lies (the block is their only parameter).
typedef PagedAttentionArgs __attribute__((address_space(4))) arguments_t;

constexpr unsigned int kNoPage = 0xFFFFFFFFu;  // a table entry outside the cache: reported, never read through

// Workgroup id -> (unit = sequence * kv_heads + kv head, row tile, key split); false for ids past the units.
// Workgroup i runs on XCD i % 8: the row tiles of one (sequence, kv head) share an XCD and its L2.
//
// Plain form (a.compact == 0; calls where no sequence can have more than one row tile, decoding above all): the grid
// covers every sequence's longest possible run of rows.  Within an XCD the order is band by band of 32 row tiles:
// every unit's tiles 0 .. 31 (a unit's side by side, walking its keys together), then every unit's tiles 32 .. 63,
// and so on.  The splits of one (unit, row tile) are neighbours.
//
// Compact form (a.compact != 0): the row tiles of all sequences form one list in sequence order (or longest sequence
// first, see a.longest_first), sequence s owning
// max(1, ceil(queries_s * groups / ROWS)) of them (ROWS: the rows of a workgroup, 128 or 256) (one even without queries, so that its paging values are checked),
// and the grid covers a bound on the list's length instead of sequences x the longest possible sequence; a workgroup
// finds its entry by a prefix sum over the sequences' query counts, 64 sequences at a time.  The list is cut into
// bands of 32 entries; (band, kv head) pairs go round the XCDs, so a band's tiles for one kv head are neighbours on
// one XCD and walk their keys side by side.
// a.longest_first (at most 64 sequences, several row tiles each: chunks of a prefill): the compact list takes the
// sequences longest first (by pages held, ties by index), so that the workgroups with the most keys to walk start
// first and the short ones fill the chip's last round.  Lane s learns how many list entries come before sequence s's
// own (`mine` of them) in that order.  (Decode-shaped calls keep the sequences' own order: their workgroups are short,
// and the two loads and the ranking in front of everything else cost them more than the order gains: 62 -> 70 us on the
// decode benchmark's shape.)
template <int FORM>
SINGE_DEVICE unsigned int entries_before_longest_first(const PagedAttentionArgs& a, unsigned int mine) {
    const unsigned int s = threadIdx.x & 63u;
    unsigned int held = 0;
    if (s < a.sequences) {
        long long count;
        if constexpr (has_lengths(FORM)) count = read_index<FORM>(a.last_page_lengths, s);  // key counts
        else count = read_index<FORM>(a.page_offsets, s + 1) - read_index<FORM>(a.page_offsets, s);
        held = count < 0 ? 0u : count > 0x7fffffffll ? 0x7fffffffu : static_cast<unsigned int>(count);
    }
    unsigned int before = 0;
    for (unsigned int other = 0; other < a.sequences; ++other) {
        const unsigned int other_held = __builtin_amdgcn_readlane(held, other), other_mine = __builtin_amdgcn_readlane(mine, other);
        if (other_held > held || (other_held == held && other < s)) before += other_mine;
    }
    return before;
}

// a.alternate (at most 64 * kAlternateChunks sequences, some of which decode beside others that bring row tiles): the
// compact list takes the sequences of at most sixteen packed rows by themselves, longest first, and alternates runs of
// them with runs of the others' row tiles, as many of either as an XCD's compute units hold one of.  The first bring the
// cache from memory with the matrix cores all but idle (paged_narrow.hip.h), the others use the matrix cores on keys that
// the XCD's L2 holds; side by side on a compute unit they take little from each other, and a long sequence that starts last
// would run on by itself.  (Lengths are compared up to 4095 pages.)
// Finds the entry's sequence and row tile; kPastList past the list's end, kInOrder where offsets make no sense and the list
// is taken in sequence order.
enum class Alternating { kFound, kPastList, kInOrder };
constexpr int kAlternateChunks = 4;
template <int FORM, unsigned int ROWS>
SINGE_DEVICE Alternating locate_alternating(const PagedAttentionArgs& a, unsigned int entry, unsigned int& sequence, unsigned int& row_tile) {
    const unsigned int lane = threadIdx.x & 63u, groups = a.heads / a.kv_heads;
    constexpr unsigned int kMostHeld = 4095u, kHeldBits = 12u;
    unsigned long long narrow[kAlternateChunks];
    unsigned int held[kAlternateChunks], tiles[kAlternateChunks], through[kAlternateChunks];  // tiles: of wide sequences, and their inclusive prefix sums
    unsigned int narrow_count = 0, wide_count = 0;
    bool any_bad = false;
#pragma unroll
    for (int c = 0; c < kAlternateChunks; ++c) {
        narrow[c] = 0;
        held[c] = tiles[c] = through[c] = 0;
        if (64u * c >= a.sequences) continue;
        const unsigned int s = 64u * c + lane;
        bool is_narrow = false;
        if (s < a.sequences) {
            const long long start = read_index<FORM>(a.query_offsets, s), end = read_index<FORM>(a.query_offsets, s + 1);
            const long long pages = read_index<FORM>(a.page_offsets, s + 1) - read_index<FORM>(a.page_offsets, s);
            const bool bad = bad_queries<FORM>(start, end, a.tokens);
            any_bad |= bad;
            const unsigned long long rows = bad ? 0ull : static_cast<unsigned long long>(end - start) * groups;
            is_narrow = rows <= 16u;
            held[c] = pages < 0 ? 0u : pages > static_cast<long long>(kMostHeld) ? kMostHeld : static_cast<unsigned int>(pages);
            tiles[c] = is_narrow ? 0u : static_cast<unsigned int>((rows + ROWS - 1) / ROWS);
        }
        narrow[c] = __ballot(is_narrow);
        narrow_count += static_cast<unsigned int>(__builtin_popcountll(narrow[c]));
        through[c] = tiles[c];
#pragma unroll
        for (int step = 1; step < 64; step <<= 1) {
            const unsigned int below = __shfl_up(through[c], step, 64);
            if (lane >= static_cast<unsigned int>(step)) through[c] += below;
        }
        wide_count += __builtin_amdgcn_readlane(through[c], 63);
    }
    if (__any(any_bad)) return Alternating::kInOrder;
    const unsigned int run = a.kv_heads >= 256u ? 1u : 256u / a.kv_heads;
    const unsigned int narrow_runs = narrow_count / run, wide_runs = wide_count / run, pairs = narrow_runs < wide_runs ? narrow_runs : wide_runs;
    bool takes_narrow;
    unsigned int index;
    if (entry < 2u * run * pairs) {
        const unsigned int within = entry % (2u * run);
        takes_narrow = within >= run;
        index = entry / (2u * run) * run + (takes_narrow ? within - run : within);
    } else {
        const unsigned int rest = entry - 2u * run * pairs, wide_left = wide_count - run * pairs;
        takes_narrow = rest >= wide_left;
        index = run * pairs + (takes_narrow ? rest - wide_left : rest);
    }
    if (takes_narrow) {
        if (index >= narrow_count) return Alternating::kPastList;
        // The index-th longest: bit by bit from the top, keep the candidates that have the bit where enough of them do.
#pragma unroll 1
        for (int bit = kHeldBits - 1; bit >= 0; --bit) {
            unsigned long long with[kAlternateChunks];
            unsigned int count = 0;
#pragma unroll
            for (int c = 0; c < kAlternateChunks; ++c) {
                with[c] = narrow[c] == 0 ? 0ull : __ballot((held[c] >> bit & 1u) != 0u) & narrow[c];
                count += static_cast<unsigned int>(__builtin_popcountll(with[c]));
            }
            const bool enough = index < count;
            if (!enough) index -= count;
#pragma unroll
            for (int c = 0; c < kAlternateChunks; ++c) narrow[c] = enough ? with[c] : narrow[c] & ~with[c];
        }
#pragma unroll
        for (int c = 0; c < kAlternateChunks; ++c) {
            const unsigned int here = static_cast<unsigned int>(__builtin_popcountll(narrow[c]));
            if (index < here) {
                const bool mine = (narrow[c] >> lane & 1ull) != 0 && static_cast<unsigned int>(__builtin_popcountll(narrow[c] & ((1ull << lane) - 1ull))) == index;
                sequence = 64u * c + static_cast<unsigned int>(__builtin_ctzll(__ballot(mine)));
                row_tile = 0;
                return Alternating::kFound;
            }
            index -= here;
        }
        return Alternating::kPastList;
    }
#pragma unroll
    for (int c = 0; c < kAlternateChunks; ++c) {
        const unsigned int total = __builtin_amdgcn_readlane(through[c], 63);
        if (index < total) {
            const unsigned int owner = static_cast<unsigned int>(__builtin_ctzll(__ballot(index < through[c])));
            sequence = 64u * c + owner;
            row_tile = index - (__builtin_amdgcn_readlane(through[c], owner) - __builtin_amdgcn_readlane(tiles[c], owner));
            return Alternating::kFound;
        }
        index -= total;
    }
    return Alternating::kPastList;
}

// kPacked only: packed sequences may overlap, and their row tiles can then outnumber the list the grid was sized for.
// Workgroups come back for another `round` of entries as long as `more` says there may be one.
template <int FORM, unsigned int ROWS>
SINGE_DEVICE bool locate(const PagedAttentionArgs& a, unsigned int& unit, unsigned int& row_tile, unsigned int& split, unsigned int round,
                         bool& more) {
    constexpr unsigned int kBand = 32;
    const unsigned int xcd = blockIdx.x & 7u;
    unsigned int within = blockIdx.x >> 3;
    split = within % a.splits;
    within /= a.splits;
    if (a.compact != 0) {
        const unsigned int bands = (a.row_tiles + kBand - 1) / kBand;
        const unsigned int pair = xcd + 8u * (within / kBand);
        if (pair >= a.kv_heads * bands) return false;
        const unsigned int kv_head = pair % a.kv_heads;
        // (overlapping sequences can have more row tiles in all than 32 bits count)
        std::conditional_t<FORM == kPacked, unsigned long long, unsigned int> entry = (pair / a.kv_heads) * kBand + within % kBand;
        if (entry >= a.row_tiles) return false;
        if constexpr (FORM == kPacked) entry += static_cast<unsigned long long>(round) * a.row_tiles;
        more = true;
        if constexpr (FORM == kCsrI32 || FORM == kCsrI64) {
            if (a.alternate != 0) {
                unsigned int sequence;
                const Alternating found = locate_alternating<FORM, ROWS>(a, entry, sequence, row_tile);
                if (found == Alternating::kPastList) return false;
                if (found == Alternating::kFound) {
                    unit = sequence * a.kv_heads + kv_head;
                    return true;
                }
            }
        }
        const unsigned int lane = threadIdx.x & 63u, groups = a.heads / a.kv_heads;
        auto tiles_of = [&](unsigned int s, bool& bad) __attribute__((always_inline)) {
            return row_tiles_of<FORM, ROWS>(a.query_offsets, a.query_lengths, a.tokens, groups, s, bad);
        };
        bool bad = false;
        const unsigned int first_mine = a.longest_first != 0 && lane < a.sequences ? tiles_of(lane, bad) : 0u;
        if (a.longest_first != 0 && !__any(bad)) {
            const unsigned int mine = first_mine;
            const unsigned int before = entries_before_longest_first<FORM>(a, mine);
            const unsigned long long holds = __ballot(entry >= before && entry - before < mine);
            if (holds == 0) return false;
            if constexpr (FORM == kPacked) more = __ballot(before + mine > (round + 1u) * a.row_tiles) != 0;
            const unsigned int owner = static_cast<unsigned int>(__builtin_ctzll(holds));
            unit = owner * a.kv_heads + kv_head;
            row_tile = static_cast<unsigned int>(entry) - __shfl(before, owner, 64);
            // (packed prompts see as many keys as they have tokens before them: their last tiles are the long ones)
            if constexpr (FORM == kPacked) row_tile = __shfl(mine, owner, 64) - 1u - row_tile;
            return true;
        }
        // (from here on `entry` counts from the first row tile of the sequences looked at, `left` what the list holds from there)
        unsigned int left = a.row_tiles;
        for (unsigned int first = 0; first < a.sequences; first += 64u) {
            const unsigned int s = first + lane;
            const unsigned int mine = s < a.sequences ? tiles_of(s, bad) : 0u;
            unsigned int through = mine;  // inclusive prefix sum over the wave
#pragma unroll
            for (int step = 1; step < 64; step <<= 1) {
                const unsigned int below = __shfl_up(through, step, 64);
                if (lane >= static_cast<unsigned int>(step)) through += below;
            }
            const unsigned int total = __shfl(through, 63, 64);
            if (entry < total) {
                const unsigned long long holds = __ballot(entry < through);  // first lane whose range reaches the entry
                const unsigned int owner = static_cast<unsigned int>(__builtin_ctzll(holds));
                const unsigned int owner_through = __shfl(through, owner, 64), owner_mine = __shfl(mine, owner, 64);
                if (!has_lengths(FORM) && owner_through > left) return false;  // (only behind offsets that make no sense: see bad_queries)
                unit = (first + owner) * a.kv_heads + kv_head;
                row_tile = static_cast<unsigned int>(entry) - (owner_through - owner_mine);
                return true;
            }
            entry -= total;
            left -= total;
        }
        return false;
    }
    const unsigned int units_per_xcd = (a.sequences * a.kv_heads + 7u) / 8u;
    const unsigned int full_bands = a.row_tiles / kBand, band = within / (units_per_xcd * kBand);
    unsigned int local_unit;
    if (band < full_bands) {
        const unsigned int rest = within % (units_per_xcd * kBand);
        local_unit = rest / kBand;
        row_tile = band * kBand + rest % kBand;
    } else {
        const unsigned int rest = within - full_bands * units_per_xcd * kBand, tail = a.row_tiles - full_bands * kBand;
        local_unit = rest / tail;
        row_tile = full_bands * kBand + rest % tail;
    }
    unit = local_unit * 8u + xcd;
    more = false;
    return unit < a.sequences * a.kv_heads;
}

template <int FORM, unsigned int ROWS>
SINGE_DEVICE bool locate(const PagedAttentionArgs& a, unsigned int& unit, unsigned int& row_tile, unsigned int& split) {
    bool more;
    return locate<FORM, ROWS>(a, unit, row_tile, split, 0u, more);
}

}  // namespace
