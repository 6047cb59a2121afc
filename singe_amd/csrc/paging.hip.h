// Reading and checking one sequence's paging values on the device, shared by the paged kernels.
// Paging arrives as FlashInfer CSR vectors of i32 or i64 (singe/src/tensor/neural.rs:409-457), or as the
// block table of the singe-kernel surface: u32 table rows plus i32 per-sequence query offsets, query
// lengths and key lengths (singe-kernel/src/cpu/attention.rs:1248-1276).
#pragma once

#include "common.hip.h"

// kPacked: no paging at all.  Sequences packed one after the other in plain key and value tensors (ragged prefill):
// i32 per-sequence offsets (shared by a sequence's queries and keys), query lengths and key lengths.
enum : int { kCsrI32 = 0, kCsrI64 = 1, kTable = 2, kPacked = 3 };

// The forms of the singe-kernel surface: per-sequence query lengths and key lengths, queries aligned with a sequence's
// first keys, a natural-log log-sum-exp.
constexpr bool has_lengths(int form) { return form == kTable || form == kPacked; }

template <int FORM>
SINGE_DEVICE long long read_index(const void* values, size_t at) {
    if constexpr (FORM == kCsrI64)
        return static_cast<const long long*>(values)[at];
    else
        return static_cast<long long>(static_cast<const int*>(values)[at]);
}

template <int FORM>
SINGE_DEVICE unsigned long long read_page(const void* pages, size_t at) {
    if constexpr (FORM == kTable)
        return static_cast<const unsigned int*>(pages)[at];
    else
        return static_cast<unsigned long long>(read_index<FORM>(pages, at));  // negative ids wrap above any cache
}

// A page id as it sits in memory, and the load of one with no arithmetic on the result (a consumer that
// wants to keep the load in flight widens it later: static_cast<unsigned long long> sign-extends the CSR
// forms, so negative ids wrap above any cache, and zero-extends a block table's u32).
template <int FORM> struct RawPageType { typedef int type; };
template <> struct RawPageType<kCsrI64> { typedef long long type; };
template <> struct RawPageType<kTable> { typedef unsigned int type; };
template <int FORM> using RawPage = typename RawPageType<FORM>::type;

template <int FORM>
SINGE_DEVICE RawPage<FORM> read_raw_page(const void* pages, size_t at) {
    return static_cast<const RawPage<FORM>*>(pages)[at];
}

// The same load from an address every lane shares, through the constant address space (paging vectors are
// not written while a kernel that reads them runs), which lets it run on the scalar unit.
template <int FORM>
SINGE_DEVICE RawPage<FORM> read_raw_page_uniform(const void* pages, size_t at) {
    typedef const RawPage<FORM> __attribute__((address_space(4))) * constant_pages_t;
    return ((constant_pages_t)pages)[at];
}

struct SequenceSpan {
    long long query_start;  // first token of the sequence in the packed queries
    long long page_start;   // first entry of the sequence in `pages`
    unsigned int queries;
    unsigned int keys;
    bool valid;             // false: some value would address outside the queries or the page table
};

// The checks of paged_attention.rs:210-238 (CPU: spec/neural/attention.rs:372-406): offsets monotone
// inside [0, tokens] / [0, page_table], last_page_length in [0, page_size] unless the sequence has no
// pages.  keys = (page_count - 1) * page_size + last_page_length (paged_attention.rs:256).
template <int FORM>
SINGE_DEVICE SequenceSpan load_span(unsigned int sequence, const void* query_offsets, const void* page_offsets,
                                    const void* last_page_lengths, const void* query_lengths, unsigned int tokens,
                                    unsigned int page_table, unsigned int page_size) {
    SequenceSpan span;
    long long query_count, key_count;
    if constexpr (FORM == kTable) {
        span.query_start = read_index<FORM>(query_offsets, sequence);
        query_count = read_index<FORM>(query_lengths, sequence);
        key_count = read_index<FORM>(last_page_lengths, sequence);
        span.page_start = static_cast<long long>(sequence) * page_table;
        span.valid = !(span.query_start < 0 || query_count < 0 || span.query_start + query_count > static_cast<long long>(tokens) ||
                       key_count < 0 || key_count > static_cast<long long>(page_table) * page_size);
    } else if constexpr (FORM == kPacked) {
        // Counts are clamped to the tensors (`tokens` query rows, `page_table` key rows), as the one-wave-per-row kernel
        // clamps them; nothing is reported.
        span.query_start = span.page_start = read_index<FORM>(query_offsets, sequence);
        query_count = read_index<FORM>(query_lengths, sequence);
        key_count = read_index<FORM>(last_page_lengths, sequence);
        const long long rows = static_cast<long long>(tokens) - span.query_start, room = static_cast<long long>(page_table) - span.page_start;
        span.valid = span.query_start >= 0 && query_count > 0 && rows > 0;
        query_count = query_count < rows ? query_count : rows;
        key_count = key_count < room ? key_count : room;
        key_count = key_count < 0 ? 0 : key_count;
    } else {
        span.query_start = read_index<FORM>(query_offsets, sequence);
        const long long query_end = read_index<FORM>(query_offsets, sequence + 1);
        span.page_start = read_index<FORM>(page_offsets, sequence);
        const long long page_end = read_index<FORM>(page_offsets, sequence + 1);
        const long long last_length = read_index<FORM>(last_page_lengths, sequence);
        span.valid = !(span.query_start < 0 || query_end < span.query_start || query_end > static_cast<long long>(tokens) ||
                       span.page_start < 0 || page_end < span.page_start || page_end > static_cast<long long>(page_table) ||
                       (page_end > span.page_start && (last_length < 0 || last_length > static_cast<long long>(page_size))));
        query_count = query_end - span.query_start;
        const long long page_count = page_end - span.page_start;
        key_count = page_count == 0 ? 0 : (page_count - 1) * page_size + last_length;
    }
    span.queries = span.valid ? static_cast<unsigned int>(query_count) : 0u;
    span.keys = span.valid ? static_cast<unsigned int>(key_count) : 0u;
    return span;
}

// Whether a CSR sequence's query offsets make no sense (its own checks report it).  Such a sequence has one entry, and a list
// that holds one is taken in sequence order whatever the call asked for: the sequences before the first of them follow one
// another inside [0, tokens] and fit the grid, and it comes next, so the error is reported however many row tiles the
// sequences after it claim.  (Those may then lie past the grid; a sequence of which any row tile does is not attended.)
template <int FORM>
SINGE_DEVICE bool bad_queries(long long start, long long end, unsigned int tokens) {
    if constexpr (has_lengths(FORM)) return false;
    return start < 0 || end < start || end > static_cast<long long>(tokens);
}

// Entries of sequence `s` in the list; `bad` as above.
template <int FORM, unsigned int ROWS>
SINGE_DEVICE unsigned int row_tiles_of(const void* query_offsets, const void* query_lengths, unsigned int tokens, unsigned int groups,
                                       unsigned int s, bool& bad) {
    long long count;
    bad = false;
    if constexpr (has_lengths(FORM)) {
        count = read_index<FORM>(query_lengths, s);
        count = count < 0 ? 0 : count > static_cast<long long>(tokens) ? static_cast<long long>(tokens) : count;
    } else {
        const long long start = read_index<FORM>(query_offsets, s), end = read_index<FORM>(query_offsets, s + 1);
        bad = bad_queries<FORM>(start, end, tokens);
        count = bad ? 0 : end - start;
    }
    const unsigned long long tiles = (static_cast<unsigned long long>(count) * groups + ROWS - 1) / ROWS;
    return tiles == 0 ? 1u : static_cast<unsigned int>(tiles);
}

// The rows of the `THREADS` tokens from `first` on that no attended sequence owns: zeros and a log-sum-exp of -inf, for
// callers whose output holds nothing yet.  One workgroup of THREADS; `owned` is THREADS / 32 + 1 words of LDS.  No row is
// written here and by an attention workgroup as well: behind a sequence whose query offsets make no sense others may claim
// more entries of the list than the grid has (`limit`; ROWS rows of `groups` to a token each), and those are left out here by
// the rule by which they are not attended.
template <int FORM, unsigned int THREADS, unsigned int ROWS>
SINGE_DEVICE void clear_unowned_tokens(unsigned int* owned, unsigned int first, const void* query_offsets, const void* page_offsets,
                                       const void* last_page_lengths, unsigned int tokens, unsigned int sequences, unsigned int page_table,
                                       unsigned int page_size, unsigned int groups, unsigned int limit, void* output, unsigned int token_bytes,
                                       float* lse, unsigned int heads, unsigned int* status) {
    constexpr unsigned int kWords = THREADS / 32u;
    const unsigned int tid = threadIdx.x;
    auto span_of = [&](unsigned int s) __attribute__((always_inline)) {
        return load_span<FORM>(s, query_offsets, page_offsets, last_page_lengths, nullptr, tokens, page_table, page_size);
    };
    auto mark = [&](const SequenceSpan& span) __attribute__((always_inline)) {
        if (!span.valid || span.queries == 0) return;
        const long long from = span.query_start - static_cast<long long>(first), until = from + span.queries;
        const unsigned int low = from < 0 ? 0u : from > static_cast<long long>(THREADS) ? THREADS : static_cast<unsigned int>(from);
        const unsigned int high = until < 0 ? 0u : until > static_cast<long long>(THREADS) ? THREADS : static_cast<unsigned int>(until);
        for (unsigned int word = low / 32u; word * 32u < high; ++word) {
            const unsigned int begin = word * 32u < low ? low - word * 32u : 0u, end = high - word * 32u < 32u ? high - word * 32u : 32u;
            if (begin < end) atomicOr(&owned[word], (end == 32u ? ~0u : (1u << end) - 1u) & ~((1u << begin) - 1u));
        }
    };
    if (tid <= kWords) owned[tid] = 0u;
    __syncthreads();
    for (unsigned int s = tid; s < sequences; s += THREADS) {
        const SequenceSpan span = span_of(s);
        if (bad_queries<FORM>(span.query_start, read_index<FORM>(query_offsets, s + 1), tokens)) atomicOr(&owned[kWords], 1u);
        mark(span);
    }
    __syncthreads();
    if (owned[kWords] != 0u) {
        if (tid == 0) report_index_error(status);
        if (tid < kWords) owned[tid] = 0u;
        __syncthreads();
        if (tid < 64u) {
            unsigned int left = limit;
            for (unsigned int chunk = 0; chunk < sequences; chunk += 64u) {
                const unsigned int s = chunk + tid;
                bool bad;
                unsigned int through = s < sequences ? row_tiles_of<FORM, ROWS>(query_offsets, nullptr, tokens, groups, s, bad) : 0u;
#pragma unroll
                for (int step = 1; step < 64; step <<= 1) {
                    const unsigned int below = __shfl_up(through, step, 64);
                    if (tid >= static_cast<unsigned int>(step)) through += below;
                }
                if (s < sequences && through <= left) mark(span_of(s));
                const unsigned int total = __shfl(through, 63, 64);
                if (total > left) break;
                left -= total;
            }
        }
        __syncthreads();
    }
    for (unsigned int word = 0; word < kWords; ++word) {
        for (unsigned int left = ~owned[word]; left != 0u; left &= left - 1u) {
            const unsigned int token = first + word * 32u + static_cast<unsigned int>(__builtin_ctz(left));
            if (token >= tokens) return;
            unsigned char* row = static_cast<unsigned char*>(output) + static_cast<size_t>(token) * token_bytes;
            for (unsigned int at = tid * 8u; at < token_bytes; at += THREADS * 8u) *reinterpret_cast<uint2*>(row + at) = make_uint2(0u, 0u);
            if (lse != nullptr)
                for (unsigned int head = tid; head < heads; head += THREADS) lse[static_cast<size_t>(token) * heads + head] = -INFINITY;
        }
    }
}

// Packed sequences may overlap, and then the last one that owns a token writes its rows, as the CPU loop's later writes
// win.  Whether any sequence after `sequence` reaches into its `queries` tokens (the same answer in every lane) ...
SINGE_DEVICE bool later_sequence_overlaps(const void* offsets, const void* query_lengths, unsigned int sequences, unsigned int sequence,
                                          long long start, unsigned int queries) {
    bool any = false;
    for (unsigned int first = sequence + 1; first < sequences; first += 64u) {
        const unsigned int s = first + (threadIdx.x & 63u);
        bool mine = false;
        if (s < sequences) {
            const long long offset = read_index<kPacked>(offsets, s), count = read_index<kPacked>(query_lengths, s);
            mine = offset >= 0 && count > 0 && offset < start + static_cast<long long>(queries) && offset + count > start;
        }
        any = any || __builtin_amdgcn_ballot_w64(mine) != 0;
    }
    return any;
}
// ... and whether one of them owns `token`.
SINGE_DEVICE bool later_sequence_owns(const void* offsets, const void* query_lengths, unsigned int sequences, unsigned int sequence, long long token) {
    bool owned = false;
    for (unsigned int s = sequence + 1; s < sequences; ++s) {
        const long long offset = read_index<kPacked>(offsets, s), count = read_index<kPacked>(query_lengths, s);
        owned = owned || (offset >= 0 && token >= offset && token < offset + count);
    }
    return owned;
}

// Workgroup units in sequence order: sequence s owns max(1, ceil(rows_s * heads / rows_per_unit)) of them (one even
// without rows, so that its paging values are checked), rows_s being its query count (from the offsets, or from
// `query_lengths` in the block-table form; counts that make no sense are held to [0, tokens] and their sequence's
// checks report them).  Every wave finds the owner of `unit` for itself by a prefix sum over the sequences, 64 at a
// time; false for a unit past the last sequence's.  A grid of tokens * heads / rows_per_unit + sequences units
// covers them all.
template <int FORM>
SINGE_DEVICE bool find_row_unit(const void* query_offsets, const void* query_lengths, unsigned int sequences, unsigned int tokens,
                                unsigned int heads, unsigned int rows_per_unit, unsigned int unit, unsigned int& sequence,
                                unsigned int& unit_of_sequence) {
    const unsigned int lane = threadIdx.x & 63u;
    unsigned int base = 0;
    for (unsigned int first = 0; first < sequences; first += 64u) {
        const unsigned int s = first + lane;
        unsigned int mine = 0;
        if (s < sequences) {
            long long count;
            if constexpr (has_lengths(FORM)) count = read_index<FORM>(query_lengths, s);
            else count = read_index<FORM>(query_offsets, s + 1) - read_index<FORM>(query_offsets, s);
            count = count < 0 ? 0 : count > static_cast<long long>(tokens) ? static_cast<long long>(tokens) : count;
            const unsigned long long units = (static_cast<unsigned long long>(count) * heads + rows_per_unit - 1) / rows_per_unit;
            mine = units == 0 ? 1u : static_cast<unsigned int>(units);
        }
        unsigned int through = mine;  // inclusive prefix sum over the wave
#pragma unroll
        for (int step = 1; step < 64; step <<= 1) {
            const unsigned int below = __shfl_up(through, step, 64);
            if (lane >= static_cast<unsigned int>(step)) through += below;
        }
        const unsigned int total = __shfl(through, 63, 64);
        if (unit < base + total) {
            const unsigned long long holds = __ballot(unit < base + through);  // first lane whose range reaches the unit
            const unsigned int owner = static_cast<unsigned int>(__builtin_ctzll(holds));
            const unsigned int owner_through = __shfl(through, owner, 64), owner_mine = __shfl(mine, owner, 64);
            sequence = first + owner;
            unit_of_sequence = unit - (base + owner_through - owner_mine);
            return true;
        }
        base += total;
    }
    return false;
}
