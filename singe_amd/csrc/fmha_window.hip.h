// Dense causal attention under a short window over grouped heads (bf16 / f16): a workgroup of eight waves walks along a
// run of a (batch, kv head) pair's rows, with the keys and values its windows reach kept in LDS.
//
// Rows are (query, head of the group) pairs, row r being query r / group of head kv_head * group + r % group, and a step is
// 256 of them, 32 a wave: 256 / group queries, whose windows overlap almost whole.  Keys live in LDS in blocks of 32, block b
// (keys 32 b .. 32 b + 31) in place b % ring_blocks; a step's blocks are there when it starts, and those that the next step
// needs besides, 256 / group keys of them, are loaded beneath it into places that this step does not read.  So a key is
// fetched once for a run of rows, a wave folds exactly the blocks its own 32 rows see, without a barrier between them, and
// the queries' and keys' round trips to memory are spent beneath the step before.
//
// The layouts of blocks and registers and the functions that fold a block are those of prefill_blocks.hip.h.
//
// What bounds it is the queries' way in and the outputs' way out (64 / 8 heads x 8192 x 64, bf16: 151 MB, 31 us at the 4.8 TB/s
// of a copy) with the folding beside them: window 16 31 us, 128 41 us, 256 55 us, where tiles of 128 rows in workgroups of their
// own, each with round trips of its own at either end and a barrier to 64 keys, take 48, 58 and 70 us; at head_dim 128 62, 75
// and 98 us against 96, 125 and 151.  (One call's buffers over and over; many calls in turn over 600 MB: 40, 51 and 65 us
// against 50, 62 and 74; window 128 at head_dim 128 95 against 121.)  The outputs leave as 64 contiguous bytes a row, past the
// caches (see store_row_16): as 32 bytes a row and through them they cost 11 us more at head_dim 128; 32 bytes a row past the
// caches 11 us more at head_dim 64 too.  The queries come through the caches (past them +8 us at 64, +30 us at 128), 64 bytes a
// row at a time or 32 alike.  Up to head_dim 64 a compute unit holds two workgroups of at most 128 registers, which is why lane
// offsets are worked out again from step to step.
#pragma once

#include "prefill_blocks.hip.h"

namespace prefill {

constexpr unsigned int kWindowStepRows = 32u * kWindowPrefillWaves;

// Rows of whole 64-byte pieces leave past the caches; the others end inside pieces, which past them go out in parts.  Past /
// through the caches (tiles of 128 rows), us, many calls in turn over 600 MB:
//   28 / 4 heads x 112, 4 x 9401, window 16  219 / 120 (153)   40 / 8 x 80, 4 x 3764, 20  92 / 56 (78)   64 / 8 x 48, 4 x 2325, 16  49 / 33 (46)
SINGE_DEVICE void store_row_16(unsigned char* address, uint4 bits) {
    if constexpr (kHeadDim % 32 == 0) stream_store_16(address, bits);
    else *reinterpret_cast<uint4*>(address) = bits;
}

template <class Half>
SINGE_DEVICE void fmha_window_body(const PrefillArgs& a, unsigned char* lds) {
    constexpr unsigned int kWaveLoadRows = 1024u / kRowBytes;  // key rows one load instruction of a wave brings in
    static_assert(kWindowPrefillWaves == 8, "a block's rows are dealt out to eight waves");
    const unsigned int tid = threadIdx.x, lane = tid & 63u, hi = lane >> 5;
    const unsigned int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const unsigned int group = a.heads / a.kv_heads, pairs = a.batch * a.kv_heads;

    // Workgroup i runs on XCD i % 8: neighbouring runs of rows, whose first and last windows overlap, go to one XCD.
    const unsigned int runs = a.query_tiles, units = pairs * runs, per_xcd = (units + 7u) / 8u;
    const unsigned int unit = (blockIdx.x & 7u) * per_xcd + (blockIdx.x >> 3);
    if ((blockIdx.x >> 3) >= per_xcd || unit >= units) return;
    const unsigned int pair = unit / runs, batch = pair / a.kv_heads, kv_head = pair - batch * a.kv_heads;
    const unsigned int steps = (a.query_len * group + kWindowStepRows - 1u) / kWindowStepRows;
    const unsigned int first_step = (unit - pair * runs) * a.run_steps;
    const unsigned int end_step = steps < first_step + a.run_steps ? steps : first_step + a.run_steps;
    if (first_step >= end_step) return;

    unsigned int key_len = a.key_len;
    if (a.key_lengths != nullptr) {
        const int own = a.key_lengths[batch];
        const unsigned int bound = own > 0 ? static_cast<unsigned int>(own) : 0u;
        key_len = bound < key_len ? bound : key_len;
    }
    key_len = __builtin_amdgcn_readfirstlane(key_len);
    const unsigned int window = static_cast<unsigned int>(a.window);
    auto low = [&](unsigned int query) __attribute__((always_inline)) { return query >= window ? query - window + 1u : 0u; };  // key + window <= query is hidden

    // The blocks the rows of a step see: [first, end).
    auto step_blocks = [&](unsigned int step, unsigned int& first, unsigned int& end) __attribute__((always_inline)) {
        const unsigned int first_query = step * kWindowStepRows / group, last = (step * kWindowStepRows + kWindowStepRows - 1u) / group;
        const unsigned int last_query = last < a.query_len ? last : a.query_len - 1u;
        const unsigned int key_begin = low(first_query), key_end = last_query + 1u < key_len ? last_query + 1u : key_len;
        first = key_begin / 32u;
        end = key_begin < key_end ? (key_end + 31u) / 32u : first;
    };

    // A block's load is 1 KiB an instruction, lane l the chunk position l % 16 of row l / 16 of it (l % 8 of row l / 8 in
    // 128-byte rows, where waves 0 to 3 bring the keys and 4 to 7 the values; otherwise each wave four rows of both).
    // Offsets inside one (batch, kv head) slice fit 32 bits (checked by the host).
    const unsigned char* const k_bytes = reinterpret_cast<const unsigned char*>(a.key + batch * a.key_batch_stride + kv_head * a.key_head_stride);
    const unsigned char* const v_bytes = reinterpret_cast<const unsigned char*>(a.value + batch * a.value_batch_stride + kv_head * a.value_head_stride);
    const unsigned int key_stride = static_cast<unsigned int>(a.key_sequence_stride) * 2u, value_stride = static_cast<unsigned int>(a.value_sequence_stride) * 2u;
    const unsigned int ring = a.ring_blocks, values_at = ring * static_cast<unsigned int>(kBlockBytes);
    const unsigned int lds_at = static_cast<unsigned int>(reinterpret_cast<__UINTPTR_TYPE__>((lds_words_t)lds));
    const unsigned int part = kRowBytes == 128 ? wave & 3u : wave;
    auto load_block = [&](unsigned int block, unsigned int place) __attribute__((always_inline)) {
        unsigned int own = tid;
        asm volatile("" : "+v"(own));  // (worked out again for every block: held, these registers are ones the folding spills)
        const unsigned int load_row = kWaveLoadRows * part + (own & 63u) / kRowChunks, position = own % kRowChunks;
        unsigned int row = load_row;  // (rows past the last key re-read it, and are masked)
        if (32u * block + 32u > key_len) row = 32u * block + row < key_len ? row : key_len - 1u - 32u * block;
        const unsigned int dest = lds_at + place * static_cast<unsigned int>(kBlockBytes) + part * 1024u;
        // (a global row narrower than an LDS row has fewer chunks: the lanes whose position holds one past its end fetch nothing)
        auto load = [&](const unsigned char* rows, unsigned int stride, unsigned int chunk, unsigned int to) __attribute__((always_inline)) {
            if (kGlobalRowBytes == kRowBytes || chunk < static_cast<unsigned int>(kGlobalRowBytes))
                load_16_to_lds(rows + static_cast<size_t>(32u * block) * stride, row * stride + chunk, to);
        };
        if (kRowBytes != 128 || wave < 4u) load(k_bytes, key_stride, (position ^ key_chunk_flip(load_row)) * 16u, dest);
        if (kRowBytes != 128 || wave >= 4u) load(v_bytes, value_stride, (position ^ value_chunk_flip(load_row)) * 16u, dest + values_at);
    };

    const float factor = fabsf(a.scale_log2e);
    const unsigned int flip = a.scale_log2e < 0.0f ? 0x80008000u : 0u;
    const Half half{};
    // (a batch entry's queries and its output rows lie within 32 bits of their first one, checked by the host)
    const unsigned char* const q_bytes = reinterpret_cast<const unsigned char*>(a.query + batch * a.query_batch_stride);
    unsigned char* const out_bytes = reinterpret_cast<unsigned char*>(a.out + batch * a.output_batch_stride);
    const unsigned int query_stride = static_cast<unsigned int>(a.query_sequence_stride) * 2u, query_head_stride = static_cast<unsigned int>(a.query_head_stride) * 2u;
    const unsigned int out_stride = static_cast<unsigned int>(a.output_sequence_stride) * 2u, out_head_stride = static_cast<unsigned int>(a.output_head_stride) * 2u;
    uint4 q[kSteps];
    uint16_t sink_bits = 0;
    // The rows of a wave in a step, and its queries on their way to the registers that hold them (a row past the last one
    // takes the last one's place and is not stored).
    auto row_query = [&](unsigned int step, unsigned int& query, unsigned int& head) __attribute__((always_inline)) {
        unsigned int own = tid;
        asm volatile("" : "+v"(own));
        const unsigned int row = step * kWindowStepRows + wave * 32u + (own & 31u);
        query = row / group;
        head = kv_head * group + (row - query * group);
    };
    auto load_queries = [&](unsigned int step) __attribute__((always_inline)) {
        unsigned int query, head;
        row_query(step, query, head);
        query = query < a.query_len ? query : a.query_len - 1u;
        const unsigned int at = query * query_stride + head * query_head_stride + 16u * hi;
#pragma unroll
        for (int s = 0; s < kSteps; ++s) q[s] = *reinterpret_cast<const uint4*>(q_bytes + at + 32 * s);
        sink_bits = *(a.sinks != nullptr ? a.sinks + head : a.query);  // (some word without one)
    };

    unsigned int first_block, end_block;
    step_blocks(first_step, first_block, end_block);
    unsigned int first_place = first_block % ring;  // of the step's first block
    {
        unsigned int place = first_place;
        for (unsigned int block = first_block; block < end_block; ++block) {
            load_block(block, place);
            place = place + 1u == ring ? 0u : place + 1u;
        }
    }
    load_queries(first_step);
    loads_landed();
    __syncthreads();

    const ReadOffsets offsets = read_offsets(lane);
    for (unsigned int step = first_step; step < end_step; ++step) {
        const bool more = step + 1u < end_step;
        unsigned int next_first = first_block, next_end = end_block;
        if (more) {
            step_blocks(step + 1u, next_first, next_end);
            unsigned int block = next_first > end_block ? next_first : end_block;
            for (; block < next_end; ++block) load_block(block, block % ring);
        }
        unsigned int my_query, head;
        row_query(step, my_query, head);
        const unsigned int wave_query = __builtin_amdgcn_readfirstlane(my_query);
        if (wave_query < a.query_len) {
            const unsigned int last = __builtin_amdgcn_readlane(my_query, 31), wave_last_query = last < a.query_len ? last : a.query_len - 1u;
            const unsigned int my_low = low(my_query), last_low = low(wave_last_query);
            const unsigned int my_end = my_query + 1u < key_len ? my_query + 1u : key_len, my_span = my_end > my_low ? my_end - my_low : 0u;
            const unsigned int wave_begin = low(wave_query), wave_end = wave_last_query + 1u < key_len ? wave_last_query + 1u : key_len;
            unsigned int block = wave_begin / 32u;
            const unsigned int blocks_end = wave_begin < wave_end ? (wave_end + 31u) / 32u : block;
            unsigned int place = first_place + (block - first_block);
            place = place >= ring ? place - ring : place;

#pragma unroll
            for (int s = 0; s < kSteps; ++s) { q[s].x ^= flip; q[s].y ^= flip; q[s].z ^= flip; q[s].w ^= flip; }
            RowState state;
            reset(state);
            if (a.sinks != nullptr) {
                // The head's sink: a score that is always there and weighs no value.  The row starts with it as its reference
                // point and a sum of one (held by one of the row's two lanes).
                float sink;
                if constexpr (std::is_same_v<Half, F16>) sink = static_cast<float>(__builtin_bit_cast(_Float16, sink_bits));
                else sink = __builtin_bit_cast(float, static_cast<unsigned int>(sink_bits) << 16);
                state.reference = sink * kLog2e;
                state.running_sum = hi == 0 && state.reference != -INFINITY ? 1.0f : 0.0f;
            }
            // Only the blocks that the window's or the causal mask's edge crosses for some row of the wave look at their keys.
            auto begin = [&](unsigned int b, f32x16_t& s) __attribute__((always_inline)) {
                const unsigned int key0 = 32u * b;
                if (key0 + 31u > wave_query || key0 + 32u > key_len || key0 < last_low) {
                    asm volatile("");  // (kept a branch: the compiler turns short ones into selects on every block)
                    const unsigned int from = key0 + 4u * hi - my_low;
#pragma unroll
                    for (int r = 0; r < 16; ++r)
                        if (from + (8u * (r >> 2) + (r & 3)) >= my_span) s[r] = -INFINITY;
                }
                return begin_block(state, s, hi, factor, false, [](unsigned int) { return false; });
            };
            f32x16_t scores;
            if (block < blocks_end) {
                score_block(half, scores, q, lds + place * kBlockBytes, offsets);
                for (; block + 1u < blocks_end; ++block) {
                    const unsigned int next = place + 1u == ring ? 0u : place + 1u;
                    const float shift = begin(block, scores);
                    finish_block<true>(half, state, scores, factor, shift, lds + values_at + place * kBlockBytes, offsets, scores, q, lds + next * kBlockBytes);
                    __builtin_amdgcn_sched_barrier(0);
                    place = next;
                }
                const float shift = begin(block, scores);
                if (more) load_queries(step + 1u);
                finish_block<false>(half, state, scores, factor, shift, lds + values_at + place * kBlockBytes, offsets, scores, q, lds);
            } else if (more) {
                load_queries(step + 1u);
            }
            // Normalise and store.  Lane (query, hi) holds dims 32db + 8(r / 4) + 4hi + (r % 4); its partner in the other half
            // of the wave holds the four dims beside each of its fours, and a swap leaves either with eight neighbours.
            // (The waits for this step's loads come before its stores, whose own way to memory is the next step's.)
            const float sum = swap32_sum(state.running_sum);
            const float inverse = sum > 0.0f ? 1.0f / sum : 0.0f;
            uint4 packed[kHeadDim / 16];
#pragma unroll
            for (int pair_of = 0; pair_of < kHeadDim / 16; ++pair_of) {
                const int db = pair_of / 2, at = 8 * (pair_of % 2);
                auto two = [&](int r) __attribute__((always_inline)) { return pack_pair(half, state.out[db][at + r] * inverse, state.out[db][at + r + 1] * inverse); };
                unsigned int lower[2] = {two(0), two(2)}, upper[2] = {two(4), two(6)};
                asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %2\n\tv_permlane32_swap_b32 %1, %3"
                             : "+v"(lower[0]), "+v"(lower[1]), "+v"(upper[0]), "+v"(upper[1]));
                packed[pair_of] = make_uint4(lower[0], lower[1], upper[0], upper[1]);
            }
            // Two pieces of a row and of the row sixteen below it change places likewise where there are pairs of pieces, so that a
            // store writes sixteen rows, 64 bytes of each, in place of thirty-two rows' 32 bytes.
            constexpr int kPieces = kHeadDim / 16;
            row_query(step, my_query, head);
            const unsigned int mine = my_query < a.query_len ? my_query * out_stride + head * out_head_stride : ~0u;
            unsigned int at = mine, other = mine;
            asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(at), "+v"(other));
#pragma unroll
            for (int p = 0; p + 1 < kPieces; p += 2)
                asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %4\n\tv_permlane16_swap_b32 %1, %5\n\t"
                             "v_permlane16_swap_b32 %2, %6\n\tv_permlane16_swap_b32 %3, %7"
                             : "+v"(packed[p].x), "+v"(packed[p].y), "+v"(packed[p].z), "+v"(packed[p].w),
                               "+v"(packed[p + 1].x), "+v"(packed[p + 1].y), "+v"(packed[p + 1].z), "+v"(packed[p + 1].w));
            loads_landed();
            unsigned char* const to = out_bytes + 16u * hi;
#pragma unroll
            for (int p = 0; p + 1 < kPieces; p += 2) {
                if (at != ~0u) store_row_16(to + 2u * (lane & 16u) + at + 32 * p, packed[p]);
                if (other != ~0u) store_row_16(to + 2u * (lane & 16u) + other + 32 * p, packed[p + 1]);
            }
            if (kPieces % 2 != 0 && mine != ~0u) *reinterpret_cast<uint4*>(to + mine + 32 * (kPieces - 1)) = packed[kPieces - 1];
            if (my_query < a.query_len) {
                if (a.lse != nullptr && hi == 0)
                    a.lse[(static_cast<size_t>(batch) * a.heads + head) * a.query_len + my_query] =
                        sum > 0.0f ? (state.reference + fast_log2(sum)) * kLn2 : -INFINITY;
            }
        } else {
            loads_landed();
        }
        if (!more) break;
        __syncthreads();  // everyone has read this step's blocks, and the next step's have landed
        first_place += next_first - first_block;
        first_place = first_place >= ring ? first_place % ring : first_place;
        first_block = next_first;
        end_block = next_end > end_block ? next_end : end_block;
    }
}

}  // namespace prefill
