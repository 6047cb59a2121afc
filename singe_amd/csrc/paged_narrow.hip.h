// Row tiles of at most sixteen packed rows: a sequence that decodes (one token and the query heads of a kv head, or a few
// tokens of few) beside prompts in a mixed step, or in a step that the decode kernels do not take.
//
// The 128-row loop gives such a sequence one wave with sixteen live rows of 32 or fewer, three waves that only load, a
// barrier a tile and at most two tiles on their way.  What bounds the work is the cache rows' way from memory, so here:
//   * the four waves take turns at groups of sixteen keys and meet once, at the end (through LDS);
//   * a wave keeps its own ring of five LDS slots, sixteen rows of K or of V each, in the order K(0) V(0) K(1) V(1) ...,
//     and reloads a slot as soon as it has read it: four or five slots on their way at any time, 64 KiB and more a
//     workgroup and 128 KiB a compute unit, with no barrier and no wait but for the slot that is read next;
//   * S^T = K Q^T on v_mfma_f32_16x16x32 (the rows are the sixteen columns), O^T += V^T P^T on v_mfma_f32_16x16x16, whose
//     B operand is the score registers as they are: lane (row, g) holds keys 4 g .. 4 g + 3 of its row.
// A group's matrix and vector work is a tenth of the 32-row fold's, which leaves the matrix cores to the prompts' row tiles
// on the same compute unit.
//
// Kernel times, 64 / 8 heads x 128, bf16: 62 tokens over 2112 keys each 105 -> 89 us (6.0 TB/s; loads alone in this pattern
// 82 us), over 128 to 4096 keys 138 -> 107 us (the longest sequence's turns, 0.4 us each where nothing else runs), with two
// chunks of 512 tokens beside them 194 -> 130 us (the chunks alone 99 us).
#pragma once

#include "kernel_args.h"
#include "paging.hip.h"
#include "prefill_blocks.hip.h"
#include "row_alone.hip.h"

namespace {

using namespace prefill;

constexpr unsigned int kNarrowRows = 16, kNarrowKeys = 16;  // rows of a workgroup, keys of a group
constexpr unsigned int kNarrowSlots = 5;                    // of a wave's ring
constexpr unsigned int kNarrowSlotBytes = kNarrowKeys * kRowBytes;
constexpr unsigned int kNarrowWaveBytes = kNarrowSlots * kNarrowSlotBytes;
static_assert(4 * kNarrowWaveBytes <= kStagedLdsBytes, "the rings take the place of the tiles' stages");
// (behind a wave's sums in its ring's place, in floats: a row that is worked out by itself)
constexpr unsigned int kNarrowRowAt = kNarrowRows * (kHeadDim + 2);
static_assert((kNarrowRowAt + kHeadDim) * 4 <= kNarrowWaveBytes, "a wave's sums take the place of its ring");
// A score product takes 32 dims and needs all of them.
constexpr bool kNarrowBuild = kHeadDim % 32 == 0;

SINGE_DEVICE f32x4_t narrow_scores(Bf16, uint4 a, uint4 b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}
SINGE_DEVICE f32x4_t narrow_scores(F16, uint4 a, uint4 b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8v_t, a), __builtin_bit_cast(f16x8v_t, b), c, 0, 0, 0);
}
typedef _Float16 f16x4v_t __attribute__((ext_vector_type(4)));
SINGE_DEVICE f32x4_t narrow_values(Bf16, v4i16_t a, uint2 b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, __builtin_bit_cast(v4i16_t, b), c, 0, 0, 0);
}
SINGE_DEVICE f32x4_t narrow_values(F16, v4i16_t a, uint2 b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(f16x4v_t, a), __builtin_bit_cast(f16x4v_t, b), c, 0, 0, 0);
}

// The four loads of a slot, each lane's 16 bytes of load i from `base` + `offset[i]` to LDS at `dest` + 1024 i + 16 * lane.
// Non-temporal: a decoding sequence's rows are read once (the same pattern of loads alone reads 6.6 TB/s so, 5.8 without).
// As text, like load_16_to_lds (common.hip.h), the M0 that carries the LDS address stepped on from load to load.
SINGE_DEVICE void narrow_load(const unsigned char* base, const unsigned int (&offset)[4], const unsigned int (&chunk)[4], unsigned int dest) {
    if constexpr (kGlobalRowBytes != kRowBytes) {
        // Lanes whose place holds no chunk of a shorter row fetch nothing (some lane of every instruction does: each counts).
        // (Not non-temporal: a row shares its lines or its 256 bytes of memory with the next kv head's; head_dim 64 and 96 of
        // the mixed step 94 and 134 us, 99 and 145 non-temporal.)
#pragma unroll
        for (unsigned int i = 0; i < 4; ++i) {
            if (chunk[i] < kGlobalRowBytes)
                load_16_to_lds(base, offset[i], dest + i * 4u * kRowBytes);
        }
        return;
    }
    const unsigned int first = __builtin_amdgcn_readfirstlane(dest);
    const unsigned long long bits = reinterpret_cast<unsigned long long>(base);
    const unsigned int low_word = __builtin_amdgcn_readfirstlane(static_cast<unsigned int>(bits));
    const unsigned int high_word = __builtin_amdgcn_readfirstlane(static_cast<unsigned int>(bits >> 32));
    const unsigned long long scalar = static_cast<unsigned long long>(low_word) | (static_cast<unsigned long long>(high_word) << 32);
    unsigned int kept;
    asm volatile(
        "s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %3, %2 nt\n\t"
        "s_add_u32 m0, m0, 0x400\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %4, %2 nt\n\t"
        "s_add_u32 m0, m0, 0x400\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %5, %2 nt\n\t"
        "s_add_u32 m0, m0, 0x400\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %6, %2 nt\n\ts_mov_b32 m0, %0"
        : "=&s"(kept)
        : "s"(first), "s"(scalar), "v"(offset[0]), "v"(offset[1]), "v"(offset[2]), "v"(offset[3])
        : "memory", "scc");
}

// Until at most `count` items of four loads each are still on their way; what the compiler reads from LDS stays behind it.
SINGE_DEVICE void narrow_wait(unsigned int count) {
    if (count >= 4) asm volatile("s_waitcnt vmcnt(16)" ::: "memory");
    else if (count == 3) asm volatile("s_waitcnt vmcnt(12)" ::: "memory");
    else if (count == 2) asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
    else if (count == 1) asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}
// Until the LDS reads in front of it are done, so that their slot may be loaded into.
SINGE_DEVICE void narrow_slot_read() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// A row of a (sequence, kv head) over its pages, for row_alone; its output goes to LDS.
template <int FORM, class Half>
struct PagedRow {
    const uint16_t* query_row;
    const PagedAttentionArgs& a;
    size_t page_start;
    unsigned int head_at;  // of the kv head in a key's row
    float* out_row;
    SINGE_DEVICE size_t place(unsigned int k) const {
        const unsigned long long id = read_page<FORM>(a.pages, page_start + (k >> a.page_shift));
        const size_t page = id < static_cast<unsigned long long>(a.cache_pages) ? static_cast<size_t>(id) : 0;  // (reported by who looked it up first)
        return (page * a.page_size + (k & (a.page_size - 1u))) * a.kv_heads * kHeadDim + head_at;
    }
    SINGE_DEVICE float query(unsigned int d) const { return widen(Half{}, query_row[d]); }
    SINGE_DEVICE float key(size_t at, unsigned int d) const { return widen(Half{}, a.key_cache[at + d]); }
    SINGE_DEVICE float value(size_t at, unsigned int d) const { return widen(Half{}, a.value_cache[at + d]); }
    SINGE_DEVICE void store(unsigned int d, float value) const { out_row[d] = value; }
};

// The `packed` packed rows of one (sequence, kv head) from `first_row` on, keys [key_begin, key_end) of the sequence (multiples
// of sixteen, but for the end), of which a row sees what its position and the window leave it.  Pages of at least sixteen keys,
// a power of two of them.  finish(row, quad, values, lse2) takes values 4 quad .. of a row, normalised, and its base-two
// log-sum-exp (a row that sees no key: zeros and -inf).  WIDE: the weights meet the values at f32's precision (split_pair), by a
// second value product that the memory-bound loop has room for.  An infinity among the values is a NaN to that product, so
// values that come out not finite are worked out again there, from the keys the row sees and no others (row_alone); and a row
// with a score that is NaN or +inf has a log-sum-exp of NaN beside its values, so that whoever merges it with others can tell it
// from a row that sees no key.
template <bool SOFTCAP, int FORM, bool WIDE, unsigned int WAVES, class Half, class Finish>
SINGE_DEVICE void narrow_rows(const PagedAttentionArgs& a, unsigned char* lds, const SequenceSpan& span, unsigned int kv_head, unsigned int first_row,
                              unsigned int packed, unsigned int key_begin, unsigned int key_end, Finish&& finish) {
    const unsigned int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63u;
    const unsigned int column = lane & 15u, g = lane >> 4;
    const unsigned int groups = a.heads / a.kv_heads;
    const unsigned int queries = span.queries, keys = span.keys;
    const bool causal = a.causal != 0, windowed = a.window >= 0;
    const unsigned int window = !windowed ? 0u : a.window > 0x7fffffffll ? 0x7fffffffu : static_cast<unsigned int>(a.window);
    const Half half{};
    auto position_of = [&](unsigned int row) __attribute__((always_inline)) {
        const long long position = static_cast<long long>(keys) - static_cast<long long>(queries) + (first_row + row) / groups;
        return position < 0 ? 0u : static_cast<unsigned int>(position);
    };
    const bool row_valid = column < packed;
    const unsigned int my_row = row_valid ? column : 0u, my_position = position_of(my_row);
    const unsigned int low_position = position_of(0), high_position = position_of(packed - 1u);

    // Q^T: lane (row, g) holds dims 32 s + 8 g .. + 8; a negative scale moves into it.
    constexpr int kNarrowSteps = (kHeadDim + 31) / 32, kNarrowBlocks = kHeadDim / 16;
    const float factor = SOFTCAP ? 1.0f : fabsf(a.scale_log2e);
    const unsigned int flip = (SOFTCAP ? a.softcap_scale : a.scale_log2e) < 0.0f ? 0x80008000u : 0u;
    uint4 q[kNarrowSteps];
    {
        const unsigned int at = first_row + my_row;
        const size_t flat = (static_cast<size_t>(span.query_start) + at / groups) * a.heads + kv_head * groups + at % groups;
        const uint16_t* row = a.query_rows + flat * kHeadDim + 8u * g;
#pragma unroll
        for (int s = 0; s < kNarrowSteps; ++s) {
            uint4 bits = *reinterpret_cast<const uint4*>(row + 32 * s);
            if (!row_valid) bits = make_uint4(0, 0, 0, 0);
            bits.x ^= flip; bits.y ^= flip; bits.z ^= flip; bits.w ^= flip;
            q[s] = bits;
        }
    }

    // A slot is filled by four instructions, four rows each: lane l of instruction i brings what belongs at chunk place
    // l % 16 of row 4 i + l / 16 (K keeps chunk c of a row at c ^ row, V at c ^ 4 (row & 3)).
    const unsigned int load_row = lane >> 4, place = lane & 15u;
    const unsigned int head_bytes = kv_head * kGlobalRowBytes, slot_bytes = a.kv_heads * kGlobalRowBytes;
    unsigned int key_chunk_of[4], value_chunk_of[4], key_offset[4], value_offset[4];  // of instruction i: the lane's chunk, and its place behind the group's first row
#pragma unroll
    for (unsigned int i = 0; i < 4; ++i) {
        key_chunk_of[i] = 16u * (place ^ (4u * i + load_row));
        value_chunk_of[i] = 16u * (place ^ (4u * load_row));
        key_offset[i] = (4u * i + load_row) * slot_bytes + key_chunk_of[i];
        value_offset[i] = (4u * i + load_row) * slot_bytes + value_chunk_of[i];
    }
    const unsigned int lds_start = static_cast<unsigned int>(reinterpret_cast<__UINTPTR_TYPE__>((lds_words_t)lds)) + wave * kNarrowWaveBytes;
    unsigned char* const ring = lds + wave * kNarrowWaveBytes;

    // The wave's groups: key_begin / 16 + wave, and every WAVES-th one from there.
    const unsigned int first_group = key_begin / kNarrowKeys + wave, end_group = (key_end + kNarrowKeys - 1u) / kNarrowKeys;
    const unsigned int count = __builtin_amdgcn_readfirstlane(first_group < end_group ? (end_group - first_group + WAVES - 1u) / WAVES : 0u);
    auto key_of = [&](unsigned int t) __attribute__((always_inline)) { return (first_group + WAVES * t) * kNarrowKeys; };
    // Page ids come 64 groups at a time, lane l that of group `first` + l, by a vector load: a scalar load would share its
    // counter with the LDS reads, which would then wait for it in every group.  An id outside the cache is reported and
    // replaced by page 0.
    auto look_up = [&](unsigned int first) __attribute__((always_inline)) {
        unsigned int id = 0;
        if (first + lane < count) {
            const unsigned long long page = read_page<FORM>(a.pages, static_cast<size_t>(span.page_start) + (key_of(first + lane) >> a.page_shift));
            if (page < static_cast<unsigned long long>(a.cache_pages)) id = static_cast<unsigned int>(page);
            else report_index_error(a.status);
        }
        return id;
    };
    auto bring = [&](auto is_value, unsigned int t, unsigned int page, unsigned int slot) __attribute__((always_inline)) {
        constexpr bool kValue = decltype(is_value)::value;
        const unsigned int key0 = key_of(t);
        const unsigned char* base = reinterpret_cast<const unsigned char*>(kValue ? a.value_cache : a.key_cache) +
                                    (static_cast<size_t>(page) * a.page_size + (key0 & (a.page_size - 1u))) * slot_bytes + head_bytes;
        const unsigned int dest = lds_start + slot * kNarrowSlotBytes;
        if (key0 + kNarrowKeys <= keys) {
            narrow_load(base, kValue ? value_offset : key_offset, kValue ? value_chunk_of : key_chunk_of, dest);
        } else {
            // (kept a branch: as selects its arithmetic would be every group's)
            asm volatile("s_nop 0");
            const unsigned int last = keys - 1u - key0;  // rows past the last key re-read it and are masked
            unsigned int offset[4];
#pragma unroll
            for (unsigned int i = 0; i < 4; ++i) {
                const unsigned int row = 4u * i + load_row;
                offset[i] = (row < last ? row : last) * slot_bytes + (kValue ? value_chunk_of[i] : key_chunk_of[i]);
            }
            narrow_load(base, offset, kValue ? value_chunk_of : key_chunk_of, dest);
        }
    };

    f32x4_t out[kNarrowBlocks];  // lane (row, g): dims 16 db + 4 g + r
#pragma unroll
    for (int db = 0; db < kNarrowBlocks; ++db) out[db] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    float reference = -INFINITY, running_sum = 0.0f;  // (the sum of this lane's keys)

    // Read places: K row `column`, chunk 4 s + g; V^T keys 4 g + column / 4, chunk 2 db + (column & 3) / 2, half by column & 1.
    const unsigned int key_at = column * kRowBytes;
    const unsigned int value_at = (4u * g + (column >> 2)) * kRowBytes + 8u * (column & 1u), value_flip = 4u * (column >> 2) ^ ((column & 3u) >> 1);

    if (count > 0) {
        // K(0) V(0) K(1) V(1) K(2) go out; `page` is that of the last group whose K did.
        unsigned int ids = look_up(0), page = __builtin_amdgcn_readlane(ids, 0);
        bring(std::false_type{}, 0u, page, 0u);
        bring(std::true_type{}, 0u, page, 1u);
        if (count > 1) {
            page = __builtin_amdgcn_readlane(ids, 1);
            bring(std::false_type{}, 1u, page, 2u);
            bring(std::true_type{}, 1u, page, 3u);
        }
        if (count > 2) {
            page = __builtin_amdgcn_readlane(ids, 2);
            bring(std::false_type{}, 2u, page, 4u);
        }
        unsigned int read_slot = 0;
        for (unsigned int t = 0; t < count; ++t) {
            const unsigned int key0 = key_of(t);
            // What comes after K(t), and then after V(t): at most four items are on their way by then.
            const unsigned int behind = 2u * (count - t) - 1u;
            narrow_wait(behind);
            const unsigned int key_slot = read_slot;
            const unsigned char* keys_at = ring + key_slot * kNarrowSlotBytes;
            read_slot = read_slot + 1u == kNarrowSlots ? 0u : read_slot + 1u;
            uint4 operand[kNarrowSteps];
#pragma unroll
            for (int s = 0; s < kNarrowSteps; ++s) operand[s] = *reinterpret_cast<const uint4*>(keys_at + key_at + 16u * ((4u * s + g) ^ column));
            __builtin_amdgcn_sched_barrier(0);  // (all reads before the first product, or each would be waited for by itself)
            f32x4_t scores = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int s = 0; s < kNarrowSteps; ++s) scores = narrow_scores(half, operand[s], q[s], scores);
            narrow_slot_read();
            if (t + 2u < count) bring(std::true_type{}, t + 2u, page, key_slot);
            // V(t)'s operands on their way while the scores become weights.
            narrow_wait(behind - 1u);
            const unsigned int value_slot = read_slot;
            const unsigned char* values_at = ring + value_slot * kNarrowSlotBytes;
            read_slot = read_slot + 1u == kNarrowSlots ? 0u : read_slot + 1u;
            typedef v4i16_t __attribute__((address_space(3))) * lds_v4_t;
            v4i16_t value[kNarrowBlocks];
#pragma unroll
            for (int db = 0; db < kNarrowBlocks; ++db)
                value[db] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4_t)(values_at + value_at + 16u * ((2u * db) ^ value_flip)));
            __builtin_amdgcn_sched_barrier(0);
            float x[4] = {scores[0], scores[1], scores[2], scores[3]};
            if constexpr (SOFTCAP) {
                const float cap_scale = fabsf(a.softcap_scale);
#pragma unroll
                for (int r = 0; r < 4; ++r) x[r] = fast_tanh(x[r] * cap_scale) * a.softcap_log2e;
            }
            if (key0 + kNarrowKeys > keys || (causal && key0 + kNarrowKeys - 1u > low_position) || (windowed && key0 + window <= high_position)) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const unsigned int key = key0 + 4u * g + r;
                    if (key >= keys || (causal && key > my_position) || (windowed && key + window <= my_position)) x[r] = -INFINITY;
                }
            }
            const float largest = across_groups_max(fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3]))) * factor;  // (not max2: nothing would wait for the products)
            if (__any(largest > reference + kMaxLag || (reference == -INFINITY && largest != -INFINITY))) {
                const float moved = fmaxf(reference, largest), base = moved == -INFINITY ? 0.0f : moved;
                const float rescale = fast_exp2(reference - base);
                running_sum *= rescale;
#pragma unroll
                for (int db = 0; db < kNarrowBlocks; ++db)
#pragma unroll
                    for (int r = 0; r < 4; ++r) out[db][r] *= rescale;
                reference = moved;
            }
            const float shift = reference == -INFINITY ? 0.0f : -reference;
            float p[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                p[r] = fast_exp2(fmaf(x[r], factor, shift));
                running_sum += p[r];
            }
            uint2 weights, rest;
            if constexpr (WIDE) {
                split_pair(half, p[0], p[1], weights.x, rest.x);
                split_pair(half, p[2], p[3], weights.y, rest.y);
            } else {
                weights = make_uint2(pack_pair(half, p[0], p[1]), pack_pair(half, p[2], p[3]));
            }
#pragma unroll
            for (int db = 0; db < kNarrowBlocks; ++db) out[db] = narrow_values(half, value[db], weights, out[db]);
            if constexpr (WIDE) {
#pragma unroll
                for (int db = 0; db < kNarrowBlocks; ++db) out[db] = narrow_values(half, value[db], rest, out[db]);
            }
            narrow_slot_read();
            if (t + 3u < count) {
                if (((t + 3u) & 63u) == 0) ids = look_up(t + 3u);
                page = __builtin_amdgcn_readlane(ids, (t + 3u) & 63u);
                bring(std::false_type{}, t + 3u, page, value_slot);
            }
        }
    }

    // The waves' sums meet in LDS, each in the place of the wave's ring, which nobody else reads or loads into.
    const float sum = across_groups_sum(running_sum);
    float* mine = reinterpret_cast<float*>(ring);
#pragma unroll
    for (int db = 0; db < kNarrowBlocks; ++db)
        *reinterpret_cast<float4*>(mine + column * kHeadDim + 16 * db + 4 * g) = make_float4(out[db][0], out[db][1], out[db][2], out[db][3]);
    if (g == 0) {
        mine[kNarrowRows * kHeadDim + 2u * column] = reference;
        mine[kNarrowRows * kHeadDim + 2u * column + 1u] = sum;
    }
    __syncthreads();
    const unsigned int items = packed * (kHeadDim / 4u);
    for (unsigned int first = 64u * wave; first < items; first += 64u * WAVES) {  // (with all of a wave's lanes)
        const unsigned int item = first + lane, at = item < items ? item : items - 1u, row = at / (kHeadDim / 4u), quad = at % (kHeadDim / 4u);
        float references[WAVES], sums[WAVES], largest = -INFINITY;
#pragma unroll
        for (unsigned int w = 0; w < WAVES; ++w) {
            const float* from = reinterpret_cast<const float*>(lds + w * kNarrowWaveBytes) + kNarrowRows * kHeadDim + 2u * row;
            references[w] = from[0];
            sums[w] = from[1];
            largest = fmaxf(largest, references[w]);
        }
        float4 merged = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        float total = 0.0f;
#pragma unroll
        for (unsigned int w = 0; w < WAVES; ++w) {
            const float weight = references[w] == -INFINITY ? 0.0f : fast_exp2(references[w] - largest);
            const float4 part = *reinterpret_cast<const float4*>(reinterpret_cast<const float*>(lds + w * kNarrowWaveBytes) + row * kHeadDim + 4u * quad);
            total = fmaf(weight, sums[w], total);
            merged.x = fmaf(weight, part.x, merged.x);
            merged.y = fmaf(weight, part.y, merged.y);
            merged.z = fmaf(weight, part.z, merged.z);
            merged.w = fmaf(weight, part.w, merged.w);
        }
        const float inverse = (total > 0.0f ? 1.0f / total : 0.0f) * (WIDE ? 1.0f / kWideScale<Half> : 1.0f);
        merged.x *= inverse; merged.y *= inverse; merged.z *= inverse; merged.w *= inverse;
        float lse2 = total > 0.0f ? largest + fast_log2(total) : -INFINITY;
        if constexpr (WIDE) {
            static_assert(!SOFTCAP, "row_alone takes the scores as they are");
            if (total != total) lse2 = total;  // (and so are all of the row's values)
            const float values[4] = {merged.x, merged.y, merged.z, merged.w};
            const bool bad = total == total && not_finite(4, [&](int i) { return values[i]; });
            for (unsigned long long left = __builtin_amdgcn_ballot_w64(bad); left != 0;) {
                const unsigned int r = __builtin_amdgcn_readlane(row, __builtin_ctzll(left)), packed_row = first_row + r, position = position_of(r);
                const size_t flat = (static_cast<size_t>(span.query_start) + packed_row / groups) * a.heads + kv_head * groups + packed_row % groups;
                const unsigned int seen = windowed && position >= window ? position - window + 1u : 0u, reach = causal && position < key_end ? position + 1u : key_end;
                float* const apart = mine + kNarrowRowAt;
                row_alone<kHeadDim>(PagedRow<FORM, Half>{a.query_rows + flat * kHeadDim, a, static_cast<size_t>(span.page_start), kv_head * kHeadDim, apart},
                                    key_begin > seen ? key_begin : seen, reach, a.scale_log2e);
                narrow_slot_read();  // (and written: a lane's values are other lanes' stores)
                if (bad && row == r) merged = *reinterpret_cast<const float4*>(apart + 4u * quad);
                narrow_slot_read();
                left &= ~__builtin_amdgcn_ballot_w64(row == r);
            }
        }
        if (item < items) finish(row, quad, merged, lse2);
    }
}

}  // namespace
