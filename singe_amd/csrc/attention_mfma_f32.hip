// Dense f32 attention on the matrix cores (fmha_prefill_f32, fmha_prefill_lse_f32, softcapped_window_attention_f32 without a
// cap, singe-kernel/src/cuda/attention/fmha.rs:48-290, CPU forms cpu/attention.rs:1758-1925; and the singe crate's
// scaled_dot_product_attention of f32 tensors with a causal mask, a window or key lengths,
// singe/src/backend/cpu/normalization/attention.rs:191-276): f32 operands, f32 products and sums throughout
// (v_mfma_f32_32x32x2_f32), head dimensions 32, 64, 96 and 128, 16-byte aligned rows.
//
// Everything is kept transposed, as in the 16-bit kernels (prefill_core.hip.h): S^T[key, query] = K . Q^T, then
// O^T[dim, query] += V^T . P^T.  A wave owns a tile of ROWS query rows, 32 (v_mfma_f32_32x32x2_f32) or 16
// (v_mfma_f32_16x16x4_f32), and walks its keys 32 at a time.  A product contracts one value from each of the wave's
// 64 / ROWS lane groups, and which ones is ours to choose:
//   scores   lane (row = lane % ROWS of K or Q, g = lane / ROWS) holds every (64 / ROWS)-th 16-byte chunk of its row, chunk
//            t * 64 / ROWS + g, so a row comes in 16-byte loads and step (t, j) contracts the j-th value of each group's t-th;
//   values   accumulator register r of lane (query, g) is the score of key 4 g + r (16 rows), 8 (r / 4) + 4 g + (r % 4) (32
//            rows), so the weights are the B operand of step r as they lie, and the A operand is that row of V, of which
//            lane (m = lane % ROWS, g) takes the D / ROWS neighbouring dims m D / ROWS .. and dim block db contracts the db-th.
// Neither operand passes through LDS: 32 keys cost a 32-row wave D products of 64 cycles (D = 64: 4096 cycles) for 256 D
// bytes of K and V, which the caches deliver many times over; a block's V is asked for before its score products, and the
// next block's K before its value products.
//
// What bounds it: the f32 matrix rate (256 flop a cycle and compute unit) where a call fills the chip; below that, how
// long a lone wave takes to walk its row tile's keys.  So a row tile's blocks are dealt out over 1, 2, 4 or 8 waves of its
// workgroup (key_waves, chosen by the host so that the launch fills the SIMDs), which merge their states through LDS, and
// small calls take 16-row tiles, which are twice as many, and fewer of them to a workgroup (row_waves) while compute units
// would be idle: waves on one SIMD take turns at its matrix core.  With 32 rows at head_dim 96 and 128 a wave is alone on its SIMD,
// so what it adds up between its products (see mma_f32) is time of its own.  Measured: see dense_f32_matrix in fmha_prefill.cpp, where both
// are chosen.
#include "common.hip.h"
#include "kernel_args.h"
#include "row_alone.hip.h"

namespace {

// Sums of f32 products: a running sum of n terms of either sign carries a rounding error that grows with sqrt(n), and a
// score's goes into its weight whole.  So a chain of products covers 4 dims of a score up to head_dim 64 (16 rows), 8 or (32
// rows, 96 and up) 16, partial sums meeting in pairs, and 8 or 16 keys of the values: every 32-key block starts two or four
// new sums, which are added to the running ones.  Error against float64, of the norm, and time, with one chain a score and
// one a row's values / as it is / on the row kernels with their per-lane sums:
//   1 x 8 x 512 x 64 causal         2.4e-7  10.3 us  /  1.20e-7  11.3 us  /  1.23e-7   38 us
//   1 x 8 x 512 x 128 causal        3.1e-7  18.8 us  /  1.30e-7  18.8 us  /  1.34e-7   53 us
//   4 x 12 x 1024 x 64              4.2e-7   156 us  /  1.71e-7   142 us  /  2.07e-7  1140 us
//   4 x 12 x 1024 x 128             5.8e-7   240 us  /  1.87e-7   280 us  /  2.20e-7  1740 us
SINGE_DEVICE f32x16_t mma_f32(float a, float b, f32x16_t c) { return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0); }
SINGE_DEVICE f32x4_t mma_f32(float a, float b, f32x4_t c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// A query row's value in its lane groups (lanes l, l ^ 32; with 16-row tiles l ^ 16, l ^ 48 too) combined; equal in all of
// them afterwards.
template <int ROWS>
SINGE_DEVICE float row_max(float value) {
    float kept, taken;
    if constexpr (ROWS == 16) return across_groups_max(value);
    swap_with_self<32>(value, kept, taken);
    return fmaxf(kept, taken);
}
template <int ROWS>
SINGE_DEVICE float row_sum(float value) {
    float kept, taken;
    if constexpr (ROWS == 16) return across_groups_sum(value);
    swap_with_self<32>(value, kept, taken);
    return kept + taken;
}

// N neighbouring floats, in the widest pieces that their alignment (4 N bytes) allows.
template <int N>
SINGE_DEVICE void load_dims(const float* at, float (&value)[N]) {
    constexpr int kWide = N % 4 == 0 ? 4 : N % 2 == 0 ? 2 : 1;
#pragma unroll
    for (int i = 0; i < N; i += kWide) {
        if constexpr (kWide == 4) {
            const float4 four = *reinterpret_cast<const float4*>(at + i);
            value[i] = four.x; value[i + 1] = four.y; value[i + 2] = four.z; value[i + 3] = four.w;
        } else if constexpr (kWide == 2) {
            const float2 two = *reinterpret_cast<const float2*>(at + i);
            value[i] = two.x; value[i + 1] = two.y;
        } else {
            value[i] = at[i];
        }
    }
}
template <int N>
SINGE_DEVICE void store_dims(float* at, const float (&value)[N]) {
    constexpr int kWide = N % 4 == 0 ? 4 : N % 2 == 0 ? 2 : 1;
#pragma unroll
    for (int i = 0; i < N; i += kWide) {
        if constexpr (kWide == 4) *reinterpret_cast<float4*>(at + i) = make_float4(value[i], value[i + 1], value[i + 2], value[i + 3]);
        else if constexpr (kWide == 2) *reinterpret_cast<float2*>(at + i) = make_float2(value[i], value[i + 1]);
        else at[i] = value[i];
    }
}

// Scores of chunks FIRST .. FIRST + COUNT - 1 (of 64 / ROWS lane groups' four dims each): chains of CHAIN products (1, 2, or
// those of whole chunks), summed in pairs.  TIGHT: registers are short, so that the sums must not all be alive at once.
template <int FIRST, int COUNT, int CHAIN, bool TIGHT, class Tile, int TILES, int CHUNKS>
SINGE_DEVICE void score_chunks(Tile (&s)[TILES], const float4 (&k)[TILES][CHUNKS], const float4 (&q)[CHUNKS]) {
    Tile zero;
#pragma unroll
    for (int r = 0; r < static_cast<int>(sizeof(Tile) / 4); ++r) zero[r] = 0.0f;
    if constexpr (4 * COUNT <= CHAIN) {
#pragma unroll
        for (int t = FIRST; t < FIRST + COUNT; ++t) {
#pragma unroll
            for (int kt = 0; kt < TILES; ++kt) s[kt] = mma_f32(k[kt][t].x, q[t].x, t == FIRST ? zero : s[kt]);
#pragma unroll
            for (int kt = 0; kt < TILES; ++kt) s[kt] = mma_f32(k[kt][t].y, q[t].y, s[kt]);
#pragma unroll
            for (int kt = 0; kt < TILES; ++kt) s[kt] = mma_f32(k[kt][t].z, q[t].z, s[kt]);
#pragma unroll
            for (int kt = 0; kt < TILES; ++kt) s[kt] = mma_f32(k[kt][t].w, q[t].w, s[kt]);
        }
    } else if constexpr (COUNT > 1) {
        Tile more[TILES];
        score_chunks<FIRST, COUNT / 2, CHAIN, TIGHT>(s, k, q);
        score_chunks<FIRST + COUNT / 2, COUNT - COUNT / 2, CHAIN, TIGHT>(more, k, q);
#pragma unroll
        for (int kt = 0; kt < TILES; ++kt) s[kt] += more[kt];
        if constexpr (TIGHT) __builtin_amdgcn_sched_barrier(0);
    } else {
#pragma unroll
        for (int kt = 0; kt < TILES; ++kt) {
            const Tile x = mma_f32(k[kt][FIRST].x, q[FIRST].x, zero), y = mma_f32(k[kt][FIRST].y, q[FIRST].y, CHAIN > 1 ? x : zero);
            const Tile z = mma_f32(k[kt][FIRST].z, q[FIRST].z, zero), w = mma_f32(k[kt][FIRST].w, q[FIRST].w, CHAIN > 1 ? z : zero);
            if constexpr (CHAIN > 1) s[kt] = y + w;
            else s[kt] = (x + y) + (z + w);
        }
    }
}

// The sum of values FIRST .. FIRST + COUNT - 1 of a tile, in pairs.
template <int FIRST, int COUNT, class Tile>
SINGE_DEVICE float tile_sum(const Tile& s) {
    if constexpr (COUNT == 1) return s[FIRST];
    else return tile_sum<FIRST, COUNT / 2>(s) + tile_sum<FIRST + COUNT / 2, COUNT - COUNT / 2>(s);
}

// A row of the problem, for row_alone.
struct DenseF32Row {
    const float* query_row;
    const float* keys;    // of the batch entry and kv head
    const float* values;
    size_t key_stride, value_stride;
    float* out_row;
    SINGE_DEVICE unsigned int place(unsigned int k) const { return k; }
    SINGE_DEVICE float query(unsigned int d) const { return query_row[d]; }
    SINGE_DEVICE float key(unsigned int k, unsigned int d) const { return keys[k * key_stride + d]; }
    SINGE_DEVICE float value(unsigned int k, unsigned int d) const { return values[k * value_stride + d]; }
    SINGE_DEVICE void store(unsigned int d, float value) const { out_row[d] = value; }
};

template <int D, int ROWS, int WAVES>
SINGE_DEVICE void attention_mfma_f32_body(const PrefillF32Args& a, float* lds) {
    constexpr int kLaneGroups = 64 / ROWS;
    constexpr int kDimBlocks = D / ROWS, kChunks = D / (4 * kLaneGroups);  // ROWS-dim blocks of O^T; 16-byte chunks a lane holds of a row
    constexpr int kRegs = ROWS * ROWS / 64, kKeyTiles = 32 / ROWS;         // of a score tile; score tiles of a 32-key block
    typedef std::conditional_t<ROWS == 32, f32x16_t, f32x4_t> Tile;
    // Products to a chain of a score, of 64 / ROWS dims each, and sums that a block's keys are dealt out to (see mma_f32).
    constexpr int kScoreChain = ROWS == 16 ? (D <= 64 ? 1 : 2) : (D <= 64 ? 4 : 8), kValueSums = ROWS == 16 && D == 64 ? 4 : 2;
    constexpr bool kTight = WAVES == 8;
    const unsigned int lane = threadIdx.x & 63u;
    const unsigned int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const unsigned int column = lane % ROWS, lane_group = lane / ROWS;
    // Row of an accumulator tile (key of a score tile, dim block of an output tile) that register r holds.
    auto tile_row = [&](int r) __attribute__((always_inline)) { return ROWS == 32 ? 8u * (r >> 2) + 4u * lane_group + (r & 3) : 4u * lane_group + r; };
    const unsigned int key_waves = a.key_waves, row_waves = a.row_waves;
    const unsigned int key_wave = wave % key_waves, row_wave = wave / key_waves;

    // Workgroup -> (batch, head), row tiles: heads side by side (neighbouring workgroups go to different XCDs, and with a
    // multiple of eight (batch, head) pairs a pair's workgroups share one), the last rows, which under the causal mask have
    // the most keys, first.
    const unsigned int pairs = a.batch * a.heads, groups = (a.query_len + ROWS * row_waves - 1) / (ROWS * row_waves);
    const unsigned int bh = blockIdx.x % pairs, group = groups - 1u - blockIdx.x / pairs;
    const unsigned int batch = bh / a.heads, head = bh % a.heads, kv_head = head / (a.heads / a.kv_heads);
    const unsigned int first_row = (group * row_waves + row_wave) * ROWS;
    const bool live = first_row < a.query_len;

    unsigned int key_len = a.key_len;
    if (a.key_lengths != nullptr) {
        const int own = a.key_lengths[batch];
        const unsigned int bound = own > 0 ? static_cast<unsigned int>(own) : 0u;
        key_len = bound < key_len ? bound : key_len;
    }
    // Row `row` sees keys lowest(row) .. end(row) - 1.
    auto lowest = [&](unsigned int row) { return row > a.look_back ? row - a.look_back : 0u; };
    auto end_of = [&](unsigned int row) {
        const unsigned long long end = static_cast<unsigned long long>(row) + a.look_ahead + 1ull;
        return end < key_len ? static_cast<unsigned int>(end) : key_len;
    };
    const unsigned int row = first_row + column < a.query_len ? first_row + column : a.query_len - 1u;
    const unsigned int last_row = first_row + (ROWS - 1) < a.query_len ? first_row + (ROWS - 1) : a.query_len - 1u;
    const unsigned int row_low = lowest(row), row_end = end_of(row);
    const unsigned int tile_end = live ? __builtin_amdgcn_readfirstlane(end_of(last_row)) : 0u;
    const unsigned int first_block = __builtin_amdgcn_readfirstlane(lowest(live ? first_row : 0u)) / 32u, end_block = (tile_end + 31u) / 32u;
    // Blocks from `whole_begin` up to, not including, `whole_end` are seen whole by every row of the tile.
    const unsigned int whole_begin = (__builtin_amdgcn_readfirstlane(lowest(last_row)) + 31u) / 32u;
    const unsigned int whole_end = __builtin_amdgcn_readfirstlane(end_of(live ? first_row : 0u)) / 32u;

    const float* const keys = a.key + batch * a.key_batch_stride + kv_head * a.key_head_stride + 4u * lane_group;
    const float* const values = a.value + batch * a.value_batch_stride + kv_head * a.value_head_stride + column * kDimBlocks;
    // The scale stays out of the scores and goes into the exponent's multiply-add; a negative one moves its sign into Q.
    const float factor = fabsf(a.scale_log2e), sign = a.scale_log2e < 0.0f ? -1.0f : 1.0f;
    float4 q[kChunks];
    {
        const float* at = a.query + batch * a.query_batch_stride + static_cast<size_t>(row) * a.query_sequence_stride + head * a.query_head_stride + 4u * lane_group;
#pragma unroll
        for (int t = 0; t < kChunks; ++t) {
            q[t] = *reinterpret_cast<const float4*>(at + 4 * kLaneGroups * t);
            q[t].x *= sign; q[t].y *= sign; q[t].z *= sign; q[t].w *= sign;
        }
    }

    Tile out[kDimBlocks];
#pragma unroll
    for (int db = 0; db < kDimBlocks; ++db)
#pragma unroll
        for (int r = 0; r < kRegs; ++r) out[db][r] = 0.0f;
    float largest = -INFINITY, total = 0.0f;  // of the row's scaled scores (base two); of this lane's weights

    // A key past the last one the tile sees re-reads that one and is masked.
    const unsigned int last_key = tile_end > 0 ? tile_end - 1u : 0u;
    float4 k[kKeyTiles][kChunks];
    auto load_keys = [&](unsigned int block) __attribute__((always_inline)) {
#pragma unroll
        for (int kt = 0; kt < kKeyTiles; ++kt) {
            const unsigned int wanted = block * 32u + ROWS * kt + column, key = wanted < last_key ? wanted : last_key;
            const float* at = keys + static_cast<size_t>(key) * a.key_sequence_stride;
#pragma unroll
            for (int t = 0; t < kChunks; ++t) k[kt][t] = *reinterpret_cast<const float4*>(at + 4 * kLaneGroups * t);
        }
    };
    unsigned int block = first_block + key_wave;
    if (block < end_block) load_keys(block);
    for (; block < end_block; block += key_waves) {
        float v[kKeyTiles][kRegs][kDimBlocks];
#pragma unroll
        for (int kt = 0; kt < kKeyTiles; ++kt)
#pragma unroll
            for (int r = 0; r < kRegs; ++r) {
                const unsigned int wanted = block * 32u + ROWS * kt + tile_row(r), key = wanted < last_key ? wanted : last_key;
                load_dims(values + static_cast<size_t>(key) * a.value_sequence_stride, v[kt][r]);
            }
        Tile s[kKeyTiles];
        score_chunks<0, kChunks, kScoreChain, kTight>(s, k, q);
#pragma unroll
        for (int kt = 0; kt < kKeyTiles; ++kt) asm volatile("" : "+v"(s[kt]));  // (summed here, not after the loads below)
        if (block + key_waves < end_block) load_keys(block + key_waves);
        if (block < whole_begin || block >= whole_end) {
            asm volatile("");  // keeps this a branch: as selects it would be paid in every block
#pragma unroll
            for (int kt = 0; kt < kKeyTiles; ++kt)
#pragma unroll
                for (int r = 0; r < kRegs; ++r) {
                    const unsigned int key = block * 32u + ROWS * kt + tile_row(r);
                    s[kt][r] = key < row_low || key >= row_end ? -INFINITY : s[kt][r];
                }
        }
        float most = -INFINITY;
#pragma unroll
        for (int kt = 0; kt < kKeyTiles; ++kt)
#pragma unroll
            for (int r = 0; r < kRegs; ++r) most = fmaxf(most, s[kt][r]);
        most = row_max<ROWS>(most) * factor;
        if (__any(most > largest)) {
            const float moved = fmaxf(largest, most), base = moved == -INFINITY ? 0.0f : moved;
            const float rescale = fast_exp2(largest - base);
            total *= rescale;
#pragma unroll
            for (int db = 0; db < kDimBlocks; ++db)
#pragma unroll
                for (int r = 0; r < kRegs; ++r) out[db][r] *= rescale;
            largest = moved;
        }
        const float base = largest == -INFINITY ? 0.0f : largest;
#pragma unroll
        for (int kt = 0; kt < kKeyTiles; ++kt)
#pragma unroll
            for (int r = 0; r < kRegs; ++r) {
                s[kt][r] = fast_exp2(fmaf(s[kt][r], factor, -base));
            }
        if constexpr (ROWS == 16) total += tile_sum<0, kRegs>(s[0]) + tile_sum<0, kRegs>(s[kKeyTiles - 1]);
        else total += tile_sum<0, kRegs>(s[0]);
        constexpr int kSumKeys = kKeyTiles * kRegs / kValueSums;  // products of each of the block's sums
        Tile ready;
#pragma unroll
        for (int db = 0; db < kDimBlocks; ++db) {
            Tile part[kValueSums];
#pragma unroll
            for (int h = 0; h < kValueSums; ++h)
#pragma unroll
                for (int r = 0; r < kRegs; ++r) part[h][r] = 0.0f;
            if constexpr (kTight) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < kSumKeys; ++i)
#pragma unroll
                for (int h = 0; h < kValueSums; ++h) {
                    const int at = h * kSumKeys + i, kt = at / kRegs, r = at % kRegs;
                    part[h] = mma_f32(v[kt][r][db], s[kt][r], part[h]);
                }
            // (the sums are added while the next dim block's products run)
            if (db > 0) out[db - 1] += ready;
            if constexpr (kValueSums == 4) ready = (part[0] + part[1]) + (part[2] + part[3]);
            else ready = part[0] + part[1];
        }
        out[kDimBlocks - 1] += ready;
    }
    total = row_sum<ROWS>(total);

    float* const out_row = a.out + batch * a.output_batch_stride + static_cast<size_t>(row) * a.output_sequence_stride + head * a.output_head_stride;
    const bool stored = live && first_row + column < a.query_len;
    auto store = [&](int r, const float (&value)[kDimBlocks]) __attribute__((always_inline)) { store_dims(out_row + kDimBlocks * tile_row(r), value); };
    // A row that sees no key stays zero; its log-sum-exp is ln 0.
    auto store_lse = [&](float reference, float sum) __attribute__((always_inline)) {
        if (a.lse != nullptr && stored && lane_group == 0)
            a.lse[(static_cast<size_t>(batch) * a.heads + head) * a.query_len + row] = sum > 0.0f ? fmaf(reference, kLn2, log2f(sum) * kLn2) : -INFINITY;
    };
    // Rows of the tile (bit r: row r) whose sums a value that is not finite has spoilt: worked out by themselves.  (Where the
    // weights' sum is NaN, so is the score of a key the row sees, and every output of it either way.)
    const unsigned long long spoiled = __builtin_amdgcn_ballot_w64(stored && total == total && not_finite(kRegs * kDimBlocks, [&](int i) { return out[i / kRegs][i % kRegs]; }));
    unsigned int alone = static_cast<unsigned int>(spoiled | spoiled >> 32);
    if constexpr (ROWS == 16) alone = (alone | alone >> 16) & 0xffffu;
    auto redo = [&](unsigned int rows) __attribute__((always_inline)) {
        for (; rows != 0; rows &= rows - 1u) {
            const unsigned int own = first_row + static_cast<unsigned int>(__builtin_ctz(rows));
            row_alone<D>(DenseF32Row{a.query + batch * a.query_batch_stride + static_cast<size_t>(own) * a.query_sequence_stride + head * a.query_head_stride,
                                     a.key + batch * a.key_batch_stride + kv_head * a.key_head_stride,
                                     a.value + batch * a.value_batch_stride + kv_head * a.value_head_stride, a.key_sequence_stride, a.value_sequence_stride,
                                     a.out + batch * a.output_batch_stride + static_cast<size_t>(own) * a.output_sequence_stride + head * a.output_head_stride},
                         lowest(own), end_of(own), a.scale_log2e);
        }
    };
    if (key_waves == 1) {
        const float inverse = total > 0.0f ? 1.0f / total : 0.0f;
        if (stored && ((alone >> column) & 1u) == 0) {
#pragma unroll
            for (int r = 0; r < kRegs; ++r) {
                float value[kDimBlocks];
#pragma unroll
                for (int db = 0; db < kDimBlocks; ++db) value[db] = out[db][r] * inverse;
                store(r, value);
            }
        }
        store_lse(largest, total);
        redo(alone);
        return;
    }
    // The row tile's waves leave their states in LDS, and each merges and stores a share of the accumulator registers.
    constexpr unsigned int kSlot = 64u * (kRegs * kDimBlocks + 2);
    float* const mine = lds + (row_wave * key_waves + key_wave) * kSlot + lane;
#pragma unroll
    for (int r = 0; r < kRegs; ++r)
#pragma unroll
        for (int db = 0; db < kDimBlocks; ++db) mine[64 * (r * kDimBlocks + db)] = out[db][r];
    mine[64 * kRegs * kDimBlocks] = largest;
    mine[64 * (kRegs * kDimBlocks + 1)] = total;
    unsigned int* const alone_of = reinterpret_cast<unsigned int*>(lds + WAVES * kSlot);  // a word a wave
    if (lane == 0) alone_of[row_wave * key_waves + key_wave] = alone;
    __syncthreads();
    for (unsigned int w = 0; w < key_waves; ++w) alone |= alone_of[row_wave * key_waves + w];
    alone = __builtin_amdgcn_readfirstlane(alone);
    const float* const tile = lds + row_wave * key_waves * kSlot + lane;
    float reference = -INFINITY;
    for (unsigned int w = 0; w < key_waves; ++w) reference = fmaxf(reference, tile[w * kSlot + 64 * kRegs * kDimBlocks]);
    const float base = reference == -INFINITY ? 0.0f : reference;
    float sum = 0.0f;
    for (unsigned int w = 0; w < key_waves; ++w)
        sum += tile[w * kSlot + 64 * (kRegs * kDimBlocks + 1)] * fast_exp2(tile[w * kSlot + 64 * kRegs * kDimBlocks] - base);
    const float inverse = sum > 0.0f ? 1.0f / sum : 0.0f;
    // (with more waves than registers, the last ones have none)
    for (unsigned int r = key_wave; r < static_cast<unsigned int>(kRegs); r += key_waves) {
        float value[kDimBlocks] = {};
        for (unsigned int w = 0; w < key_waves; ++w) {
            const float weight = fast_exp2(tile[w * kSlot + 64 * kRegs * kDimBlocks] - base);
#pragma unroll
            for (int db = 0; db < kDimBlocks; ++db) value[db] = fmaf(tile[w * kSlot + 64 * (r * kDimBlocks + db)], weight, value[db]);
        }
#pragma unroll
        for (int db = 0; db < kDimBlocks; ++db) value[db] *= inverse;
        if (stored && ((alone >> column) & 1u) == 0) store(static_cast<int>(r), value);
    }
    if (key_wave == 0) store_lse(reference, sum);
    // (row r of the tile falls to wave r % key_waves)
    unsigned int share = 0;
    for (unsigned int r = key_wave; r < ROWS; r += key_waves) share |= 1u << r;
    redo(alone & share);
}

}  // namespace

// From head_dim 96 on a 32-row wave needs more than half a SIMD's registers: four waves a workgroup, one a SIMD.
#define SINGE_ATTENTION_MFMA_F32_KERNEL(DIM, ROWS, WAVES)                                                                 \
    extern "C" __global__ __launch_bounds__(64 * WAVES, WAVES / 4) void singe_attention_mfma_f32_d##DIM##_r##ROWS(PrefillF32Args args) { \
        __shared__ float lds[WAVES * (ROWS * DIM + 128 + 1)];                                                                 \
        attention_mfma_f32_body<DIM, ROWS, WAVES>(args, lds);                                                             \
    }

SINGE_ATTENTION_MFMA_F32_KERNEL(32, 16, 8)
SINGE_ATTENTION_MFMA_F32_KERNEL(64, 16, 8)
SINGE_ATTENTION_MFMA_F32_KERNEL(96, 16, 8)
SINGE_ATTENTION_MFMA_F32_KERNEL(128, 16, 8)
SINGE_ATTENTION_MFMA_F32_KERNEL(64, 32, 8)
SINGE_ATTENTION_MFMA_F32_KERNEL(96, 32, 4)
SINGE_ATTENTION_MFMA_F32_KERNEL(128, 32, 4)
