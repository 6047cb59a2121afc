// One query row by itself, on a whole wave and without the matrix cores: what a row tile's kernel falls back to for a row
// whose sums met a value that is not finite.
//
// The matrix products weigh every value of a block, those of keys that the row does not see by zero, and 0 * inf and
// 0 * NaN are NaN.  So a value that is not finite at one key spoils every row of the tiles that reach it, also the rows
// that the key is hidden from.  A row so spoiled holds something that is not finite in its sums (nothing takes it away
// again), which costs one pass over the accumulators to see (`not_finite`); its output is then worked out again here from
// the keys it sees and no others, as a kernel with a wave a row would have done.  Rows of finite values never come here.
#pragma once

#include "common.hip.h"

namespace {

// Whether any of `count` values is an infinity or NaN: x * 0 is zero for every other.
template <class Values>
SINGE_DEVICE bool not_finite(int count, Values&& value) {
    float sum = 0.0f;
#pragma unroll
    for (int i = 0; i < count; ++i) sum = fmaf(value(i), 0.0f, sum);
    return sum != sum;
}

//   row.place(k)                                   where key k lies, as the next two take it
//   row.query(d), row.key(at, d), row.value(at, d) the operands as f32
//   row.store(d, value)                            takes the output
// The row sees keys begin .. end - 1.  Called by all 64 lanes with the same arguments.
template <int D, class Row>
SINGE_DEVICE void row_alone(const Row& row, unsigned int begin, unsigned int end, float scale_log2e) {
    constexpr int kHeld = (D + 63) / 64;  // dims of a lane: lane, lane + 64
    unsigned int lane = threadIdx.x & 63u;
    asm volatile("" : "+v"(lane));  // (what is worked out from it here stays here, out of the caller's loops and registers)
    float out[kHeld];
#pragma unroll
    for (int h = 0; h < kHeld; ++h) out[h] = 0.0f;
    float largest = -INFINITY, total = 0.0f;
    for (unsigned int first = begin; first < end; first += 64u) {  // a key a lane for the scores
        float score = -INFINITY;
        if (first + lane < end) {
            const auto at = row.place(first + lane);
            float dot = 0.0f;
#pragma unroll 4
            for (int d = 0; d < D; ++d) dot = fmaf(row.query(d), row.key(at, d), dot);
            score = dot * scale_log2e;
        }
        float most = score;
#pragma unroll
        for (int step = 32; step > 0; step >>= 1) most = fmaxf(most, __shfl_xor(most, step, 64));
        const float moved = fmaxf(largest, most), base = moved == -INFINITY ? 0.0f : moved, rescale = fast_exp2(largest - base);
        largest = moved;
        float weight = fast_exp2(score - base), sum = weight;
#pragma unroll
        for (int step = 32; step > 0; step >>= 1) sum += __shfl_xor(sum, step, 64);
        total = fmaf(total, rescale, sum);
#pragma unroll
        for (int h = 0; h < kHeld; ++h) out[h] *= rescale;
        const unsigned int count = end - first < 64u ? end - first : 64u;
        for (unsigned int k = 0; k < count; ++k) {
            if (__shfl(score, k, 64) == -INFINITY) continue;
            const float w = __shfl(weight, k, 64);
            const auto at = row.place(first + k);
#pragma unroll
            for (int h = 0; h < kHeld; ++h)
                if (lane + 64u * h < D) out[h] = fmaf(w, row.value(at, lane + 64u * h), out[h]);
        }
    }
    const float inverse = total > 0.0f ? 1.0f / total : 0.0f;
#pragma unroll
    for (int h = 0; h < kHeld; ++h)
        if (lane + 64u * h < D) row.store(lane + 64u * h, out[h] * inverse);
}

}  // namespace
