// Host side of dense prefill: FmhaPrefillConfig validation as the reference does it
// (singe-kernel/src/cuda/attention/mod.rs:1602-1756, 3369-3398, 3647-3677) and the launch.
#include <atomic>
#include <cmath>

#include "kernel_args.h"
#include "module.h"
#include "singe_hip_attention.h"
#include "validate.h"
#include "window_runs.h"

using namespace singe_hip;

namespace {

// Query rows a wave of the dense bf16 / f16 prefill takes: 0 = chosen by problem size, 32, or 64 where the two-tile
// kernel takes the call (singe_hip_set_dense_prefill_rows_per_wave).
std::atomic<uint32_t> g_rows_per_wave{0};

int32_t validate_config(const SingeFmhaPrefillConfig& c) {
    const size_t extents[] = {c.batch, c.query_len, c.key_len, c.heads, c.kv_heads, c.head_dim,
                              c.query_batch_stride, c.key_batch_stride, c.value_batch_stride, c.output_batch_stride,
                              c.query_sequence_stride, c.key_sequence_stride, c.value_sequence_stride,
                              c.output_sequence_stride, c.query_head_stride, c.key_head_stride,
                              c.value_head_stride, c.output_head_stride};
    for (size_t extent : extents)
        if (extent == 0) return fail(SINGE_HIP_INVALID_LENGTH, "config");
    if (!std::isfinite(c.scale) || c.heads % c.kv_heads != 0) return fail(SINGE_HIP_INVALID_LENGTH, "config");
    return 0;
}

// projected_layout_reach (mod.rs:3647-3668): elements one batch item can address.
bool layout_reach(size_t sequence_len, size_t heads, size_t head_dim, size_t sequence_stride, size_t head_stride, size_t* out) {
    size_t sequence_span, head_span;
    if (sequence_len == 0 || heads == 0) return false;
    return checked_mul(sequence_len - 1, sequence_stride, &sequence_span) && checked_mul(heads - 1, head_stride, &head_span) &&
           checked_add(sequence_span, head_span, out) && checked_add(*out, head_dim, out);
}

// batched_reach (mod.rs:3670-3677).
bool batched_reach(size_t batch, size_t item_len, size_t batch_stride, size_t* out) {
    size_t span;
    if (batch == 0) return false;
    return checked_mul(batch - 1, batch_stride, &span) && checked_add(span, item_len, out);
}

int32_t ensure_reach(const char* name, size_t actual, size_t batch, size_t sequence_len, size_t heads, size_t head_dim,
                     size_t batch_stride, size_t sequence_stride, size_t head_stride) {
    size_t item = 0, need = 0;
    if (!layout_reach(sequence_len, heads, head_dim, sequence_stride, head_stride, &item) ||
        !batched_reach(batch, item, batch_stride, &need))
        return fail(SINGE_HIP_SIZE_OVERFLOW, name);
    return ensure_len_at_least(name, actual, need);
}

// FmhaPrefillConfig::validate_lengths / validate_output_lengths (mod.rs:1634-1756), in their order,
// then the null checks every DevicePointer implies.
int32_t validate_call(const SingeFmhaPrefillConfig& c, const void* out, size_t out_len, const void* lse, size_t lse_len,
                      bool with_lse, const void* query, size_t query_len, const void* key, size_t key_len,
                      const void* value, size_t value_len) {
    if (int32_t status = validate_config(c)) return status;
    if (int32_t status = ensure_reach("query", query_len, c.batch, c.query_len, c.heads, c.head_dim, c.query_batch_stride,
                                      c.query_sequence_stride, c.query_head_stride)) return status;
    if (int32_t status = ensure_reach("key", key_len, c.batch, c.key_len, c.kv_heads, c.head_dim, c.key_batch_stride,
                                      c.key_sequence_stride, c.key_head_stride)) return status;
    if (int32_t status = ensure_reach("value", value_len, c.batch, c.key_len, c.kv_heads, c.head_dim, c.value_batch_stride,
                                      c.value_sequence_stride, c.value_head_stride)) return status;
    if (int32_t status = ensure_reach("out", out_len, c.batch, c.query_len, c.heads, c.head_dim, c.output_batch_stride,
                                      c.output_sequence_stride, c.output_head_stride)) return status;
    if (with_lse) {
        size_t rows = 0;
        if (!checked_mul(c.batch, c.heads, &rows) || !checked_mul(rows, c.query_len, &rows)) return fail(SINGE_HIP_SIZE_OVERFLOW, "lse");
        if (int32_t status = ensure_len_at_least("lse", lse_len, rows)) return status;
        if (lse == nullptr) return fail(SINGE_HIP_NULL_POINTER, "lse");
    }
    const void* pointers[] = {out, query, key, value};
    const char* names[] = {"out", "query", "key", "value"};
    for (int i = 0; i < 4; ++i)
        if (pointers[i] == nullptr) return fail(SINGE_HIP_NULL_POINTER, names[i]);
    if (!fits_i32(c.query_len) || !fits_i32(c.key_len) || !fits_i32(c.batch) || !fits_i32(c.heads))
        return fail(SINGE_HIP_LENGTH_EXCEEDS_I32, "config");
    return 0;
}

// Small calls without shared heads that the row kernel (a workgroup per (batch, query, kv head)) is done with first: a
// matrix-core wave's one or two blocks take it as long however few rows there are.  Kernel times in us, row / matrix-core
// kernel (batch x heads x queries x keys):
//   head_dim 128   1 x 1 x 64 x 64 6.0 / 7.0    1 x 1 x 200 x 200 9.6 / 11.9   1 x 1 x 512 x 512 18.4 / 19.1
//                  1 x 8 x 64 x 64 7.1 / 7.2    1 x 8 x 100 x 100 10.9 / 9.0   1 x 1 x 64 x 4096 105 / 94
//   head_dim 64    1 x 1 x 16 x 16 4.0 / 4.2    1 x 1 x 100 x 100  6.1 / 6.0   1 x 8 x 64 x 64 5.7 / 5.6
// With heads that share their keys the row kernel takes longer the more there are (1 x 8 over 2 x 64 x 64 x 1024: 73 / 32).
bool rows_f32_is_faster(const PrefillF32Args& a) {
    if (a.heads != a.kv_heads) return false;
    const uint64_t rows = static_cast<uint64_t>(a.batch) * a.heads * a.query_len;
    return (a.head_dim == 128 && rows <= 512 && a.key_len <= 1024) || (a.head_dim == 64 && rows <= 192 && a.key_len <= 64);
}

int32_t prefill_f32(void* stream, float* out, size_t out_len, float* lse, size_t lse_len, bool with_lse, const float* query,
                    size_t query_len, const float* key, size_t key_len, const float* value, size_t value_len,
                    const SingeFmhaPrefillConfig* config, size_t window_size, bool has_soft_cap, float soft_cap,
                    const char* op) {
    if (config == nullptr) return fail(SINGE_HIP_NULL_POINTER, "config");
    const SingeFmhaPrefillConfig& c = *config;
    if (int32_t status = validate_call(c, out, out_len, lse, lse_len, with_lse, query, query_len, key, key_len, value, value_len))
        return status;
    if (c.head_dim > 256) return fail(SINGE_HIP_UNSUPPORTED_WIDTH, op, c.head_dim, 0);
    // (the cap first, then the window: validate_softcapped_window_attention_config, singe-kernel/src/cuda/attention/mod.rs:3418-3430)
    if (has_soft_cap && !(std::isfinite(soft_cap) && soft_cap > 0.0f)) return fail(SINGE_HIP_INVALID_LENGTH, "soft_cap");
    if (!fits_i32(window_size)) return fail(SINGE_HIP_LENGTH_EXCEEDS_I32, "window_size");
    PrefillF32Args args;
    args.query = query;
    args.key = key;
    args.value = value;
    args.out = out;
    args.lse = with_lse ? lse : nullptr;
    args.query_batch_stride = c.query_batch_stride;
    args.query_sequence_stride = c.query_sequence_stride;
    args.query_head_stride = c.query_head_stride;
    args.key_batch_stride = c.key_batch_stride;
    args.key_sequence_stride = c.key_sequence_stride;
    args.key_head_stride = c.key_head_stride;
    args.value_batch_stride = c.value_batch_stride;
    args.value_sequence_stride = c.value_sequence_stride;
    args.value_head_stride = c.value_head_stride;
    args.output_batch_stride = c.output_batch_stride;
    args.output_sequence_stride = c.output_sequence_stride;
    args.output_head_stride = c.output_head_stride;
    args.batch = static_cast<uint32_t>(c.batch);
    args.query_len = static_cast<uint32_t>(c.query_len);
    args.key_len = static_cast<uint32_t>(c.key_len);
    args.heads = static_cast<uint32_t>(c.heads);
    args.kv_heads = static_cast<uint32_t>(c.kv_heads);
    args.head_dim = static_cast<uint32_t>(c.head_dim);
    args.causal = c.causal ? 1u : 0u;
    args.window_size = static_cast<uint32_t>(window_size);
    args.has_soft_cap = has_soft_cap ? 1u : 0u;
    args.soft_cap = soft_cap;
    args.scale = c.scale;
    if (!has_soft_cap && !rows_f32_is_faster(args) && dense_f32_matrix_takes(args)) {
        if (window_size > 0) args.look_back = args.look_ahead = static_cast<uint32_t>(window_size);
        if (c.causal) args.look_ahead = 0;
        return dense_f32_matrix(stream, args);
    }
    // Head dimensions that are powers of two from 4 to 256 take the row kernel (a workgroup per (batch, query, kv
    // head), several keys per wave step); the rest the one-wave-per-row kernel below.
    const size_t widths[] = {4, 8, 16, 32, 64, 128, 256};
    for (int index = 0; index < 7; ++index) {
        if (c.head_dim != widths[index]) continue;
        const size_t strides[] = {c.query_batch_stride, c.query_sequence_stride, c.query_head_stride, c.key_batch_stride,
                                  c.key_sequence_stride, c.key_head_stride, c.value_batch_stride, c.value_sequence_stride,
                                  c.value_head_stride};
        bool aligned = ((reinterpret_cast<uintptr_t>(query) | reinterpret_cast<uintptr_t>(key) | reinterpret_cast<uintptr_t>(value)) & 15u) == 0;
        for (size_t stride : strides) aligned = aligned && stride % 4 == 0;
        args.aligned = aligned ? 1u : 0u;
        const uint64_t units = static_cast<uint64_t>(c.batch) * c.query_len * c.kv_heads;
        if (units > 0x7fffffffull) return fail(SINGE_HIP_UNSUPPORTED_CONFIGURATION, "too many workgroups");
        return launch(static_cast<KernelId>(kPrefillRowsF32 + index), static_cast<unsigned>(units), 1, 1, 256, stream, args);
    }
    const uint64_t rows = static_cast<uint64_t>(c.batch) * c.heads * c.query_len;
    const uint64_t groups = (rows + 3) / 4;
    if (groups > 0x7fffffffull) return fail(SINGE_HIP_UNSUPPORTED_CONFIGURATION, "too many workgroups");
    const KernelId kernel = c.head_dim <= 32 ? kPrefillF32D32 : c.head_dim <= 64 ? kPrefillF32D64
                            : c.head_dim <= 128 ? kPrefillF32D128 : kPrefillF32D256;
    return launch(kernel, static_cast<unsigned>(groups), 1, 1, 256, stream, args);
}

}  // namespace

namespace singe_hip {

bool dense_f32_matrix_takes(const PrefillF32Args& a) {
    if (a.head_dim != 32 && a.head_dim != 64 && a.head_dim != 96 && a.head_dim != 128) return false;
    const uintptr_t addresses = reinterpret_cast<uintptr_t>(a.query) | reinterpret_cast<uintptr_t>(a.key) | reinterpret_cast<uintptr_t>(a.value) |
                                reinterpret_cast<uintptr_t>(a.out);
    const uint64_t strides = a.query_batch_stride | a.query_sequence_stride | a.query_head_stride | a.key_batch_stride | a.key_sequence_stride |
                             a.key_head_stride | a.value_batch_stride | a.value_sequence_stride | a.value_head_stride | a.output_batch_stride |
                             a.output_sequence_stride | a.output_head_stride;
    return addresses % 16 == 0 && strides % 4 == 0 &&
           static_cast<uint64_t>(a.batch) * a.heads * ((static_cast<uint64_t>(a.query_len) + 15) / 16) <= 0x7fffffffull;
}

int32_t dense_f32_matrix(void* stream, PrefillF32Args& a) {
    a.scale_log2e = logit_factor(a.scale);
    // 16-row tiles where 32-row ones are too few for the chip (up to 5/8 of a tile a compute unit; at head_dim 32 always, where
    // a wave's loads and softmax weigh more than its products), and a tile's keys over as many waves as leave the SIMDs two to
    // four waves each.  Kernel times in us (B x H x L, causal; 16 rows with 1 / 2 / 4 / 8 waves, then 32 rows with 1 / 2 / 4 / 8):
    //   head_dim 64   1 x 8 x 512     30 / 18 / 12 / 12     45 / 27 / 17 / 18     (the row kernel: 38)
    //                 1 x 12 x 1024   67 / 40 / 34 / 36     87 / 58 / 37 / 32
    //                 4 x 12 x 1024   97 / 98 / 111 / 129  116 / 89 / 92 / 102
    //   head_dim 128  1 x 8 x 512     48 / 27 / 18 / 19     84 / 47 / 29 (four waves a workgroup)
    //                 4 x 8 x 512     53 / 54 / 45 / 52     88 / 52 / 44
    //                 4 x 12 x 1024  169 / 174 / 198 / 232 178 / 172 / 188;  not causal 341 / 280 / 319 / 375  355 / 283 / 303
    //   head_dim 96   4 x 12 x 1024  132 / 135 / 150 / 177 141 / 137 / 150
    //   head_dim 32   4 x 12 x 1024   68 / 50 / 52 / 55
    // A wave without a block of its own costs nothing: 7 blocks on 8 waves take 12.1 us, on 4 waves 18.8 (1 x 8 x 200 x 128).
    const uint64_t pairs = static_cast<uint64_t>(a.batch) * a.heads, blocks = (static_cast<uint64_t>(a.key_len) + 31) / 32, units = compute_units();
    const uint32_t rows = a.head_dim == 32 || pairs * ((static_cast<uint64_t>(a.query_len) + 31) / 32) * 8 <= 5 * units ? 16 : 32;
    const uint32_t waves = rows == 16 || a.head_dim <= 64 ? 8 : 4;  // of a workgroup
    const uint64_t tiles = (static_cast<uint64_t>(a.query_len) + rows - 1) / rows, most = (rows == 16 ? 32 : 2 * waves) * units;
    a.key_waves = 1;
    while (a.key_waves < waves && pairs * tiles * a.key_waves < most && a.key_waves < blocks) a.key_waves *= 2;
    a.row_waves = waves / a.key_waves;
    while (a.row_waves > 1 && pairs * ((tiles + a.row_waves - 1) / a.row_waves) < units) a.row_waves /= 2;
    const uint64_t groups = (tiles + a.row_waves - 1) / a.row_waves;
    const int kernel = kAttentionMfmaF32 + static_cast<int>(rows == 16 ? a.head_dim / 32 - 1 : a.head_dim / 32 + 2);
    return launch(static_cast<KernelId>(kernel), static_cast<unsigned>(pairs * groups), 1, 1, 64 * a.key_waves * a.row_waves, stream, a);
}

}  // namespace singe_hip

namespace {

// Whether a call without options runs on the kernel that gives a wave two 32-row tiles: a head_dim that is a multiple of 16
// up to 128, a positive scale, no heads packed into one tile, and (unless the knob says 64) where it is the faster one:
// enough of its workgroups (pairs of 256-row tiles, one to a compute unit) in whole rounds of the chip, and enough keys to
// each that the ends of a tile do not weigh.  32-row / two-tile kernel, us, batch * heads x length (workgroups; equal
// query and key counts, a seventh of the shapes timed):
//   head_dim 128, causal  128 x 600 (256) 35 / 41    256 x 768 (512) 65 / 85     256 x 1280 (768)  141 / 151   96 x 1536 (288) 101 / 112
//                         64 x 1536 (192) 71 / 56    128 x 1536 (384) 102 / 113  256 x 1536 (768)  186 / 185   64 x 1792 (256)  81 / 67
//                         64 x 2048 (256) 81 / 77    64 x 2560 (320) 149 / 155   128 x 2048 (512)  156 / 151   32 x 3072 (192) 111 / 87
//                         64 x 3072 (384) 183 / 183  128 x 3072 (768) 326 / 298  128 x 4096 (1024) 558 / 506
//   head_dim 128, full    128 x 768 (256) 53 / 54    256 x 768 (512) 97 / 103    256 x 1024 (512)  149 / 142   96 x 1280 (288)  90 / 110
//                         64 x 1280 (192) 76 / 68    32 x 2560 (160) 137 / 117   32 x 2048 (128)    73 / 97    128 x 4096       1037 / 918
//   head_dim 96           causal 64 x 1536 64 / 50, 128 x 1536 91 / 99, 128 x 4096 479 / 425; full 96 x 1280 78 / 97, 128 x 4096 880 / 770
//   head_dim 64, causal   96 x 1536 (288) 54 / 83    128 x 1024 (256) 32 / 38    256 x 1280 (768)   80 / 112   128 x 4096 (1024) 332 / 346
//   head_dim 64, full     128 x 1280 (384) 75 / 105  128 x 2048 (512) 175 / 170  256 x 2048 (1024) 322 / 327   64 x 4096 (512)   337 / 310
// (Up to 64 the 32-row kernel holds three workgroups a compute unit and the softmax's vector instructions bound both: two or
// three waves a SIMD share them out better than one.)
// Where the two lengths differ, in the same units, batch * heads x queries x keys:
//   a causal row past the last key sees them all, so that tiles are as even as without the mask
//     head_dim 128          128 x 4096 x 1024 (1024) 278 / 267    64 x 4096 x 1500 (512) 189 / 176    64 x 2048 x 700 (256) 54 / 56
//     head_dim 64           64 x 4096 x 1500 (512) 137 / 129      32 x 8192 x 2048 (512) 187 / 158    (64 x 4096 x 4096 (512) 179 / 172)
//   few keys without the mask: only for a round of full tiles, 2048 queries and up
//     head_dim 128          64 x 2048 x 512 (256) 47 / 45         32 x 4096 x 800 (256) 65 / 60       256 x 1024 x 512 (512) 90 / 91
//     head_dim 96           64 x 2048 x 860 (256) 59 / 56         64 x 4096 x 300 (512) 57 / 64       128 x 2048 x 512 (512) 76 / 77
//   one 256-row tile to a head takes its keys from memory once, two 128-row tiles of a workgroup twice
//     head_dim 48           512 x 160 x 1024 (512) 73 / 51        1024 x 256 x 512 (1024) 82 / 68     256 x 256 x 512 (256) 18 / 19
//     head_dim 64           1024 x 256 x 2048 (1024) 263 / 206    512 x 256 x 1024 (512) 55 / 55      1024 x 256 x 512 (1024) 64 / 67
//     head_dim 80           512 x 256 x 1024 (512) 89 / 67        1024 x 160 x 512 (1024) 92 / 79     1024 x 256 x 1024, causal 55 / 67
// Narrow heads without the mask in two rounds: 64 x 3500 (448) 279 / 256 at head_dim 64, 272 / 251 at 48; of short rows, whose last
// tiles are not whole, 256 x 700 x 3000 (512) 172 / 226.  What the lines cost against the faster kernel, of 520 shapes: up to 11 %
// for narrow heads without the mask in many rounds (head_dim 48, 256 x 4096 (2048) 1154 / 1281, on the two-tile kernel), 9 % under it
// at head_dim 48 (32 x 8192 (512) 331 / 305, on the 32-row one), 7 % for 128 x 2048 (512) at 64 without it (174 / 162) and from 80 up.
// (Workgroups are counted with (batch, head)s rounded up to a multiple of eight, as the lines were drawn, though the launch deals
// them out evenly: counted as dealt, 28 x 2560, 18 x 4096 and 12 x 6000 without the mask would go to the 32-row kernel, 132, 205 and
// 296 us in place of 113, 171 and 246.)
bool two_tiles_a_wave(const SingeFmhaPrefillConfig& c) {
    const uint32_t wanted = g_rows_per_wave.load(std::memory_order_relaxed);
    if (wanted == 32 || !has_pair_build(static_cast<long long>(c.head_dim)) || c.key_len == 0 || !(c.scale > 0.0f) || dense_prefill_packs_heads(c))
        return false;
    if (wanted == 64) return true;
    const uint64_t rows = (static_cast<uint64_t>(c.batch) * c.heads + 7) / 8 * 8, pair_tiles = (c.query_len + 255) / 256;
    const uint64_t units = compute_units(), workgroups = rows * ((pair_tiles + 1) / 2), rounds = (workgroups + units - 1) / units;
    const uint64_t seen = c.causal && c.query_len < c.key_len ? c.query_len : c.key_len;
    const uint64_t share = 100 * workgroups / (rounds * units);  // of the rounds' places that a workgroup takes, in percent
    if (c.head_dim < 48) return false;
    if (!c.causal && pair_tiles == 1 && c.query_len > 128 && workgroups >= 2 * units && seen >= (c.head_dim == 64 ? 2048 : 512)) return true;
    const bool two_whole_rounds = rounds == 2 && share >= 85;
    if (c.head_dim <= 64) {
        if (c.causal) return c.head_dim == 64 && two_whole_rounds && share >= 95 && c.query_len >= 4096 && seen >= 1000;
        return (seen >= 4096 && workgroups >= units && share >= 90) || (two_whole_rounds && seen >= 3000 && c.query_len >= 3000);
    }
    if (4 * workgroups < 3 * units) return !c.causal && seen >= 2560 && 8 * workgroups >= 5 * units;
    if (!c.causal)
        return (seen >= 900 && !(rounds == 2 && 4 * workgroups < 5 * units && seen < 1536)) ||
               (rounds == 1 && share >= 95 && c.query_len >= 2048 && seen >= 512);
    if (2 * c.query_len >= 5 * c.key_len && c.key_len >= 1024 && share >= 90) return true;
    return seen >= 3072 || (seen >= 2048 && share >= 70) || (seen >= 1536 && (rounds == 1 || share >= 95));
}

// Short causal windows over grouped heads, where a workgroup of eight waves walks along a run of rows with the keys its windows
// reach kept in LDS (fmha_window.hip.h): how many blocks of 32 keys it holds, how many runs a (batch, kv head) pair's rows are
// cut into and how many steps of 256 rows a run has; no runs where the call is not for that kernel, which are windows whose
// blocks do not fit LDS (half of it where rows are 128 bytes, since a compute unit must hold two workgroups there: one took
// 0.97 to 1.3 x the row tiles' time), and launches that do not give a compute unit its step (129 steps and up; at most 1.13 x
// below).  Row tiles / runs, us (heads x head_dim, batch x length, window; steps of all pairs):
//   64 / 8 x 64    1 x 8192, 16 (2048)  48 / 31     128   58 / 41     256   70 / 55     512   98 / 100 (left on row tiles)
//                  4 x 8192, 128 (8192) 224 / 173   1 x 1500, 128 (376) 12.5 / 11.9, 256 15.5 / 16.2 (a second step on some
//                  compute units only, and ten blocks to bring in first: left on row tiles)   1 x 512, 128 (128) 9.7 / 9.7
//   64 / 8 x 128   1 x 8192, 128 (2048) 125 / 75    256  151 / 98     1 x 2048, 128 (512) 31 / 21   1 x 512, 128 (128) 11.4 / 11.9
//   32 / 8 x 128   2 x 4096, 128 (1024) 59 / 39     160   61 / 42
//   28 / 4 x 128   1 x 3000, 128 (332)  26 / 21     64 / 8 x 96, 1 x 4096, 128 (1024) 47 / 34
struct WindowRuns {
    uint32_t ring_blocks, runs, run_steps;
};

WindowRuns window_runs(const SingeFmhaPrefillConfig& c, uint64_t window) {
    constexpr uint64_t kStepRows = 32 * kWindowPrefillWaves, kLdsBytes = 160 * 1024;
    const uint64_t group = c.heads / c.kv_heads, row_bytes = c.head_dim <= 64 ? 128 : 256;
    // The kernel counts a batch entry's queries and output rows in 32 bits of bytes.
    const uint64_t query_reach = (c.query_len - 1) * c.query_sequence_stride + (c.heads - 1) * c.query_head_stride + c.head_dim;
    const uint64_t output_reach = (c.query_len - 1) * c.output_sequence_stride + (c.heads - 1) * c.output_head_stride + c.head_dim;
    if (query_reach > 0x7fffffffull || output_reach > 0x7fffffffull) return {0, 0, 0};
    // The keys from the first one that a step's first row sees to the last one that the next step's last row does, in blocks
    // of 32; where every step starts with a query that is a multiple of 32 the first key's place in its block is known.
    const bool whole = kStepRows % group == 0 && kStepRows / group % 32 == 0;
    const uint64_t keys = window + (whole ? 2 * kStepRows / group - 1 : (2 * kStepRows - 1 + group - 1) / group);
    const uint64_t ring = ((whole ? (32 - (window + 31) % 32) % 32 : 31) + keys - 1) / 32 + 1, bytes = ring * 64 * row_bytes;
    if (bytes > (c.head_dim <= 64 ? kLdsBytes / 2 : kLdsBytes)) return {0, 0, 0};
    const uint64_t units = compute_units(), places = units * (c.head_dim <= 64 ? 2 : 1);
    const uint64_t pairs = static_cast<uint64_t>(c.batch) * c.kv_heads, steps = (c.query_len * group + kStepRows - 1) / kStepRows, all = pairs * steps;
    if (2 * all <= units || (c.head_dim <= 64 && ring > 8 && all > units && 2 * all < 3 * units)) return {0, 0, 0};
    const uint64_t run_steps = window_run_steps(steps, pairs, places);
    return {static_cast<uint32_t>(ring), static_cast<uint32_t>((steps + run_steps - 1) / run_steps), static_cast<uint32_t>(run_steps)};
}

int32_t prefill(void* stream, uint16_t* out, size_t out_len, float* lse, size_t lse_len, bool with_lse,
                const uint16_t* query, size_t query_len, const uint16_t* key, size_t key_len, const uint16_t* value,
                size_t value_len, const SingeFmhaPrefillConfig* config, bool f16 = false, const DenseOptions& options = DenseOptions()) {
    if (config == nullptr) return fail(SINGE_HIP_NULL_POINTER, "config");
    const SingeFmhaPrefillConfig& c = *config;
    if (int32_t status = validate_call(c, out, out_len, lse, lse_len, with_lse, query, query_len, key, key_len, value, value_len))
        return status;

    // What the gfx950 kernel takes: head_dim 128 and rows it can fetch 16 bytes at a time.
    if (!has_matrix_core_build(static_cast<long long>(c.head_dim))) {
        // Other head dimensions (the reference's matrix path takes 16 and 32 too: fmha.rs:752-755) run on the
        // one-wave-per-row kernel, up to 256; without the dense op's options, which only reach here at 64 and 128.
        DenseGeneralOperands o;
        o.query = query, o.key = key, o.value = value, o.out = out, o.lse = with_lse ? lse : nullptr;
        o.query_strides[0] = c.query_batch_stride, o.query_strides[1] = c.query_head_stride, o.query_strides[2] = c.query_sequence_stride;
        o.key_strides[0] = c.key_batch_stride, o.key_strides[1] = c.key_head_stride, o.key_strides[2] = c.key_sequence_stride;
        o.value_strides[0] = c.value_batch_stride, o.value_strides[1] = c.value_head_stride, o.value_strides[2] = c.value_sequence_stride;
        o.out_strides[0] = c.output_batch_stride, o.out_strides[1] = c.output_head_stride, o.out_strides[2] = c.output_sequence_stride;
        o.batch = c.batch, o.heads = c.heads, o.kv_heads = c.kv_heads, o.query_len = c.query_len, o.key_len = c.key_len;
        o.head_dim = o.value_dim = c.head_dim;
        o.causal = c.causal != 0, o.scale = c.scale, o.scale_wide = c.scale;
        return dense_general(f16 ? SINGE_HIP_F16 : SINGE_HIP_BF16, stream, f16 ? "fmha_prefill_f16" : "fmha_prefill_bf16", o);
    }
    const size_t strides[] = {c.query_batch_stride, c.key_batch_stride, c.value_batch_stride, c.output_batch_stride,
                              c.query_sequence_stride, c.key_sequence_stride, c.value_sequence_stride,
                              c.output_sequence_stride, c.query_head_stride, c.key_head_stride,
                              c.value_head_stride, c.output_head_stride};
    for (size_t stride : strides)
        if (stride % 8 != 0) return fail(SINGE_HIP_UNSUPPORTED_CONFIGURATION, "strides must be multiples of 8 elements");
    const uintptr_t addresses[] = {reinterpret_cast<uintptr_t>(out), reinterpret_cast<uintptr_t>(query),
                                   reinterpret_cast<uintptr_t>(key), reinterpret_cast<uintptr_t>(value)};
    for (uintptr_t address : addresses)
        if (address % 16 != 0) return fail(SINGE_HIP_UNSUPPORTED_CONFIGURATION, "buffers must be 16-byte aligned");
    // The kernel addresses the keys of one (batch, head) slice with 32-bit byte offsets.
    const size_t widest = c.key_sequence_stride > c.value_sequence_stride ? c.key_sequence_stride : c.value_sequence_stride;
    size_t slice_bytes = 0;
    if (!checked_mul(c.key_len, widest, &slice_bytes) || !checked_mul(slice_bytes, 2, &slice_bytes) || slice_bytes > 0xffffffffull)
        return fail(SINGE_HIP_UNSUPPORTED_CONFIGURATION, "key_len * sequence stride beyond 4 GiB");
    PrefillArgs args;
    args.query = query;
    args.key = key;
    args.value = value;
    args.out = out;
    args.lse = with_lse ? lse : nullptr;
    args.query_batch_stride = c.query_batch_stride;
    args.query_sequence_stride = c.query_sequence_stride;
    args.query_head_stride = c.query_head_stride;
    args.key_batch_stride = c.key_batch_stride;
    args.key_sequence_stride = c.key_sequence_stride;
    args.key_head_stride = c.key_head_stride;
    args.value_batch_stride = c.value_batch_stride;
    args.value_sequence_stride = c.value_sequence_stride;
    args.value_head_stride = c.value_head_stride;
    args.output_batch_stride = c.output_batch_stride;
    args.output_sequence_stride = c.output_sequence_stride;
    args.output_head_stride = c.output_head_stride;
    args.batch = static_cast<uint32_t>(c.batch);
    args.query_len = static_cast<uint32_t>(c.query_len);
    args.key_len = static_cast<uint32_t>(c.key_len);
    args.heads = static_cast<uint32_t>(c.heads);
    args.kv_heads = static_cast<uint32_t>(c.kv_heads);
    constexpr size_t kTileRows = 32 * kDensePrefillWaves;
    args.query_tiles = static_cast<uint32_t>((c.query_len + kTileRows - 1) / kTileRows);
    args.scale_log2e = logit_factor(c.scale);
    args.sinks = options.sinks;
    args.key_lengths = options.key_lengths;
    // (a window of as many keys as there are queries hides none: key + window <= query has no solution)
    const long long window = options.window >= 0 && static_cast<unsigned long long>(options.window) >= c.query_len ? -1 : options.window;
    const bool with_options = options.mask != nullptr || window >= 0 || options.softcap != 0.0f;
    args.mask = options.mask;
    for (int i = 0; i < 4; ++i) args.mask_strides[i] = options.mask_strides[i];
    args.mask_packed = options.mask != nullptr && options.mask_strides[3] == 1 && options.mask_strides[0] % 4 == 0 &&
                               options.mask_strides[1] % 4 == 0 && options.mask_strides[2] % 4 == 0 &&
                               (reinterpret_cast<uintptr_t>(options.mask) & 7u) == 0
                           ? 1u : 0u;
    args.window = window;
    if (options.softcap != 0.0f) {
        args.cap_scale = std::fabs(c.scale / options.softcap);
        args.cap_log2e = std::fabs(options.softcap) * 1.4426950408889634074f;
    }
    // A decode step through the dense op (few query rows, grouped heads, no causal mask): the query heads of a kv head
    // share one tile, so its keys and values are fetched once.
    args.packed_heads = dense_prefill_packs_heads(c) ? 1u : 0u;
    const uint64_t rows = static_cast<uint64_t>(c.batch) * (args.packed_heads ? c.kv_heads : c.heads);
    const DenseShares shares = dense_prefill_shares(c);
    args.single_tiles = shares.single_tiles ? 1u : 0u;
    // Whole (batch, head)s to an XCD leave some of them with one more than others where those are no multiple of eight, and such an
    // XCD's compute units with a workgroup more: so every XCD gets an eighth of the tiles.  Batch entries of their own key counts
    // are dealt so only up to a tile a compute unit; up to three, long ones go by their lengths, and the rest by whole (batch,
    // head)s as they come (by length 16 x 8 heads x 300 takes 11.6 us, as they come 10.2; 16 x 12 x 1500 122 and 118).  us, whole
    // (batch, head)s / now, head_dim 64 where not said:
    //   no lengths   1 x 6 heads x 1500  20.4 / 18.0   3 x 6  36 / 19.4   7 x 6  42 / 32.7   8 x 6  42.6 / 42.8
    //                causal 1 x 28 / 4 x 4096 x 128 (two tiles a wave)  124 / 114   1 x 28 / 4 x 4096 x 96  104 / 100   3 x 28 / 4 x 1500 x 96,
    //                no mask  114 / 85   causal 2 x 32 / 8 x 2048 x 128  76 / 71 (query heads that share keys share an XCD's L2)
    //   lengths of half the keys to all of them   1 x 6 x 1500  16.8 / 14.9   3 x 6  29.4 / 19.5   4 x 6  28.7 / 25.8   5 x 6  29.2 / 26.4
    //                7 x 6  36.4 / 31.4   8 x 6  37.4 / 32.1   9 x 6  38.8 / 34.7   10 x 6  40.8 / 39.1   5 x 12 x 700  17.1 / 15.9
    const uint64_t units = rows * (shares.single_tiles ? args.query_tiles : (args.query_tiles + 1) / 2);
    // Single tiles under the causal mask, more of them than the compute units hold at once, go by whole (batch, head)s too: an eighth that
    // ends inside one ends on its first tiles, which are its longest and run on by themselves.  Whole / evenly
    //   45 heads x 1500 x 128  48.5 / 56.3   30 x 2560  73 / 81   20 x 6000 x 64  137 / 148   (all at once: 36 x 2560 x 64  53.6 / 51.8)
    const uint64_t at_once = compute_units() * (c.head_dim > 64 ? 2 : c.head_dim > 32 ? 3 : 4);
    args.deal = c.causal && args.single_tiles != 0 && units > at_once ? kDealWhole : kDealEvenly;
    if (options.key_lengths != nullptr && units > compute_units())
        args.deal = !c.causal && args.single_tiles != 0 && args.packed_heads == 0 && c.batch <= 64 && c.key_len >= 512 && units <= 3 * compute_units()
                        ? kDealByLength : kDealWhole;
    auto dealt = [&](uint64_t each) { return args.deal == kDealEvenly ? (rows * each + 7) / 8 * 8 : (rows + 7) / 8 * 8 * each; };  // workgroups, `each` to a row
    uint64_t groups = dealt(shares.single_tiles ? args.query_tiles : (args.query_tiles + 1) / 2);
    if (groups > 0x7fffffffull) return fail(SINGE_HIP_UNSUPPORTED_CONFIGURATION, "too many workgroups");
    // Key splits, when the caller lent scratch for them and the launch is too small to fill the chip.
    uint32_t splits = options.scratch != nullptr ? shares.splits : 1;
    // (the merge counts rows in 32 bits)
    if (splits > 1 && static_cast<uint64_t>(c.batch) * c.heads * c.query_len > 0xffffffffull) splits = 1;
    if (splits > 1 && (options.scratch_bytes < dense_prefill_scratch_bytes(c, splits) || groups * splits > 0x7fffffffull)) splits = 1;
    // Two sets of waves to a tile instead, each on one half of its keys, where a tile a compute unit is all there is and its
    // keys are worth it (and, up to half as many tiles, no more shares could be lent for; a caller's own split_below_blocks
    // that asks for shares gets them).  One set / two, us, f16 and bf16 alike:
    //   head_dim 128, causal  32 heads x 300 (96 tiles) 11.6 / 12.1   x 512 (128) 16.6 / 16.0   x 773 (224) 22.5 / 20.4   x 1024 (256) 27.9 / 24.3
    //                         x 1500 (384) 44.9 / 45.4                16 x 2048 (256) 46.7 / 36.9 (two shares 42)         8 x 4096 (256) 85.5 / 63.8
    //   head_dim 128, full    32 x 1024 (256) 29.1 / 26.1             32 x 1500 (384) 49.9 / 59.8  8 x 4096 (256) 89.3 / 76.4
    //   head_dim 64           causal 32 x 1024 (256) 19.8 / 16.6, 8 x 4096 (256) 60.6 / 43.4; full 64 x 512 (256) 12.9 / 11.6, 8 x 4096 63.1 / 47.8
    const uint64_t query_tiles = static_cast<uint64_t>(c.batch) * c.heads * args.query_tiles, seen = c.causal && c.query_len < c.key_len ? c.query_len : c.key_len;
    const bool halves = !with_options && args.packed_heads == 0 && args.single_tiles != 0 && query_tiles <= compute_units() && seen >= 512 &&
                        (splits == 1 || (2 * query_tiles > compute_units() && split_below_is_default()));
    if (halves) splits = 1;
    args.splits = splits;
    if (splits > 1) {
        const size_t row_count = static_cast<size_t>(c.batch) * c.heads * c.query_len;
        args.partial_out = static_cast<float*>(options.scratch);
        args.partial_lse = args.partial_out + static_cast<size_t>(splits) * row_count * c.head_dim;
        groups *= splits;
    }
    const long long head_dim = static_cast<long long>(c.head_dim);
    // Long rows without options: the kernel that gives a wave two 32-row tiles (256 query rows a
    // workgroup, one workgroup a compute unit), when its launch still fills the chip; a build of its own where the last
    // key tile is not whole.
    if (!with_options && splits == 1 && two_tiles_a_wave(c)) {
        const uint32_t pair_tiles = static_cast<uint32_t>((c.query_len + 255) / 256);
        args.query_tiles = pair_tiles;
        args.deal = options.key_lengths != nullptr ? kDealWhole : kDealEvenly;
        const uint64_t pair_groups = dealt((pair_tiles + 1) / 2);
        // (the builds that take a last tile that is not whole also take a key count of their own for every batch entry)
        const bool ragged = c.key_len % 64 != 0 || options.key_lengths != nullptr;
        const KernelId pair = static_cast<KernelId>(pair_kernels_at(static_cast<long long>(c.head_dim), false) + (c.causal ? 0 : 1) + (f16 ? 2 : 0) + (ragged ? 4 : 0));
        return launch(pair, static_cast<unsigned>(pair_groups), 1, 1, 256, stream, args);
    }
    // Under a causal window grouped heads share tiles: 128 rows are then 128 / group queries, whose windows overlap almost
    // whole, and a tile walks window + 128 / group keys instead of window + 128.  Not two heads under a window of three
    // quarters of the rows and more, where that saves next to nothing and a workgroup gives up the pair of a long and a short
    // tile.  Each head's own tiles / shared ones, us:
    //   64 / 8 heads x 64    1 x 8192, window 128   69 / 57    512  117 / 100   2048  319 / 282   4096  537 / 463   8191  623 / 608
    //   64 / 8 x 128         1 x 2048, window 128   39 / 32    512   57 / 50    1024   78 / 71    1536   79 / 77    2047   80 / 78
    //   32 / 8 x 128         8 x 4096, window 128  266 / 236   512  423 / 388   2048  928 / 865   3072 1061 / 1037  4095 1094 / 1094
    //   12 / 4 x 96          4 x 2048, window 128   29 / 25    512   40 / 38    1024   56 / 51    1536   66 / 52    2047   72 / 54
    //   32 / 16 x 64         2 x 2048, window 128   24 / 21    512   36 / 32    1024   49 / 43    1536   49 / 51    2047   50 / 52
    //   32 / 16 x 128        4 x 4096, window 128  139 / 130   1024 311 / 297   2048  478 / 440   3072  532 / 530   4095  549 / 558
    const uint64_t group = c.heads / c.kv_heads, packed_rows = static_cast<uint64_t>(c.query_len) * group;
    if (c.causal && window >= 0 && options.mask == nullptr && splits == 1 && group > 1 && args.packed_heads == 0 && packed_rows <= 0x7fffff00ull &&
        (group > 2 || 4 * static_cast<uint64_t>(window) < 3 * static_cast<uint64_t>(c.query_len))) {
        const WindowRuns run = options.softcap == 0.0f ? window_runs(c, static_cast<uint64_t>(window)) : WindowRuns{0, 0, 0};
        if (run.runs != 0) {
            args.ring_blocks = run.ring_blocks;
            args.query_tiles = run.runs;
            args.run_steps = run.run_steps;
            const uint64_t workgroups = (static_cast<uint64_t>(c.batch) * c.kv_heads * run.runs + 7) / 8 * 8;
            if (workgroups > 0x7fffffffull) return fail(SINGE_HIP_UNSUPPORTED_CONFIGURATION, "too many workgroups");
            return launch(static_cast<KernelId>(prefill_window_at(head_dim) + (f16 ? 1 : 0)), static_cast<unsigned>(workgroups), 1, 1,
                          64 * kWindowPrefillWaves, stream, args, run.ring_blocks * 64 * (c.head_dim <= 64 ? 128 : 256));
        }
        // (runs of eight tiles, whole rounds of the XCDs: see fmha_prefill_body)
        const uint64_t tiles = (packed_rows + kTileRows - 1) / kTileRows, runs = static_cast<uint64_t>(c.batch) * c.kv_heads * ((tiles + 7) / 8);
        if (runs <= 0x7fffff0ull) {
            args.packed_heads = 2;
            args.query_tiles = static_cast<uint32_t>(tiles);
            groups = (runs + 7) / 8 * 64;
        }
    }
    if (halves) {
        const int kernel = prefill_halves_at(head_dim) + (c.causal ? 0 : 1) + (f16 ? 2 : 0);
        return launch(static_cast<KernelId>(kernel), static_cast<unsigned>(groups), 1, 1, 128 * kDensePrefillWaves, stream, args);
    }
    const KernelId kernel = static_cast<KernelId>((f16 ? kPrefillCausalF16 : kPrefillCausal) + (c.causal ? 0 : 1) + (with_options ? 4 : 0));
    if (int32_t status = launch(at_head_dim(kernel, head_dim), static_cast<unsigned>(groups), 1, 1, 64 * kDensePrefillWaves, stream, args))
        return status;
    if (splits == 1) return 0;
    const uint64_t merge_rows = 4 * (64 / (c.head_dim / 4));  // of a workgroup (fmha_prefill_combine_body)
    const uint64_t merge_groups = (static_cast<uint64_t>(c.batch) * c.heads * c.query_len + merge_rows - 1) / merge_rows;
    if (merge_groups > 0x7fffffffull) return fail(SINGE_HIP_UNSUPPORTED_CONFIGURATION, "too many workgroups");
    const KernelId merge = static_cast<KernelId>(prefill_combine_at(head_dim) + (f16 ? 1 : 0));
    return launch(merge, static_cast<unsigned>(merge_groups), 1, 1, 256, stream, args);
}

}  // namespace

namespace singe_hip {

bool dense_prefill_packs_heads(const SingeFmhaPrefillConfig& c) {
    constexpr size_t kTileRows = 32 * kDensePrefillWaves;
    return !c.causal && c.kv_heads > 0 && c.heads > c.kv_heads && c.heads % c.kv_heads == 0 && c.query_len * (c.heads / c.kv_heads) <= kTileRows;
}

// One tile a workgroup where pairs would not fill the chip's two workgroups a compute unit.  Shares of the keys as
// attention_key_splits counts them where even single tiles leave half the compute units idle, and for a launch of one query
// tile a head (a decode step); none where there are more tiles than compute units; in between two, if the rows see so many
// keys that a workgroup's walk over them outweighs the merge: 1536 under the causal mask, whose last tile alone walks them
// all, 4096 without it.  (In between, one share took up to 1.3 times as long as pairs with their shares: 1 x 8 x 2500.)
// (Those two are for calls with a mask, a window or a cap: the others walk a tile's keys from two places at once instead, on
// two sets of waves, see `halves`, and leave the scratch alone.  The scratch is sized for both: a mask is the launch's, not the
// problem's.)
// Pairs, with the shares they were cut into before single tiles, against single tiles with 1 / 2 / 4 shares, us:
//   head_dim 128, causal    1 x 8 x 2500 (160 tiles)   46  54 / 42 / 35     1 x 16 x 2000 (256)  49  45 / 42 / 45
//                           1 x 20 x 1024 (160)        36  26 / 29 / 33     1 x 20 x 1536 (240)  46  38 / 36 / 44
//                           1 x 32 x 1024 (256)        38  27 / 32 / 40     1 x 24 x 2000 (384)  71  52 / 54 / 65
//   head_dim 96, causal     1 x 8 x 2500 (160)         39  51 / 39 / 31     1 x 12 x 2000 (192)  37  42 / 36 / 35
//   head_dim 64, causal     1 x 8 x 2500 (160)         36  39 / 30 / 26     1 x 16 x 2000 (256)  36  32 / 31 / 30
//   head_dim 128, queries x keys without a mask   64 heads x 512 x 2048 (256)   73  48 / 53 / 65
//                           64 x 512 x 16384   369  358 / 295 / 305         80 x 512 x 16384 (320) 507 428 / 448 / 408
//   head_dim 64, no mask    64 x 512 x 2048 (256)      49  33 / 33 / 39     20 x 1024 x 8192 (160) 111 114 / 77 / 70
// Pairs against single tiles with 1 / 2 / 3 / 4 shares, us with the host's part:
//   8 x 6 heads x 1500, head_dim 64, ragged keys       59 / 57 / 63        42 / 50 / 54 / 57
//   8 x 12 heads x 600, head_dim 64, ragged keys       29 / 33 / 38        17 / 32 / 34 / 39
//   1 x 32 heads x 773, head_dim 128, causal           31 / 32 / 34        23 / 30 / 34 / 35
//   1 x 32 heads x 2048, head_dim 128, causal          56 / 65 / 80        57 / 70 / 75 / 84
//   1 x 16 heads x 2000, head_dim 128, causal          52 / 44 / 47        45 / 42 / 42 / 46
//   1 x 8 heads x 2000, head_dim 64, causal            37 / 30 / 27        32 / 26 / 25 / 24
//   16 x 12 heads x 1500, head_dim 64, ragged keys    154 / 158 / 188     161 / 155 / 185 / 231
DenseShares dense_prefill_shares(const SingeFmhaPrefillConfig& c) {
    if (!has_matrix_core_build(static_cast<long long>(c.head_dim)) || c.batch == 0 || c.heads == 0 || c.query_len == 0) return {false, 1};
    constexpr size_t kTileRows = 32 * kDensePrefillWaves;
    const uint64_t query_tiles = (c.query_len + kTileRows - 1) / kTileRows, units = compute_units();
    const uint64_t rows = static_cast<uint64_t>(c.batch) * (dense_prefill_packs_heads(c) ? c.kv_heads : c.heads);
    uint64_t tiles = rows * query_tiles;
    uint32_t most = 0xffffffffu;
    const bool single = rows * ((query_tiles + 1) / 2) < 2 * units;
    if (query_tiles > 1 && 2 * tiles > units && tiles < 2 * units) {
        const uint64_t seen = c.causal && c.query_len < c.key_len ? c.query_len : c.key_len;
        if (tiles <= units && seen >= (c.causal ? 1536 : 4096)) most = 2;
        else tiles = 2 * units;  // (counts as a full chip)
    }
    const uint32_t splits = attention_key_splits(single ? tiles : rows * ((query_tiles + 1) / 2), c.key_len);
    return {single, splits < most ? splits : most};
}

uint32_t dense_prefill_splits(const SingeFmhaPrefillConfig& c) { return dense_prefill_shares(c).splits; }

size_t dense_prefill_scratch_bytes(const SingeFmhaPrefillConfig& c, uint32_t splits) {
    if (splits <= 1) return 0;
    return static_cast<size_t>(splits) * c.batch * c.heads * c.query_len * (c.head_dim + 1) * sizeof(float);
}

// The dense op's way into the matrix-core kernel: the public entry points' checks and launch, plus the op's options
// (general_attention.cpp).
bool dense_prefill_takes(const SingeFmhaPrefillConfig& c, const void* out, const void* query, const void* key, const void* value) {
    if (!has_matrix_core_build(static_cast<long long>(c.head_dim))) return false;
    const size_t strides[] = {c.query_batch_stride, c.key_batch_stride, c.value_batch_stride, c.output_batch_stride,
                              c.query_sequence_stride, c.key_sequence_stride, c.value_sequence_stride,
                              c.output_sequence_stride, c.query_head_stride, c.key_head_stride,
                              c.value_head_stride, c.output_head_stride};
    for (size_t stride : strides)
        if (stride % 8 != 0) return false;
    const uintptr_t addresses[] = {reinterpret_cast<uintptr_t>(out), reinterpret_cast<uintptr_t>(query),
                                   reinterpret_cast<uintptr_t>(key), reinterpret_cast<uintptr_t>(value)};
    for (uintptr_t address : addresses)
        if (address % 16 != 0) return false;
    const size_t widest = c.key_sequence_stride > c.value_sequence_stride ? c.key_sequence_stride : c.value_sequence_stride;
    size_t slice_bytes = 0;
    return checked_mul(c.key_len, widest, &slice_bytes) && checked_mul(slice_bytes, 2, &slice_bytes) && slice_bytes <= 0xffffffffull;
}

int32_t dense_prefill_with_options(void* stream, bool f16, uint16_t* out, size_t out_len, const uint16_t* query, size_t query_len,
                                   const uint16_t* key, size_t key_len, const uint16_t* value, size_t value_len,
                                   const SingeFmhaPrefillConfig* config, const DenseOptions& options) {
    return prefill(stream, out, out_len, nullptr, 0, false, query, query_len, key, key_len, value, value_len, config, f16, options);
}

}  // namespace singe_hip

extern "C" {

int32_t singe_hip_fmha_prefill_config_validate(const SingeFmhaPrefillConfig* config) {
    if (config == nullptr) return fail(SINGE_HIP_NULL_POINTER, "config");
    return validate_config(*config);
}

int32_t singe_hip_fmha_prefill_f32(void* stream, float* out, size_t out_len, const float* query, size_t query_len,
                                   const float* key, size_t key_len, const float* value, size_t value_len,
                                   const SingeFmhaPrefillConfig* config) {
    return prefill_f32(stream, out, out_len, nullptr, 0, false, query, query_len, key, key_len, value, value_len, config, 0,
                       false, 0.0f, "fmha_prefill_f32");
}

int32_t singe_hip_fmha_prefill_lse_f32(void* stream, float* out, size_t out_len, float* lse, size_t lse_len,
                                       const float* query, size_t query_len, const float* key, size_t key_len,
                                       const float* value, size_t value_len, const SingeFmhaPrefillConfig* config) {
    return prefill_f32(stream, out, out_len, lse, lse_len, true, query, query_len, key, key_len, value, value_len, config, 0,
                       false, 0.0f, "fmha_prefill_lse_f32");
}

int32_t singe_hip_softcapped_window_attention_f32(void* stream, float* out, size_t out_len, const float* query,
                                                  size_t query_len, const float* key, size_t key_len, const float* value,
                                                  size_t value_len, const SingeSoftcappedWindowAttentionConfig* config) {
    if (config == nullptr) return fail(SINGE_HIP_NULL_POINTER, "config");
    return prefill_f32(stream, out, out_len, nullptr, 0, false, query, query_len, key, key_len, value, value_len,
                       &config->attention, config->window_size, config->has_soft_cap != 0, config->soft_cap,
                       "softcapped_window_attention_f32");
}

int32_t singe_hip_fmha_prefill_bf16(void* stream, uint16_t* out, size_t out_len, const uint16_t* query, size_t query_len,
                                    const uint16_t* key, size_t key_len, const uint16_t* value, size_t value_len,
                                    const SingeFmhaPrefillConfig* config) {
    return prefill(stream, out, out_len, nullptr, 0, false, query, query_len, key, key_len, value, value_len, config);
}

int32_t singe_hip_fmha_prefill_lse_bf16(void* stream, uint16_t* out, size_t out_len, float* lse, size_t lse_len,
                                        const uint16_t* query, size_t query_len, const uint16_t* key, size_t key_len,
                                        const uint16_t* value, size_t value_len, const SingeFmhaPrefillConfig* config) {
    return prefill(stream, out, out_len, lse, lse_len, true, query, query_len, key, key_len, value, value_len, config);
}

// fmha_prefill_f16 / fmha_prefill_lse_f16 (fmha.rs): the same kernels on f16 operands.
int32_t singe_hip_fmha_prefill_f16(void* stream, uint16_t* out, size_t out_len, const uint16_t* query, size_t query_len,
                                   const uint16_t* key, size_t key_len, const uint16_t* value, size_t value_len,
                                   const SingeFmhaPrefillConfig* config) {
    return prefill(stream, out, out_len, nullptr, 0, false, query, query_len, key, key_len, value, value_len, config, true);
}

int32_t singe_hip_fmha_prefill_lse_f16(void* stream, uint16_t* out, size_t out_len, float* lse, size_t lse_len,
                                       const uint16_t* query, size_t query_len, const uint16_t* key, size_t key_len,
                                       const uint16_t* value, size_t value_len, const SingeFmhaPrefillConfig* config) {
    return prefill(stream, out, out_len, lse, lse_len, true, query, query_len, key, key_len, value, value_len, config, true);
}

}  // extern "C"

extern "C" void singe_hip_set_dense_prefill_rows_per_wave(uint32_t rows) { g_rows_per_wave.store(rows, std::memory_order_relaxed); }

extern "C" uint32_t singe_hip_dense_prefill_rows_per_wave(const SingeFmhaPrefillConfig* config) {
    if (config == nullptr) return 0;
    return has_matrix_core_build(static_cast<long long>(config->head_dim)) ? (two_tiles_a_wave(*config) ? 64u : 32u) : 0u;
}
