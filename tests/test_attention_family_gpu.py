"""The rest of the singe-kernel dense family on the GPU, through the C ABI, against the CPU oracle on the same seeded inputs:
softcapped_window_attention_{bf16,f16}, attention_sink_prefill_{f32,bf16,f16}, fmha_decode_lse_*, softcapped_window_decode_lse_*,
ragged_kv_prefill_attention_* and the sliding-window attention over dense, packed and block-table keys.  f32 within 1e-4,
bf16 within max-abs 2e-2 / mean-abs 2e-3, f16 within 5e-3 / 5e-4 (outputs; log-sum-exps within 1e-4 / 2e-2 / 5e-3)."""
import numpy as np
import pytest
import torch

import oracle
from singe_amd import _native, error
from singe_amd.kernel import attention as A

pytestmark = pytest.mark.gpu

DTYPES = [torch.float32, torch.bfloat16, torch.float16]
BOUND = {torch.float32: (1e-4, 1e-4), torch.bfloat16: (2e-2, 2e-3), torch.float16: (5e-3, 5e-4)}


def close(got, want, dtype, what=""):
    got, want = got.float().cpu().numpy(), np.asarray(want, dtype=np.float32)
    assert np.isfinite(got).all(), what
    gap = np.abs(got - want)
    worst, mean = BOUND[dtype]
    assert gap.max(initial=0.0) <= worst and (gap.size == 0 or gap.mean() <= mean), (what, gap.max(), gap.mean())


def normal(shape, dtype, seed):
    generator = torch.Generator().manual_seed(seed)
    return torch.randn(shape, generator=generator).to(dtype).cuda()


def host(tensor):
    return tensor.float().cpu().numpy()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("head_dim,causal,window,cap", [
    (128, True, 0, 5.0), (128, True, 40, None), (128, True, 33, 2.5), (128, False, 17, None), (64, False, 50, 4.0),
    (128, False, 0, None), (40, True, 9, 3.0), (256, False, 6, None)])
def test_softcapped_window_attention_16_bit(dtype, head_dim, causal, window, cap):
    batch, heads, kv_heads, query_len, key_len = 2, 4, 2, 150, 150
    q = normal((batch, heads, query_len, head_dim), dtype, 1)
    k = normal((batch, kv_heads, key_len, head_dim), dtype, 2)
    v = normal((batch, kv_heads, key_len, head_dim), dtype, 3)
    out = torch.full_like(q, float("nan"))
    scale = head_dim ** -0.5
    config = A.SoftcappedWindowAttentionConfig(A.bhsd_config(batch, heads, kv_heads, query_len, key_len, head_dim, scale, causal), window, cap)
    run = A.softcapped_window_attention_bf16 if dtype == torch.bfloat16 else A.softcapped_window_attention_f16
    run(None, out, q, k, v, config)
    torch.cuda.synchronize()
    want = oracle.softcapped_window_attention_f32(host(q), host(k), host(v), batch=batch, query_len=query_len, key_len=key_len, heads=heads,
                                                  kv_heads=kv_heads, head_dim=head_dim, scale=scale, causal=causal, window_size=window,
                                                  soft_cap=cap, threads=8)
    close(out, want, dtype)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("head_dim,query_len,key_len,start_q,window,causal", [
    (64, 40, 40, 0, 0, True), (128, 130, 130, 0, 0, True), (128, 70, 200, 130, 0, True), (128, 70, 200, 130, 25, True),
    (32, 9, 50, 3, 4, False), (128, 160, 160, 0, 30, True), (96, 5, 5, 0, 1, True), (128, 3, 64, 200, 16, True)])
def test_attention_sink_prefill(dtype, head_dim, query_len, key_len, start_q, window, causal):
    batch, heads, kv_heads = 2, 4, 2
    q = normal((batch, query_len, heads, head_dim), dtype, 4)
    k = normal((batch, key_len, kv_heads, head_dim), dtype, 5)
    v = normal((batch, key_len, kv_heads, head_dim), dtype, 6)
    sinks = (normal((heads,), torch.float32, 7) * 3).to(dtype)
    out = torch.full_like(q, float("nan"))
    scale = head_dim ** -0.5
    config = A.AttentionSinkPrefillConfig.contiguous(batch, query_len, key_len, heads, kv_heads, head_dim, start_q, window, scale, causal)
    {torch.float32: A.attention_sink_prefill_f32, torch.bfloat16: A.attention_sink_prefill_bf16,
     torch.float16: A.attention_sink_prefill_f16}[dtype](None, out, q, k, v, sinks, config)
    torch.cuda.synchronize()
    want = oracle.attention_sink_prefill_f32(host(q), host(k), host(v), host(sinks), start_q=start_q, window=window, scale=scale, causal=causal)
    close(out, want, dtype)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("head_dim,key_len,heads,kv_heads", [(128, 300, 8, 2), (64, 1, 4, 4), (80, 77, 6, 3), (256, 40, 2, 1)])
def test_fmha_decode_lse(dtype, head_dim, key_len, heads, kv_heads):
    batch = 3
    q = normal((batch, heads, head_dim), dtype, 8)
    k = normal((batch, key_len, kv_heads, head_dim), dtype, 9)
    v = normal((batch, key_len, kv_heads, head_dim), dtype, 10)
    out = torch.full_like(q, float("nan"))
    lse = torch.full((batch, heads), float("nan"), device="cuda")
    scale = head_dim ** -0.5
    config = A.FmhaDecodeConfig.contiguous(batch, key_len, heads, kv_heads, head_dim, scale)
    {torch.float32: A.fmha_decode_lse_f32, torch.bfloat16: A.fmha_decode_lse_bf16, torch.float16: A.fmha_decode_lse_f16}[dtype](
        None, out, lse, q, k, v, config)
    torch.cuda.synchronize()
    want, want_lse = oracle.fmha_prefill_lse_f32(host(q)[:, None], host(k), host(v), batch=batch, query_len=1, key_len=key_len, heads=heads,
                                                 kv_heads=kv_heads, head_dim=head_dim, scale=scale, causal=False)
    close(out, want[:, 0], dtype)
    assert np.abs(lse.cpu().numpy() - want_lse[:, :, 0]).max() <= {torch.float32: 1e-4, torch.bfloat16: 2e-2, torch.float16: 5e-3}[dtype]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("head_dim,key_len,window,cap", [(128, 500, 0, None), (128, 500, 64, None), (64, 90, 1, 2.0), (128, 33, 200, 0.5),
                                                          (48, 129, 128, 6.0)])
def test_softcapped_window_decode_lse(dtype, head_dim, key_len, window, cap):
    batch, heads, kv_heads = 2, 8, 2
    q = normal((batch, heads, head_dim), dtype, 11)
    k = normal((batch, kv_heads, key_len, head_dim), dtype, 12)
    v = normal((batch, kv_heads, key_len, head_dim), dtype, 13)
    out = torch.full_like(q, float("nan"))
    lse = torch.full((batch, heads), float("nan"), device="cuda")
    scale = head_dim ** -0.5
    config = A.SoftcappedWindowDecodeConfig.bnsd_contiguous(batch, key_len, heads, kv_heads, head_dim, scale, window, cap)
    {torch.float32: A.softcapped_window_decode_lse_f32, torch.bfloat16: A.softcapped_window_decode_lse_bf16,
     torch.float16: A.softcapped_window_decode_lse_f16}[dtype](None, out, lse, q, k, v, config)
    torch.cuda.synchronize()
    want, want_lse = oracle.softcapped_window_decode_lse_f32(host(q), host(k), host(v), scale=scale, window_size=window, soft_cap=cap)
    close(out, want, dtype)
    assert np.abs(lse.cpu().numpy() - want_lse).max() <= {torch.float32: 1e-4, torch.bfloat16: 2e-2, torch.float16: 5e-3}[dtype]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("head_dim,heads,kv_heads", [(128, 4, 2), (64, 6, 6), (24, 2, 1)])
def test_ragged_kv_prefill(dtype, causal, head_dim, heads, kv_heads):
    lens_q = [5, 0, 130, 3, 70, 2]
    lens_kv = [5, 9, 200, 0, 70, 1]
    offsets = [0, 5, 14, 214, 217, 287]   # sequence 3 has queries and no keys; tokens 289 .. 291 belong to no sequence
    tokens, kv_tokens = 292, 289
    q = normal((tokens, heads, head_dim), dtype, 14)
    k = normal((kv_tokens, kv_heads, head_dim), dtype, 15)
    v = normal((kv_tokens, kv_heads, head_dim), dtype, 16)
    out = torch.full_like(q, 7.0)
    lse = torch.full((tokens, heads), 7.0, device="cuda")
    scale = head_dim ** -0.5
    config = A.RaggedKvPrefillAttentionConfig.contiguous(len(lens_q), tokens, kv_tokens, heads, kv_heads, head_dim, causal, scale)
    index = lambda values: torch.tensor(values, dtype=torch.int32, device="cuda")
    {torch.float32: A.ragged_kv_prefill_attention_f32, torch.bfloat16: A.ragged_kv_prefill_attention_bf16,
     torch.float16: A.ragged_kv_prefill_attention_f16}[dtype](None, out, lse, q, k, v, index(lens_q), index(lens_kv), index(offsets), config)
    torch.cuda.synchronize()
    want, want_lse = oracle.ragged_kv_prefill_attention_f32(host(q), host(k), host(v), lens_q, lens_kv, offsets, causal=causal, scale=scale)
    owned = np.zeros(tokens, dtype=bool)
    for offset, count in zip(offsets, lens_q):
        owned[offset:offset + count] = True
    close(out[torch.from_numpy(owned).cuda()], want[owned], dtype)
    got_lse = lse.cpu().numpy()
    empty = want_lse == np.float32(-1e20)
    assert (got_lse[empty & owned[:, None]] == np.float32(-1e20)).all()
    live = owned[:, None] & ~empty
    assert np.abs(got_lse[live] - want_lse[live]).max() <= {torch.float32: 1e-4, torch.bfloat16: 2e-2, torch.float16: 5e-3}[dtype]
    assert (out[~torch.from_numpy(owned).cuda()].float() == 7.0).all() and (got_lse[~owned] == 7.0).all()  # left alone


@pytest.mark.parametrize("head_dim,query_len,key_len,query_start,key_start,window,output_scale", [
    (64, 20, 60, 40, 0, 8, 1.0), (128, 33, 33, 0, 0, 1, 1.0), (32, 7, 90, 100, 20, 500, 0.25), (16, 5, 12, 0, 30, 4, 1.0),
    (200, 9, 40, 31, 0, 16, 2.0)])
def test_sliding_window_attention_dense_packed_and_paged(head_dim, query_len, key_len, query_start, key_start, window, output_scale):
    batch, heads, kv_heads, block = 2, 4, 2, 8
    q = normal((batch, query_len, heads, head_dim), torch.float32, 17)
    k = normal((batch, key_len, kv_heads, head_dim), torch.float32, 18)
    v = normal((batch, key_len, kv_heads, head_dim), torch.float32, 19)
    scale = head_dim ** -0.5
    config = A.SlidingWindowAttentionConfig.contiguous(batch, query_len, key_len, heads, kv_heads, head_dim, query_start, key_start, window,
                                                       scale).with_output_scale(output_scale)
    want = oracle.sliding_window_attention_f32(host(q), host(k), host(v), batch=batch, query_len=query_len, key_len=key_len, heads=heads,
                                               kv_heads=kv_heads, head_dim=head_dim, query_start=query_start, key_start=key_start,
                                               window=window, scale=scale, output_scale=output_scale).reshape(q.shape)
    out = torch.full_like(q, float("nan"))
    A.sliding_window_attention_f32(None, out, q, k, v, config)
    torch.cuda.synchronize()
    close(out, want, torch.float32, "dense")

    packed = torch.cat([torch.zeros(5, device="cuda"), q.flatten(), k.flatten(), torch.zeros(3, device="cuda"), v.flatten()])
    out.fill_(float("nan"))
    A.sliding_window_attention_packed_qkv_f32(None, out, packed, A.PackedQkvAttentionConfig(config, 5, 5 + q.numel(), 8 + q.numel() + k.numel()))
    torch.cuda.synchronize()
    close(out, want, torch.float32, "packed")

    blocks_per = (key_len + block - 1) // block
    physical = batch * blocks_per + 3
    table = torch.from_numpy(np.random.default_rng(5).permutation(physical)[: batch * blocks_per].reshape(batch, blocks_per).astype(np.int32)).cuda()
    key_cache = torch.randn((physical, block, kv_heads, head_dim), device="cuda")
    value_cache = torch.randn((physical, block, kv_heads, head_dim), device="cuda")
    for b in range(batch):
        for j in range(key_len):
            key_cache[table[b, j // block], j % block] = k[b, j]
            value_cache[table[b, j // block], j % block] = v[b, j]
    kv_features = kv_heads * head_dim
    paged = A.PagedKvAttentionConfig(config, block, physical, blocks_per, block * kv_features, block * kv_features)
    out.fill_(float("nan"))
    A.sliding_window_attention_paged_kv_f32(None, out, q, key_cache, value_cache, table, paged)
    torch.cuda.synchronize()
    close(out, want, torch.float32, "paged")
    # A block id outside the cache hides its keys (the reference kernel's block_valid test).
    broken = table.clone()
    broken[0, 0] = physical + 9
    out.fill_(float("nan"))
    A.sliding_window_attention_paged_kv_f32(None, out, q, key_cache, value_cache, broken, paged)
    torch.cuda.synchronize()
    want_broken = oracle.sliding_window_attention_paged_kv_f32(host(q), host(key_cache), host(value_cache), broken.cpu().numpy().view(np.uint32),
                                                               key_len=key_len, query_start=query_start, key_start=key_start, window=window,
                                                               scale=scale, output_scale=output_scale)
    close(out, want_broken, torch.float32, "paged, one block outside the cache")


def test_family_validation_on_the_device():
    q = torch.zeros((1, 4, 2, 64), device="cuda")
    config = A.SlidingWindowAttentionConfig.contiguous(1, 4, 4, 2, 2, 64, 0, 0, 0, 0.1)   # window 0
    with pytest.raises(error.InvalidLength):
        A.sliding_window_attention_f32(None, q, q, q, q, config)
    good = A.SlidingWindowAttentionConfig.contiguous(1, 4, 4, 2, 2, 64, 0, 0, 2, 0.1)
    with pytest.raises(error.LengthTooShort) as caught:
        A.sliding_window_attention_f32(None, q, q, q[:, :3].contiguous(), q, good)
    assert caught.value.name == "key"
    capped = A.SoftcappedWindowDecodeConfig.bnsd_contiguous(1, 4, 2, 2, 64, 0.1, 2, -1.0)   # a cap must be positive
    lse = torch.zeros((1, 2), device="cuda")
    with pytest.raises(error.InvalidLength):
        A.softcapped_window_decode_lse_f32(None, q[:, 0].contiguous(), lse, q[:, 0].contiguous(), q, q, capped)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("head_dim", [128, 96, 80, 64, 16])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("heads,kv_heads,lens", [
    (8, 2, [1, 63, 64, 65, 16, 33]),                    # 128-row tiles: ends of key tiles and of sixteen-key groups
    (3, 1, [1] * 70 + [130, 2]),                        # more than 64 sequences, rows that no power of two divides
    (32, 16, [255, 257, 300, 1, 128, 511, 640]),        # MHA-like: two heads a kv head
    (64, 64, [1537]),                                   # one row past a tile
])
def test_packed_prefill_on_the_matrix_cores(dtype, head_dim, causal, heads, kv_heads, lens):
    tokens = sum(lens)
    offsets = np.concatenate([[0], np.cumsum(lens)[:-1]])
    q, k, v = (normal((tokens, h, head_dim), dtype, seed) for h, seed in ((heads, 20), (kv_heads, 21), (kv_heads, 22)))
    out = torch.full_like(q, float("nan"))
    lse = torch.full((tokens, heads), float("nan"), device="cuda")
    scale = head_dim ** -0.5
    config = A.RaggedKvPrefillAttentionConfig.contiguous(len(lens), tokens, tokens, heads, kv_heads, head_dim, causal, scale)
    index = lambda values: torch.tensor(np.asarray(values), dtype=torch.int32, device="cuda")
    call = A.ragged_kv_prefill_attention_bf16 if dtype == torch.bfloat16 else A.ragged_kv_prefill_attention_f16
    call(None, out, lse, q, k, v, index(lens), index(lens), index(offsets), config)
    torch.cuda.synchronize()
    # (the oracle runs on one thread: the first and the last kv head, with their query heads)
    group = heads // kv_heads
    for kv_head in {0, kv_heads - 1}:
        of = slice(kv_head * group, (kv_head + 1) * group)
        want, want_lse = oracle.ragged_kv_prefill_attention_f32(host(q)[:, of], host(k)[:, kv_head:kv_head + 1], host(v)[:, kv_head:kv_head + 1],
                                                                lens, lens, offsets, causal=causal, scale=scale)
        close(out[:, of], want, dtype)
        assert np.abs(lse.cpu().numpy()[:, of] - want_lse).max() <= {torch.bfloat16: 2e-2, torch.float16: 5e-3}[dtype]


@pytest.mark.parametrize("kv_heads", [1, 16])
@pytest.mark.parametrize("rows_per_wave", [32, 64])      # (the paged op's choice of tiles, which packed sequences do not share)
def test_packed_sequences_that_overlap_leave_the_last_owner(kv_heads, rows_per_wave):
    # Three sequences over the same tokens: more row tiles than the token count says, and the last owner's rows stand.
    heads, head_dim, tokens = kv_heads * 2, 64, 2100
    lens, keys, offsets = [2100, 1500, 700], [900, 40, 700], [0, 300, 1200]
    q, k, v = (normal((tokens, h, head_dim), torch.bfloat16, seed) for h, seed in ((heads, 23), (kv_heads, 24), (kv_heads, 25)))
    out = torch.full_like(q, float("nan"))
    lse = torch.full((tokens, heads), float("nan"), device="cuda")
    config = A.RaggedKvPrefillAttentionConfig.contiguous(3, tokens, tokens, heads, kv_heads, head_dim, False, 0.125)
    index = lambda values: torch.tensor(values, dtype=torch.int32, device="cuda")
    _native.lib().singe_hip_set_paged_attention_rows_per_wave(rows_per_wave)
    try:
        A.ragged_kv_prefill_attention_bf16(None, out, lse, q, k, v, index(lens), index(keys), index(offsets), config)
        torch.cuda.synchronize()
    finally:
        _native.lib().singe_hip_set_paged_attention_rows_per_wave(0)
    for of in {0, kv_heads - 1}:
        heads_of, kv_of = slice(2 * of, 2 * of + 2), slice(of, of + 1)
        want, want_lse = oracle.ragged_kv_prefill_attention_f32(host(q)[:, heads_of], host(k)[:, kv_of], host(v)[:, kv_of], lens, keys, offsets,
                                                                causal=False, scale=0.125)
        close(out[:, heads_of], want, torch.bfloat16)
        assert np.abs(lse.cpu().numpy()[:, heads_of] - want_lse).max() <= 1e-4   # an f32 sum, the same keys on both sides


def packed_reference_f64(q, k, v, lens, causal, scale):
    """ragged_kv_prefill_attention of non-overlapping sequences in float64 on the CPU: (out, natural-log lse)."""
    q, k, v = (x.double().cpu() for x in (q, k, v))
    group, at = q.shape[1] // k.shape[1], 0
    out, lse = torch.zeros_like(q), torch.zeros(q.shape[:2], dtype=torch.float64)
    for n in lens:
        of = slice(at, at + n)
        rows, keys, values = (x[of].transpose(0, 1) for x in (q, k.repeat_interleave(group, 1), v.repeat_interleave(group, 1)))
        scores = rows @ keys.transpose(1, 2).contiguous() * scale
        if causal:
            scores = scores.masked_fill(torch.arange(n)[None, :] > torch.arange(n)[:, None], -float("inf"))
        lse[of] = torch.logsumexp(scores, -1).transpose(0, 1)
        out[of] = (torch.softmax(scores, -1) @ values).transpose(0, 1)
        at += n
    return out, lse


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("head_dim", [128, 80, 16])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("steepness,mean", [(1.0, 0.0), (8.0, 0.0), (3.0, 1.0)])   # flat to steep weights, values with a mean
def test_packed_prefill_weighs_values_in_f32(dtype, head_dim, causal, steepness, mean):
    # The weights reach the values with f32's precision, so that the output's own rounding is all the error there is:
    # 16-bit weights, rounded as coarsely as the output, would make it about 1.4 times as large.
    lens, heads, kv_heads = [1, 33, 64, 130, 700], 4, 2
    tokens = sum(lens)
    q, k, v = (normal((tokens, h, head_dim), dtype, seed) for h, seed in ((heads, 30), (kv_heads, 31), (kv_heads, 32)))
    v = v + mean
    out = torch.full_like(q, float("nan"))
    lse = torch.full((tokens, heads), float("nan"), device="cuda")
    scale = steepness * head_dim ** -0.5
    config = A.RaggedKvPrefillAttentionConfig.contiguous(len(lens), tokens, tokens, heads, kv_heads, head_dim, causal, scale)
    index = lambda values: torch.tensor(np.asarray(values), dtype=torch.int32, device="cuda")
    call = A.ragged_kv_prefill_attention_bf16 if dtype == torch.bfloat16 else A.ragged_kv_prefill_attention_f16
    call(None, out, lse, q, k, v, index(lens), index(lens), index(np.concatenate([[0], np.cumsum(lens)[:-1]])), config)
    want, want_lse = packed_reference_f64(q, k, v, lens, causal, scale)
    error, rounding = (out.double().cpu() - want).norm().item(), (want.to(dtype).double() - want).norm().item()
    assert error <= 1.03 * rounding, (error, rounding)
    # a score is head_dim products (absolute values of 0.64 on average, less than 1 in any row here) summed in f32
    assert (lse.double().cpu() - want_lse).abs().max().item() <= head_dim * 2.0**-24 * head_dim * scale + 1e-5


def test_packed_prefill_rounds_the_log_sum_exp_once():
    # Relative to the norm, against float64: 4.4e-8 on the one-wave-per-row kernel, 4.8e-8 when the sum of the reference point
    # and the logarithm was rounded before it was scaled to natural units.
    lens, heads, kv_heads, head_dim = [64, 500, 1100], 8, 2, 128
    tokens = sum(lens)
    q, k, v = (normal((tokens, h, head_dim), torch.bfloat16, seed) for h, seed in ((heads, 40), (kv_heads, 41), (kv_heads, 42)))
    out, lse = torch.empty_like(q), torch.empty((tokens, heads), device="cuda")
    config = A.RaggedKvPrefillAttentionConfig.contiguous(len(lens), tokens, tokens, heads, kv_heads, head_dim, True, head_dim ** -0.5)
    index = lambda values: torch.tensor(values, dtype=torch.int32, device="cuda")
    A.ragged_kv_prefill_attention_bf16(None, out, lse, q, k, v, index(lens), index(lens), index([0, 64, 564]), config)
    _, want = packed_reference_f64(q, k, v, lens, True, head_dim ** -0.5)
    assert ((lse.double().cpu() - want).norm() / want.norm()).item() <= 4.6e-8
