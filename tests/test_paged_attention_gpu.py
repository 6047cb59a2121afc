"""The singe paged-attention op (FlashInfer form, bottom-right causal) on the GPU against the CPU oracle
(attend_paged restated), through the C ABI.  bf16 outputs within max-abs 2e-2 / mean-abs 2e-3, base-two
LSE within 2e-3; the paging error contract bit for bit."""
import ctypes

import numpy as np
import pytest
import torch

import oracle
from singe_amd import _native, error, neural

pytestmark = pytest.mark.gpu

MAX_ABS, MEAN_ABS, LSE_ABS = 2e-2, 2e-3, 2e-3


def layout(sequences, page_size, extra_pages=3):
    query_offsets, page_offsets, last, needed = [0], [0], [], 0
    for queries, keys in sequences:
        query_offsets.append(query_offsets[-1] + queries)
        pages = (keys + page_size - 1) // page_size
        needed += pages
        page_offsets.append(needed)
        last.append(0 if keys == 0 else keys - (pages - 1) * page_size)
    page_count = needed + extra_pages
    table = [(p * 7 + 2) % page_count for p in range(needed)] if np.gcd(7, page_count) == 1 else \
        list(np.random.default_rng(page_count).permutation(page_count)[:needed])
    return query_offsets, page_offsets, table, last, page_count


def run_case(sequences, heads, kv_heads, page_size, options, index_dtype=torch.int32, seed=0, dim=128, dtype=torch.bfloat16):
    query_offsets, page_offsets, table, last, page_count = layout(sequences, page_size)
    tokens = query_offsets[-1]
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    q = torch.randn((tokens, heads, dim), generator=gen, device="cuda").to(dtype)
    kc = torch.randn((page_count, page_size, kv_heads, dim), generator=gen, device="cuda").to(dtype)
    vc = torch.randn((page_count, page_size, kv_heads, dim), generator=gen, device="cuda").to(dtype)
    index = lambda values: torch.tensor(values, dtype=index_dtype, device="cuda")
    paging = neural.Paging(index(query_offsets), index(page_offsets), index(table), index(last))
    out, lse = neural.paged_attention(q, kc, vc, paging, options)
    torch.cuda.synchronize()
    status, want, want_lse = oracle.paged_attention_f32(
        q.float().cpu().numpy(), kc.float().cpu().numpy(), vc.float().cpu().numpy(), query_offsets, page_offsets, table,
        last, scale=options.scale, causal=options.causal, window=options.window, softcap=options.softcap, threads=8)
    assert status == 0
    got, got_lse = out.float().cpu().numpy(), lse.cpu().numpy()
    assert np.isfinite(got).all()
    gap = np.abs(got - want)
    assert gap.max() <= MAX_ABS, gap.max()
    assert gap.mean() <= MEAN_ABS, gap.mean()
    empty = np.isneginf(want_lse)
    assert np.array_equal(np.isneginf(got_lse), empty)
    assert not got[empty].any()
    assert np.abs(got_lse[~empty] - want_lse[~empty]).max(initial=0.0) <= LSE_ABS


OPTIONS = [neural.AttentionOptions(), neural.AttentionOptions(causal=True),
           neural.AttentionOptions(causal=True, window=16, softcap=30.0),
           neural.AttentionOptions(causal=True, window=100), neural.AttentionOptions(scale=0.05, softcap=5.0)]


@pytest.mark.parametrize("options", OPTIONS)
@pytest.mark.parametrize("heads,kv_heads,page_size", [(8, 2, 1), (8, 1, 16), (4, 4, 7), (64, 8, 16), (8, 2, 8), (8, 2, 32),
                                                      (4, 1, 64), (8, 2, 128), (6, 3, 48)])
def test_ragged_sequences_match_oracle(heads, kv_heads, page_size, options):
    # decode, full prefill, chunked prefill, no keys (kernel_plan/source/tests.rs:830-889), plus more
    # queries than keys, where the CPU path's saturating position applies
    sequences = [(1, 150), (70, 70), (20, 90), (3, 0), (9, 4), (130, 300)]
    run_case(sequences, heads, kv_heads, page_size, options, seed=heads + page_size)


@pytest.mark.parametrize("index_dtype", [torch.int32, torch.int64])
@pytest.mark.parametrize("heads,kv_heads,page_size,splits", [(8, 2, 16, 0), (4, 4, 16, 0), (16, 1, 8, 3)])
def test_many_ragged_sequences_find_their_row_tiles(heads, kv_heads, page_size, splits, index_dtype):
    # more sequences than one wave's prefix sum covers (64), some without queries, some without keys, query
    # counts from under one row tile to several
    rng = np.random.default_rng(heads * 31 + page_size)
    sequences = []
    for s in range(150):
        queries = int(rng.choice([0, 1, 1, 2, 5, 17, 31, 32, 33, 64, 100, 129, 200]))
        keys = 0 if s % 23 == 7 else queries + int(rng.integers(0, 120))
        sequences.append((queries, keys))
    _native.lib().singe_hip_set_paged_attention_splits(splits)
    try:
        run_case(sequences, heads, kv_heads, page_size, neural.AttentionOptions(causal=True), index_dtype=index_dtype, seed=heads)
        run_case(sequences[:70], heads, kv_heads, page_size, neural.AttentionOptions(window=40, causal=True), index_dtype=index_dtype, seed=3)
    finally:
        _native.lib().singe_hip_set_paged_attention_splits(0)


@pytest.mark.parametrize("index_dtype", [torch.int32, torch.int64])
@pytest.mark.parametrize("heads,kv_heads,page_size,splits", [(8, 2, 16, 0), (16, 1, 8, 2), (4, 4, 3, 0)])
def test_up_to_64_sequences_with_tiles_to_spare_are_taken_longest_first(heads, kv_heads, page_size, splits, index_dtype):
    # few sequences with several row tiles each: the grid lists them by pages held, longest first, ties by index;
    # equal lengths, sequences without queries or without keys, and one much longer than the rest
    groups = heads // kv_heads
    base = 128 // groups  # queries of one row tile
    sequences = [(3 * base, 700), (3 * base, 700), (0, 300), (5 * base + 1, 5 * base + 1), (2 * base, 0), (base, 2000),
                 (4 * base, 700), (1, 64), (6 * base, 1100), (2 * base + 7, 333)]
    assert sum(q for q, _ in sequences) * groups // 128 >= 2 * len(sequences)
    _native.lib().singe_hip_set_paged_attention_splits(splits)
    try:
        run_case(sequences, heads, kv_heads, page_size, neural.AttentionOptions(causal=True), index_dtype=index_dtype, seed=heads + 9)
        run_case(sequences[::-1], heads, kv_heads, page_size, neural.AttentionOptions(causal=True, window=90), index_dtype=index_dtype, seed=2)
        run_case(sequences * 6, heads, kv_heads, page_size, neural.AttentionOptions(causal=True), index_dtype=index_dtype, seed=5)  # 60 of them
    finally:
        _native.lib().singe_hip_set_paged_attention_splits(0)


@pytest.mark.parametrize("options", [neural.AttentionOptions(causal=True, softcap=-4.0), neural.AttentionOptions(scale=-0.06, softcap=5.0),
                                     neural.AttentionOptions(scale=-0.06, softcap=-5.0, causal=True, window=50)])
@pytest.mark.parametrize("heads,kv_heads,page_size", [(8, 2, 16), (4, 4, 7)])
def test_negative_caps_and_scales(heads, kv_heads, page_size, options):
    # cap * tanh(score / cap) does not care about the sign of the cap; a negative scale turns the scores round
    run_case([(1, 150), (70, 70), (20, 90)], heads, kv_heads, page_size, options, seed=heads)


@pytest.mark.parametrize("options", [neural.AttentionOptions(causal=True, window=300), neural.AttentionOptions(causal=True, window=200, softcap=8.0),
                                     neural.AttentionOptions(causal=True, window=64), neural.AttentionOptions(causal=True, softcap=6.0),
                                     neural.AttentionOptions(window=500), neural.AttentionOptions(softcap=3.0, scale=-0.05)])
@pytest.mark.parametrize("heads,kv_heads,page_size", [(8, 2, 16), (4, 4, 16), (16, 1, 5)])
def test_long_windows_and_caps(heads, kv_heads, page_size, options):
    """Sequences long enough that a wave meets tiles reaching back past the window, tiles wholly inside it (which,
    like the capped ones, take the straight-line path) and tiles on the causal edge."""
    run_case([(300, 1100), (700, 700), (1, 1300), (40, 64)], heads, kv_heads, page_size, options, seed=heads + 3)


def test_int64_indices_and_chunked_prefill_shape():
    # one sequence of the chunked-prefill shape: 512 new queries over a cached prefix, 64 query / 8 kv heads
    run_case([(512, 1536 + 512), (512, 1024 + 512)], 64, 8, 16, neural.AttentionOptions(causal=True),
             index_dtype=torch.int64, seed=4)


@pytest.mark.parametrize("rows_per_wave", [0, 64])
def test_a_bad_page_in_a_large_page_table_is_refused_and_the_rest_is_right(rows_per_wave):
    """Page sizes of 16 keys and more look their pages up on the scalar unit (the two-tile kernel: in the lanes that
    fetched them): the same error contract."""
    _native.lib().singe_hip_set_paged_attention_rows_per_wave(rows_per_wave)
    try:
        a_bad_page_is_refused_and_the_rest_is_right()
    finally:
        _native.lib().singe_hip_set_paged_attention_rows_per_wave(0)


def a_bad_page_is_refused_and_the_rest_is_right():
    gen = torch.Generator(device="cuda")
    gen.manual_seed(8)
    q = torch.randn((40, 4, 128), generator=gen, device="cuda").to(torch.bfloat16)
    cache = torch.randn((6, 32, 2, 128), generator=gen, device="cuda").to(torch.bfloat16)
    index = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    good = neural.Paging(index([0, 20, 40]), index([0, 3, 5]), index([4, 1, 0, 2, 5]), index([7, 32]))
    want, _ = neural.paged_attention(q, cache, cache, good, neural.AttentionOptions(causal=True))
    bad = neural.Paging(index([0, 20, 40]), index([0, 3, 5]), index([4, 1, 0, 2, 6]), index([7, 32]))  # page 6 of 6
    status = torch.zeros(1, dtype=torch.int32, device="cuda")
    got, _ = neural.paged_attention(q, cache, cache, bad, neural.AttentionOptions(causal=True), status=status, check=False)
    assert status.item() == 1
    assert torch.equal(got[:20], want[:20])  # the sequence with good pages is untouched by its neighbour's error
    with pytest.raises(error.IndexOutOfBounds):
        neural.paged_attention(q, cache, cache, bad, neural.AttentionOptions(causal=True))


TOKENS, HEADS, DIM, SLOTS, PAGES = 2, 2, 128, 4, 2
VALID = dict(query_offsets=[0, 2], page_offsets=[0, 1], pages=[0], last_page_lengths=[2])
INVALID = [dict(query_offsets=[0, 3]), dict(query_offsets=[-1, 2]), dict(query_offsets=[2, 0]), dict(page_offsets=[0, 2]),
           dict(page_offsets=[-1, 1]), dict(pages=[PAGES]), dict(pages=[-1]), dict(last_page_lengths=[SLOTS + 1]),
           dict(last_page_lengths=[-1])]


def attend(paging_values, dtype=torch.int64):
    # singe/tests/nn/paged_attention.rs:96-127 (head_dim 128 here: the width this build's kernel takes)
    q = torch.zeros((TOKENS, HEADS, DIM), device="cuda", dtype=torch.bfloat16)
    cache = torch.zeros((PAGES, SLOTS, HEADS, DIM), device="cuda", dtype=torch.bfloat16)
    values = {**VALID, **paging_values}
    index = lambda v: torch.tensor(v, dtype=dtype, device="cuda")
    paging = neural.Paging(index(values["query_offsets"]), index(values["page_offsets"]), index(values["pages"]),
                           index(values["last_page_lengths"]))
    return neural.paged_attention(q, cache, cache, paging, neural.AttentionOptions(causal=True))


@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
def test_paging_values_outside_their_buffers_are_refused(dtype):
    # singe/tests/nn/paged_attention.rs:24-73, 141-186
    attend({}, dtype)
    for bad in INVALID:
        with pytest.raises(error.IndexOutOfBounds):
            attend(bad, dtype)
        attend({}, dtype)  # the next valid launch succeeds
    attend(dict(last_page_lengths=[SLOTS]), dtype)
    attend(dict(query_offsets=[0, 0], page_offsets=[0, 0], pages=[PAGES + 7], last_page_lengths=[-1]), dtype)
    for bad in INVALID:
        assert oracle.check_paged_values(**{**VALID, **bad}, tokens=TOKENS, cache_pages=PAGES, page_size=SLOTS) == 1


def test_paged_equals_dense_prefill():
    # paged == dense invariant (singe/tests/nn/cross_attention.rs:120-198): one sequence whose queries
    # are all of its tokens is plain causal attention over the gathered keys.
    from singe_amd.kernel import attention as A

    length, heads, kv_heads, page_size, dim = 300, 8, 2, 16, 128
    query_offsets, page_offsets, table, last, page_count = layout([(length, length)], page_size)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(12)
    q = torch.randn((length, heads, dim), generator=gen, device="cuda").to(torch.bfloat16)
    kc = torch.randn((page_count, page_size, kv_heads, dim), generator=gen, device="cuda").to(torch.bfloat16)
    vc = torch.randn((page_count, page_size, kv_heads, dim), generator=gen, device="cuda").to(torch.bfloat16)
    index = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    out, lse = neural.paged_attention(q, kc, vc, neural.Paging(index(query_offsets), index(page_offsets), index(table), index(last)),
                                      neural.AttentionOptions(causal=True))
    rows = torch.tensor([table[k // page_size] * page_size + k % page_size for k in range(length)], device="cuda")
    k_dense = kc.view(-1, kv_heads, dim)[rows].unsqueeze(0).contiguous()
    v_dense = vc.view(-1, kv_heads, dim)[rows].unsqueeze(0).contiguous()
    dense = torch.empty((1, length, heads, dim), device="cuda", dtype=torch.bfloat16)
    dense_lse = torch.empty((1, heads, length), device="cuda")
    A.fmha_prefill_lse_bf16(None, dense, dense_lse, q.unsqueeze(0).contiguous(), k_dense, v_dense,
                            A.FmhaPrefillConfig.contiguous(1, length, length, heads, kv_heads, dim, dim ** -0.5, True))
    torch.cuda.synchronize()
    assert (out.float() - dense[0].float()).abs().max().item() <= 2 ** -6
    assert (lse - dense_lse[0].T / np.log(2.0)).abs().max().item() <= 2e-3


@pytest.mark.parametrize("splits", [2, 3, 7, 16, 64])
@pytest.mark.parametrize("options", [neural.AttentionOptions(causal=True), neural.AttentionOptions(),
                                     neural.AttentionOptions(causal=True, window=100, softcap=20.0)])
def test_key_splits_match_oracle(splits, options):
    """With scratch lent, a row tile's keys are shared out over workgroups and merged by a second kernel: decode rows
    over long and short caches, a chunk, a sequence without keys, more shares than a sequence has tiles."""
    from singe_amd import _native
    _native.lib().singe_hip_set_paged_attention_splits(splits)
    try:
        run_case([(1, 1500), (1, 40), (5, 700), (2, 0), (1, 65), (130, 300)], 8, 2, 16, options, seed=splits)
        run_case([(1, 333), (3, 64)], 8, 1, 7, options, index_dtype=torch.int64, seed=splits + 1)
    finally:
        _native.lib().singe_hip_set_paged_attention_splits(0)


def test_decode_shaped_calls_split_on_their_own_and_agree_with_the_unsplit_kernel():
    gen = torch.Generator(device="cuda")
    gen.manual_seed(21)
    lens = [4096, 512, 1000, 2047, 16, 3000, 1, 777]
    pages_of = [(n + 15) // 16 for n in lens]
    page_count = sum(pages_of) + 5
    q = torch.randn((len(lens), 32, 128), generator=gen, device="cuda").to(torch.bfloat16)
    kc = torch.randn((page_count, 16, 8, 128), generator=gen, device="cuda").to(torch.bfloat16)
    vc = torch.randn((page_count, 16, 8, 128), generator=gen, device="cuda").to(torch.bfloat16)
    index = lambda values: torch.tensor(values, dtype=torch.int32, device="cuda")
    table = np.random.default_rng(3).permutation(page_count)[:sum(pages_of)]
    paging = neural.Paging(index(list(range(len(lens) + 1))), index(np.concatenate([[0], np.cumsum(pages_of)])), index(table),
                           index([n - (p - 1) * 16 for n, p in zip(lens, pages_of)]))
    apart, apart_lse = on_row_tiles(q, kc, vc, paging, neural.AttentionOptions(causal=True))
    split, split_lse = neural.paged_attention(q, kc, vc, paging, neural.AttentionOptions(causal=True))
    # (4e-3 for 16-bit weights and the order of summation, and a step of bf16, 2^-7 of a value at most, where the two round apart:
    # outputs over sixteen keys pass one)
    assert ((apart.float() - split.float()).abs() - 2 ** -7 * apart.float().abs()).max().item() <= 4e-3
    assert (apart_lse - split_lse).abs().max().item() <= 1e-3


def test_a_stream_that_is_not_torchs_current_one_orders_the_fills_and_the_status_word():
    """The wrapper fills the output, the log-sum-exp and the status word and reads the word back: all of it has to
    run on the stream the kernel is launched on, also when that is not torch's current stream.  The current stream
    is kept busy meanwhile, so work queued on it by mistake would land after the kernel's."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(9)
    q = torch.randn((40, 4, 128), generator=gen, device="cuda").to(torch.bfloat16)
    cache = torch.randn((6, 32, 2, 128), generator=gen, device="cuda").to(torch.bfloat16)
    index = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    good = neural.Paging(index([0, 20, 40]), index([0, 3, 5]), index([4, 1, 0, 2, 5]), index([7, 32]))
    bad = neural.Paging(index([0, 20, 40]), index([0, 3, 5]), index([4, 1, 0, 2, 6]), index([7, 32]))
    want, want_lse = neural.paged_attention(q, cache, cache, good, neural.AttentionOptions(causal=True))
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    busy = torch.randn((4096, 4096), device="cuda")
    for _ in range(3):
        for _ in range(20):
            busy = busy @ busy * 1e-3  # the current stream stays busy while the side stream works
        got, got_lse = neural.paged_attention(q, cache, cache, good, neural.AttentionOptions(causal=True), stream=side)
        side.synchronize()
        assert torch.equal(got, want) and torch.equal(got_lse, want_lse)
        with pytest.raises(error.IndexOutOfBounds):
            neural.paged_attention(q, cache, cache, bad, neural.AttentionOptions(causal=True), stream=side)
    torch.cuda.synchronize()


ROW_TILES, DECODE_KERNELS, ONE_LAUNCH = 0, 1, 2


def route_of(q, kc, vc, paging, options):
    """The kernels that a call with as much scratch as it asks for runs on."""
    problem = ctypes.byref(neural._problem(q, kc, vc, paging, options))
    return _native.lib().singe_hip_paged_attention_route(problem, 256, _native.lib().singe_hip_paged_attention_scratch_bytes(problem))


def on_row_tiles(q, kc, vc, paging, options):
    """The same call on the row-tile kernel, one workgroup to a tile."""
    _native.lib().singe_hip_set_paged_attention_splits(1)
    try:
        assert route_of(q, kc, vc, paging, options) == ROW_TILES
        return neural.paged_attention(q, kc, vc, paging, options)
    finally:
        _native.lib().singe_hip_set_paged_attention_splits(0)


# A decode step (no more tokens than sequences, no cap) runs in one launch where it is small and the pages are powers of two of
# sixteen keys and up, and otherwise on the block-table decode kernels, token by token: (queries, keys) per sequence.
DECODE_STEPS = [
    [(1, 700), (1, 1), (1, 4096), (1, 33), (1, 16), (1, 2049), (1, 5003)], # a token a sequence, ragged
    [(1, 300), (0, 500), (1, 0), (1, 64), (0, 0), (1, 1500)],             # sequences without a token, a token without keys
    [(2, 2900), (0, 40), (1, 17), (0, 2000)],                             # two tokens of one sequence, as many tokens as sequences
    [(3, 2), (0, 5), (0, 7), (1, 129)],                                   # more queries than keys
    [(1, 128 * (b % 5) + b) for b in range(1, 70)],                       # more sequences than a wave has lanes
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("heads, kv_heads, page_size, dim", [(8, 2, 16, 128), (32, 4, 8, 128), (16, 1, 64, 128), (4, 4, 1, 128), (8, 2, 32, 64), (6, 1, 7, 64)])
@pytest.mark.parametrize("step", range(len(DECODE_STEPS)))
@pytest.mark.parametrize("index_dtype", [torch.int32, torch.int64])
def test_a_decode_step_through_the_op_matches_the_oracle_and_the_row_tile_kernel(step, heads, kv_heads, page_size, dim, dtype, index_dtype):
    one_launch = page_size in (16, 32, 64)
    windows = (2048, 2500, 100, 1 << 40) if dtype == torch.bfloat16 else ()
    check_decode_step(100 * step + heads, DECODE_STEPS[step], heads, kv_heads, page_size, dim, dtype, index_dtype, windows, ONE_LAUNCH if one_launch else DECODE_KERNELS)


# More keys than a step in one launch has: many sequences of over 900 keys on average, and few of many more.
LARGE_STEPS = [
    [(1, 300 + 97 * s % 1900) for s in range(68)] + [(0, 900), (1, 0), (2, 5003), (1, 1)],
    [(1, 120000), (1, 2500), (0, 40000), (1, 128000)],
]


@pytest.mark.parametrize("dtype,index_dtype", [(torch.bfloat16, torch.int32), (torch.bfloat16, torch.int64), (torch.float16, torch.int64)])
@pytest.mark.parametrize("step, heads, kv_heads, page_size, dim", [(0, 8, 2, 16, 128), (0, 16, 1, 64, 128), (0, 8, 2, 32, 64), (1, 8, 2, 16, 128), (1, 8, 2, 32, 64)])
def test_a_decode_step_past_the_one_launch_matches_the_oracle_and_the_row_tile_kernel(step, heads, kv_heads, page_size, dim, dtype, index_dtype):
    check_decode_step(100 * step + heads, LARGE_STEPS[step], heads, kv_heads, page_size, dim, dtype, index_dtype, (2048, 2500) if step == 0 else (), DECODE_KERNELS)


def check_decode_step(seed, sequences, heads, kv_heads, page_size, dim, dtype, index_dtype, windows, route):
    query_offsets, page_offsets, table, last, page_count = layout(sequences, page_size)
    tokens = query_offsets[-1]
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    rand = lambda *shape: torch.randn(shape, generator=gen, device="cuda").to(dtype)
    q, kc, vc = rand(tokens, heads, dim), rand(page_count, page_size, kv_heads, dim), rand(page_count, page_size, kv_heads, dim)
    index = lambda values: torch.tensor(values, dtype=index_dtype, device="cuda")
    paging = neural.Paging(index(query_offsets), index(page_offsets), index(table), index(last))
    # (windows from 2048 keys on take the decode kernels too: whole pages before the window are left out of a token's row,
    # the keys of its first page before the window are masked; shorter ones stay on the row-tile kernel where the step does not go in
    # one launch)
    windowed = tuple(neural.AttentionOptions(causal=True, window=window) for window in windows) + ((neural.AttentionOptions(window=2077),) if windows else ())
    for options in (neural.AttentionOptions(causal=True), neural.AttentionOptions(scale=0.05)) + windowed:
        short = options.window is not None and options.window < 2048
        assert route_of(q, kc, vc, paging, options) == (ROW_TILES if short and route == DECODE_KERNELS else route), options
        # the scratch the op asks for covers the decode kernels' rows and partials
        problem = neural._problem(q, kc, vc, paging, options)
        if options.window is None or options.window >= 2048:
            assert _native.lib().singe_hip_paged_attention_scratch_bytes(ctypes.byref(problem)) >= 2 * 256 + 4 * tokens * heads * (dim + 1)
        out, lse = neural.paged_attention(q, kc, vc, paging, options)
        tiled, tiled_lse = on_row_tiles(q, kc, vc, paging, options)
        torch.cuda.synchronize()
        status, want, want_lse = oracle.paged_attention_f32(q.float().cpu().numpy(), kc.float().cpu().numpy(), vc.float().cpu().numpy(), query_offsets,
                                                            page_offsets, table, last, scale=options.scale, causal=options.causal,
                                                            window=options.window, threads=8)
        assert status == 0
        got, got_lse = out.float().cpu().numpy(), lse.cpu().numpy()
        gap = np.abs(got - want)
        assert gap.max() <= MAX_ABS and gap.mean() <= MEAN_ABS, (options, gap.max(), gap.mean())
        empty = np.isneginf(want_lse)
        assert np.array_equal(np.isneginf(got_lse), empty) and not got[empty].any(), options
        assert np.abs(got_lse[~empty] - want_lse[~empty]).max(initial=0.0) <= LSE_ABS
        # (beyond a step of bf16, 2^-7 of a value at most, where the two round apart: outputs over two keys pass two)
        assert ((out.float() - tiled.float()).abs() - 2 ** -7 * tiled.float().abs()).max().item() <= 8e-3
        assert np.array_equal(np.isneginf(tiled_lse.cpu().numpy()), empty)


@pytest.mark.parametrize("index_dtype", [torch.int32, torch.int64])
def test_a_decode_step_keeps_the_error_contract_and_leaves_unowned_tokens_alone(index_dtype):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(4)
    q = torch.randn((3, 4, 128), generator=gen, device="cuda").to(torch.bfloat16)
    cache = torch.randn((6, 16, 2, 128), generator=gen, device="cuda").to(torch.bfloat16)
    index = lambda v: torch.tensor(v, dtype=index_dtype, device="cuda")
    options = neural.AttentionOptions(causal=True)
    good = neural.Paging(index([0, 1, 2, 3]), index([0, 2, 3, 5]), index([4, 1, 0, 2, 5]), index([7, 16, 3]))
    want, want_lse = neural.paged_attention(q, cache, cache, good, options)
    for pages, last in (([4, 1, 0, 2, 6], [7, 16, 3]), ([4, 1, 0, -1, 5], [7, 16, 3]), ([4, 1, 0, 2, 5], [7, 16, 17])):
        bad = neural.Paging(index([0, 1, 2, 3]), index([0, 2, 3, 5]), index(pages), index(last))
        status = torch.zeros(1, dtype=torch.int32, device="cuda")
        got, got_lse = neural.paged_attention(q, cache, cache, bad, options, status=status, check=False)
        assert status.item() == 1
        assert torch.equal(got[:2], want[:2]) and torch.equal(got_lse[:2], want_lse[:2])  # the sequences with good paging are right
        with pytest.raises(error.IndexOutOfBounds):
            neural.paged_attention(q, cache, cache, bad, options)
    # a page id outside the cache that no sequence with a token reads is not looked at
    unread = neural.Paging(index([0, 1, 2, 2]), index([0, 2, 3, 5]), index([4, 1, 0, 77, -3]), index([7, 16, 3]))
    got, _ = neural.paged_attention(q[:2], cache, cache, unread, options)
    assert torch.equal(got, want[:2])
    # tokens before the first sequence's and after the last one's belong to nobody: their rows stay as they were
    edges = neural.Paging(index([1, 2, 2, 2]), index([0, 2, 3, 3]), index([4, 1, 0]), index([7, 16, 0]))
    got, got_lse = neural.paged_attention(q, cache, cache, edges, options)
    tiled, tiled_lse = on_row_tiles(q, cache, cache, edges, options)
    assert (got[1].float() - tiled[1].float()).abs().max().item() <= 8e-3 and (got_lse[1] - tiled_lse[1]).abs().max().item() <= 2e-3
    assert not got[0].any() and not got[2].any() and torch.isneginf(got_lse[0]).all() and torch.isneginf(got_lse[2]).all()


@pytest.mark.parametrize("count, heads, kv_heads", [(7900, 4, 2), (3000, 16, 2), (2300, 16, 2)])
def test_a_decode_step_of_thousands_of_sequences(count, heads, kv_heads):
    """The decode kernels keep three words a token in LDS on this route: 7900 tokens fill it beside the one-hot form's
    staging; with eight heads a kv head 3000 tokens no longer fit beside the dense form's and take the one-hot form, 2300 do."""
    rng = np.random.default_rng(count)
    sequences = [(1, int(n)) for n in rng.integers(0, 40, count)]
    query_offsets, page_offsets, table, last, page_count = layout(sequences, 16)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(count)
    rand = lambda *shape: torch.randn(shape, generator=gen, device="cuda").to(torch.bfloat16)
    q, kc, vc = rand(count, heads, 128), rand(page_count, 16, kv_heads, 128), rand(page_count, 16, kv_heads, 128)
    index = lambda values: torch.tensor(values, dtype=torch.int64, device="cuda")
    paging = neural.Paging(index(query_offsets), index(page_offsets), index(table), index(last))
    out, lse = neural.paged_attention(q, kc, vc, paging, neural.AttentionOptions(causal=True))
    torch.cuda.synchronize()
    status, want, want_lse = oracle.paged_attention_f32(q.float().cpu().numpy(), kc.float().cpu().numpy(), vc.float().cpu().numpy(), query_offsets,
                                                        page_offsets, table, last, causal=True, threads=8)
    assert status == 0
    gap = np.abs(out.float().cpu().numpy() - want)
    assert gap.max() <= MAX_ABS and gap.mean() <= MEAN_ABS, (gap.max(), gap.mean())
    empty = np.isneginf(want_lse)
    assert np.array_equal(np.isneginf(lse.cpu().numpy()), empty)
    assert np.abs(lse.cpu().numpy()[~empty] - want_lse[~empty]).max() <= LSE_ABS


@pytest.fixture
def two_tiles_a_wave():
    """Sends every paged call that has the form to the kernel that gives a wave two 32-row tiles."""
    _native.lib().singe_hip_set_paged_attention_rows_per_wave(64)
    yield
    _native.lib().singe_hip_set_paged_attention_rows_per_wave(0)


@pytest.mark.parametrize("index_dtype", [torch.int32, torch.int64])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("heads,kv_heads,page_size,dim", [(8, 1, 16, 128), (64, 8, 16, 128), (8, 2, 32, 128), (4, 1, 64, 128), (8, 2, 128, 128),
                                                          (4, 4, 16, 128), (8, 1, 16, 64), (64, 8, 16, 64), (8, 2, 64, 64), (4, 4, 32, 64),
                                                          (8, 1, 16, 96), (64, 8, 16, 96), (8, 2, 64, 96), (4, 4, 32, 96),
                                                          (8, 1, 16, 112), (8, 2, 64, 112), (64, 8, 16, 80), (4, 4, 32, 80), (8, 1, 16, 48),
                                                          (8, 2, 128, 48), (64, 8, 16, 32), (4, 1, 64, 32), (8, 2, 16, 16), (4, 4, 256, 16)])
def test_two_tiles_a_wave_ragged_sequences_match_oracle(two_tiles_a_wave, heads, kv_heads, page_size, dim, causal, index_dtype):
    # the shapes of the ragged test (decode, full prefill, chunked prefill, no keys, more queries than keys) and
    # chunks long enough for several 256-row tiles, several key tiles ahead of the mask and key counts either side of
    # a tile's and a page's end
    sequences = [(1, 150), (70, 70), (20, 90), (3, 0), (9, 4), (130, 300), (300, 1000), (257, 513), (64, 1024), (512, 512)]
    run_case(sequences, heads, kv_heads, page_size, neural.AttentionOptions(causal=causal), index_dtype=index_dtype,
             seed=heads + page_size + 1, dim=dim)


def test_two_tiles_a_wave_equals_the_four_wave_kernel_at_the_chunked_prefill_shape():
    # The fourth benchmark configuration fills the chip with 256-row tiles, so the default choice is this kernel: its
    # answer against the 32-row kernel's, within the rounding of the output.
    from singe_amd import synthetic
    work = synthetic.chunked_prefill_workload(portable=True)
    index = lambda values: torch.from_numpy(np.asarray(values, dtype=np.int32)).cuda()
    paging = neural.Paging(index(work.query_offsets), index(work.page_offsets), index(work.pages), index(work.last_page_lengths))
    options = neural.AttentionOptions(causal=True)
    chosen, chosen_lse = neural.paged_attention(work.query, work.key_cache, work.value_cache, paging, options)
    _native.lib().singe_hip_set_paged_attention_rows_per_wave(32)
    try:
        narrow, narrow_lse = neural.paged_attention(work.query, work.key_cache, work.value_cache, paging, options)
    finally:
        _native.lib().singe_hip_set_paged_attention_rows_per_wave(0)
    torch.cuda.synchronize()
    assert (chosen.float() - narrow.float()).abs().max().item() <= 2 ** -6
    assert (chosen_lse - narrow_lse).abs().max().item() <= 1e-4


@pytest.mark.parametrize("rows_per_wave", [64, 32])
@pytest.mark.parametrize("index_dtype", [torch.int32, torch.int64])
def test_pages_beyond_two_and_four_gib_of_a_cache_read_the_same_as_the_first_pages(rows_per_wave, index_dtype):
    # 150 000 pages of 32 KiB: a page's first byte lies past 2^31 from id 65 536 and past 2^32 from id 131 072.  The
    # same page contents under small ids in a small cache must give the same bits.
    heads, kv_heads, page_size, cache_pages = 32, 8, 16, 150_000
    sequences = [(300, 700), (256, 512)]
    gen = torch.Generator(device="cuda")
    gen.manual_seed(77)
    page_counts = [-(-keys // page_size) for _, keys in sequences]
    used = sum(page_counts)
    high = torch.tensor([65_536 + 3, 131_072 + 5, cache_pages - 1, 70_001, 140_002, 100_000], dtype=torch.int64)
    ids_high = torch.cat([high, 90_000 + 7 * torch.arange(used - len(high))])
    ids_low = torch.randperm(used)
    small_k = torch.randn((used, page_size, kv_heads, 128), generator=gen, device="cuda").to(torch.bfloat16)
    small_v = torch.randn((used, page_size, kv_heads, 128), generator=gen, device="cuda").to(torch.bfloat16)
    big_k = torch.zeros((cache_pages, page_size, kv_heads, 128), device="cuda", dtype=torch.bfloat16)
    big_v = torch.zeros((cache_pages, page_size, kv_heads, 128), device="cuda", dtype=torch.bfloat16)
    big_k[ids_high.cuda()] = small_k[ids_low.cuda()]
    big_v[ids_high.cuda()] = small_v[ids_low.cuda()]
    tokens = sum(queries for queries, _ in sequences)
    q = torch.randn((tokens, heads, 128), generator=gen, device="cuda").to(torch.bfloat16)
    query_offsets = np.concatenate([[0], np.cumsum([queries for queries, _ in sequences])])
    page_offsets = np.concatenate([[0], np.cumsum(page_counts)])
    last = [keys - (count - 1) * page_size for (_, keys), count in zip(sequences, page_counts)]
    index = lambda values: torch.as_tensor(np.asarray(values), dtype=index_dtype).cuda()
    options = neural.AttentionOptions(causal=True)
    _native.lib().singe_hip_set_paged_attention_rows_per_wave(rows_per_wave)
    try:
        far, far_lse = neural.paged_attention(q, big_k, big_v, neural.Paging(index(query_offsets), index(page_offsets), index(ids_high.numpy()), index(last)), options)
        near, near_lse = neural.paged_attention(q, small_k, small_v, neural.Paging(index(query_offsets), index(page_offsets), index(ids_low.numpy()), index(last)), options)
    finally:
        _native.lib().singe_hip_set_paged_attention_rows_per_wave(0)
    torch.cuda.synchronize()
    assert torch.equal(far, near) and torch.equal(far_lse, near_lse)
    assert far.float().abs().max().item() > 0.1


@pytest.mark.parametrize("page_size,near_page", [(1 << 20, 512), ((1 << 20) + 3, 515)])
@pytest.mark.parametrize("queries", [2, 40])
def test_places_beyond_four_gib_of_one_page_read_the_same_as_near_its_start(queries, page_size, near_page):
    # One page of 5.4 GB (20 kv heads x 128: 5 KiB a key): its last keys, all that the window leaves, lie past byte 2^32 of it.
    # The same keys at the end of a small page must give the same bits.
    heads, kv_heads, window = 40, 20, 200
    keys, skipped = page_size - 5, page_size - near_page
    assert skipped % 64 == 0
    gen = torch.Generator(device="cuda")
    gen.manual_seed(queries)
    rand = lambda *shape: torch.randn(shape, generator=gen, device="cuda").to(torch.bfloat16)
    q, small_k, small_v = rand(queries, heads, 128), rand(1, near_page, kv_heads, 128), rand(1, near_page, kv_heads, 128)
    big_k, big_v = (torch.zeros((1, page_size, kv_heads, 128), device="cuda", dtype=torch.bfloat16) for _ in range(2))
    big_k[:, skipped:], big_v[:, skipped:] = small_k, small_v
    index = lambda *values: torch.tensor(values, dtype=torch.int32, device="cuda")
    options = neural.AttentionOptions(causal=True, window=window)
    far, far_lse = neural.paged_attention(q, big_k, big_v, neural.Paging(index(0, queries), index(0, 1), index(0), index(keys)), options)
    near, near_lse = neural.paged_attention(q, small_k, small_v, neural.Paging(index(0, queries), index(0, 1), index(0), index(keys - skipped)), options)
    torch.cuda.synchronize()
    assert torch.equal(far, near) and torch.equal(far_lse, near_lse)
    assert far.float().abs().max().item() > 0.1


NARROW = [(1, 1), (2, 15), (1, 16), (2, 17), (1, 63), (2, 64), (1, 65), (2, 0), (0, 40), (2, 1), (1, 129), (2, 1000)]


@pytest.mark.parametrize("options", OPTIONS + [neural.AttentionOptions(causal=True, scale=-0.07, window=33)])
@pytest.mark.parametrize("heads,kv_heads,page_size,dim,index_dtype", [
    (8, 1, 16, 128, torch.int64), (12, 3, 32, 64, torch.int32), (6, 6, 64, 96, torch.int64), (16, 2, 16, 32, torch.int32), (14, 2, 128, 128, torch.int32)])
def test_sequences_of_at_most_sixteen_rows_beside_a_chunk(heads, kv_heads, page_size, dim, index_dtype, options):
    """Groups of sixteen keys dealt to four waves: keys either side of a group's, a turn's and a page's end, sequences with
    fewer groups than waves, one to sixteen rows, without queries or keys, beside a chunk that fills row tiles."""
    run_case(NARROW + [(150, 400)], heads, kv_heads, page_size, options, index_dtype=index_dtype, seed=dim + heads, dim=dim)


@pytest.mark.parametrize("options", [OPTIONS[1], OPTIONS[2], OPTIONS[4]])
@pytest.mark.parametrize("heads,kv_heads,page_size,dim", [(8, 1, 16, 128), (12, 3, 32, 64), (16, 2, 16, 32)])
def test_f16_sequences_of_at_most_sixteen_rows_beside_a_chunk(heads, kv_heads, page_size, dim, options):
    run_case(NARROW + [(150, 400)], heads, kv_heads, page_size, options, seed=dim, dim=dim, dtype=torch.float16)


@pytest.mark.parametrize("heads,kv_heads,splits", [(8, 1, 0), (8, 1, 3), (4, 2, 1)])
def test_sequences_of_at_most_sixteen_rows_over_many_keys(heads, kv_heads, splits):
    # a wave looks 64 groups' page ids up at a time: 64 turns are 4096 keys
    _native.lib().singe_hip_set_paged_attention_splits(splits)
    try:
        run_case([(1, 4095), (2, 4096), (1, 4160), (1, 8300), (40, 100)], heads, kv_heads, 16, neural.AttentionOptions(causal=True), seed=splits)
    finally:
        _native.lib().singe_hip_set_paged_attention_splits(0)


@pytest.mark.parametrize("index_dtype", [torch.int32, torch.int64])
@pytest.mark.parametrize("heads,kv_heads,decoding,chunks", [(8, 1, 60, 2), (16, 2, 100, 12), (6, 3, 230, 20), (32, 32, 40, 3), (64, 8, 66, 4)])
def test_decoding_sequences_and_row_tiles_take_turns_in_the_grid(heads, kv_heads, decoding, chunks, index_dtype):
    """Long enough on average that the list of row tiles alternates runs of either: more sequences than a wave has lanes,
    fewer of either than a run, every sequence attended."""
    rng = np.random.default_rng(heads + decoding)
    sequences = [(1, int(n)) for n in rng.integers(300, 1500, size=decoding)]
    sequences += [(int(q), int(q) + int(n)) for q, n in zip(rng.integers(17, 90, size=chunks), rng.integers(0, 900, size=chunks))]
    order = rng.permutation(len(sequences))
    run_case([sequences[i] for i in order], heads, kv_heads, 16, neural.AttentionOptions(causal=True), index_dtype=index_dtype, seed=decoding)


def test_offsets_that_run_backwards_are_reported_from_a_list_that_takes_turns():
    heads, kv_heads, page_size, pages = 16, 2, 16, 80
    gen = torch.Generator(device="cuda")
    gen.manual_seed(2)
    rand = lambda *shape: torch.randn(shape, generator=gen, device="cuda").to(torch.bfloat16)
    index = lambda values: torch.tensor(values, dtype=torch.int32, device="cuda")
    # sequence 1 runs backwards, and the tokens are claimed three times over
    paging = neural.Paging(index([0, 300, 0, 300] + list(range(240, 301)) + [0, 300]), index([pages * i for i in range(67)]),
                           index([i % pages for i in range(66 * pages)]), index([16] * 66))
    with pytest.raises(error.IndexOutOfBounds):
        neural.paged_attention(rand(300, heads, 128), rand(pages, page_size, kv_heads, 128), rand(pages, page_size, kv_heads, 128), paging,
                               neural.AttentionOptions(causal=True))


def poison(*shapes):
    """Blocks of NaN given back to the allocator: what an output that nothing wrote would hold."""
    blocks = [torch.full(shape, float("nan"), device="cuda", dtype=dtype) for shape, dtype in shapes]
    torch.cuda.synchronize()
    del blocks


def run_with_faults(heads, kv_heads, tokens, offsets, page_offsets, last, rows_per_wave=0, splits=0, index_dtype=torch.int32, route=None):
    """The outputs over poisoned memory, the status word and the operands, for sequences whose paging need not make sense."""
    page_size, cache_pages = 16, 50
    gen = torch.Generator(device="cuda")
    gen.manual_seed(tokens + len(offsets))
    rand = lambda *shape: torch.randn(shape, generator=gen, device="cuda").to(torch.bfloat16)
    index = lambda values: torch.tensor([int(v) for v in values], dtype=index_dtype, device="cuda")
    q, kc, vc = rand(tokens, heads, 128), rand(cache_pages, page_size, kv_heads, 128), rand(cache_pages, page_size, kv_heads, 128)
    pages = [(7 * i + 3) % cache_pages for i in range(max(page_offsets))]
    status = torch.zeros(1, dtype=torch.int32, device="cuda")
    _native.lib().singe_hip_set_paged_attention_rows_per_wave(rows_per_wave)
    _native.lib().singe_hip_set_paged_attention_splits(splits)
    try:
        paging = neural.Paging(index(offsets), index(page_offsets), index(pages), index(last))
        assert route is None or route_of(q, kc, vc, paging, neural.AttentionOptions(causal=True)) == route
        poison(((tokens, heads, 128), torch.bfloat16), ((tokens, heads), torch.float32))
        out, lse = neural.paged_attention(q, kc, vc, paging, neural.AttentionOptions(causal=True), status=status, check=False)
    finally:
        _native.lib().singe_hip_set_paged_attention_rows_per_wave(0)
        _native.lib().singe_hip_set_paged_attention_splits(0)

    def alone(s):
        mine = pages[page_offsets[s]:page_offsets[s + 1]]
        return neural.paged_attention(q[offsets[s]:offsets[s + 1]].contiguous(), kc, vc,
                                      neural.Paging(index([0, offsets[s + 1] - offsets[s]]), index([0, len(mine)]), index(mine), index([last[s]])),
                                      neural.AttentionOptions(causal=True))

    return out, lse, int(status.item()), alone


def check_rows_are_whole(tokens, offsets, valid, out, lse, alone, attended):
    """Every row is that of a valid sequence that has its token, or zeros with a log-sum-exp of -inf: the latter where there is
    no such sequence, the former where `attended` says that its sequence is attended.  Tokens that two sequences claim have rows
    of either, head by head and share by share."""
    zero = ~out.any(dim=-1).any(dim=-1) & torch.isneginf(lse).all(dim=-1)
    right, claims, needed = zero.clone(), torch.zeros_like(zero, dtype=torch.int32), torch.zeros_like(zero)
    for s in np.flatnonzero(valid):
        rows = slice(offsets[s], offsets[s + 1])
        if offsets[s] == offsets[s + 1]:
            continue
        want, want_lse = alone(s)
        right[rows] |= ((out[rows].float() - want.float()).abs().amax(dim=(1, 2)) <= MAX_ABS) & ((lse[rows] - want_lse).abs().amax(dim=1) <= LSE_ABS)
        claims[rows] += 1
        needed[rows] |= bool(attended[s])
    assert torch.isfinite(out.float()).all() and not torch.isnan(lse).any()
    right |= claims > 1
    assert right.all(), torch.nonzero(~right).flatten().tolist()[:8]
    assert zero[claims == 0].all()
    assert not zero[needed].any()


# Sequences that claim the same tokens over and over, between them ones that run backwards: more row tiles than the grid holds in
# front of the first of those, were they taken in any order but their own.
BACKWARDS = {
    "fewer decoding sequences than a run": (8, 1, 1000, [0, 1000] * 35 + [0], [40] * 70),
    "a handful of sequences": (16, 2, 300, [0, 300] * 6, [40] * 11),
    "longest first": (16, 2, 1000, [0, 1000] * 6, [40, 1] * 5 + [40]),
    "past the last token": (16, 2, 1000, [0, 500, 1001, 1000, 200, 1000, 0, 1000], [40, 1, 1, 40, 40, 1, 40]),
    "before the first token": (16, 2, 1000, [-1000, 0, 1000, 0, 1000, 0, 1000], [1, 40, 1, 40, 1, 40]),
}


@pytest.mark.parametrize("rows_per_wave", [32, 64])
@pytest.mark.parametrize("case", BACKWARDS)
def test_offsets_that_make_no_sense_are_reported_however_many_row_tiles_are_claimed(case, rows_per_wave):
    heads, kv_heads, tokens, offsets, page_counts = BACKWARDS[case]
    ends = np.concatenate([[0], np.cumsum(page_counts)]).tolist()
    out, lse, status, alone = run_with_faults(heads, kv_heads, tokens, offsets, ends, [16] * len(page_counts), rows_per_wave)
    assert status == neural.STATUS_INDEX_OUT_OF_BOUNDS
    valid = [0 <= start <= end <= tokens for start, end in zip(offsets, offsets[1:])]
    first_bad = valid.index(False)
    check_rows_are_whole(tokens, offsets, valid, out, lse, alone, [s < first_bad for s in range(len(valid))])


# (query tokens, pages held) of the sequences, the rows a wave, the key shares; tokens before the first and after the last one
ROUTES = {
    "row tiles, longest first": ([(200, 30), (330, 50), (150, 12), (200, 40), (64, 20)], 32, 1),
    "row tiles and decoding sequences in turns": ([(1, 40 + s) for s in range(12)] + [(200, 60)] + [(1, 70), (2, 50)], 32, 1),
    "row tiles in order": ([(1, 3), (2, 5), (90, 9), (1, 6), (40, 4)], 32, 1),
    "one row tile a sequence": ([(1, 3), (2, 5), (9, 9), (1, 6), (4, 4)], 32, 1),
    "shares": ([(1, 40), (60, 45), (30, 50), (1, 60), (40, 44)], 32, 3),
    "two tiles a wave": ([(200, 30), (330, 50), (150, 12), (200, 40), (64, 20)], 64, 1),
    "one launch": ([(1, 5 + s % 7) for s in range(40)] + [(0, 2)] * 20, 0, 0),
    "one launch over many keys": ([(1, 1500), (1, 1400), (1, 1600), (1, 1500), (1, 900)] + [(0, 1)] * 20, 0, 0),
    "decode": ([(1, 5 + s % 7) for s in range(200)] + [(0, 2)] * 70, 0, 0),
    "decode over many keys": ([(1, 3500), (1, 1400), (1, 1600), (1, 1500), (1, 2900)] + [(0, 1)] * 20, 0, 0),
}


@pytest.mark.parametrize("index_dtype", [torch.int32, torch.int64])
@pytest.mark.parametrize("fault", ["query offsets", "page offsets", "last page length"])
@pytest.mark.parametrize("route", ROUTES)
def test_a_sequence_that_is_refused_leaves_the_others_whole_and_its_own_rows_zero(route, fault, index_dtype):
    sequences, rows_per_wave, splits = ROUTES[route]
    offsets = (5 + np.concatenate([[0], np.cumsum([queries for queries, _ in sequences])])).tolist()
    page_offsets = np.concatenate([[0], np.cumsum([pages for _, pages in sequences])]).tolist()
    last = [9] * len(sequences)
    tokens, bad = offsets[-1] + (9 if splits != 0 or rows_per_wave != 0 else 0), 2
    if fault == "query offsets":
        offsets[bad + 1] = offsets[bad] - 1
    elif fault == "page offsets":
        page_offsets[bad + 1] = page_offsets[bad] - 1
    else:
        last[bad] = 17
    expected = DECODE_KERNELS if route.startswith("decode") else ONE_LAUNCH if route.startswith("one launch") else ROW_TILES
    out, lse, status, alone = run_with_faults(8, 2, tokens, offsets, page_offsets, last, rows_per_wave, 0 if splits == 1 else splits, index_dtype, expected)
    assert status == neural.STATUS_INDEX_OUT_OF_BOUNDS
    valid = [s != bad for s in range(len(sequences))]
    # (the decode kernels look a token's sequence up by bisection, which offsets that run backwards lead astray)
    attended = [s < bad or fault != "query offsets" or not route.startswith("decode") for s in range(len(sequences))]
    check_rows_are_whole(tokens, offsets, valid, out, lse, alone, attended)


@pytest.mark.parametrize("index_dtype", [torch.int32, torch.int64])
@pytest.mark.parametrize("case", ["row tiles", "shares", "two tiles a wave", "step", "decode", "many keys"])
def test_tokens_no_sequence_owns_are_zero_with_a_log_sum_exp_of_minus_infinity(case, index_dtype):
    heads, kv_heads, page_size = 8, 2, 16
    tokens, owned = {"step": (40, [(5, 1), (9, 1), (10, 0), (10, 1)]), "decode": (40, [(5, 1), (9, 1), (10, 0), (10, 1)]), "many keys": (300, [(33, 1), (40, 200)])}.get(
        case, (700, [(3, 7), (10, 0), (10, 255), (265, 1), (266, 200)]))
    keys = [4000 if case == "many keys" else 90 + 10 * s for s in range(len(owned))]
    if case in ("step", "decode"):  # a token a sequence at most, sequences without tokens after them
        more = 40 if case == "step" else 300
        owned, keys = owned + [(11, 0)] * more, keys + [20] * more
    pages = [(k + page_size - 1) // page_size for k in keys]
    offsets = [start for start, _ in owned] + [owned[-1][0] + owned[-1][1]]
    # (sequences are consecutive: the gap after one goes to the next, so only the front and the back are unowned)
    mine = torch.zeros(tokens, dtype=torch.bool, device="cuda")
    mine[offsets[0]:offsets[-1]] = True
    gen = torch.Generator(device="cuda")
    gen.manual_seed(3)
    rand = lambda *shape: torch.randn(shape, generator=gen, device="cuda").to(torch.bfloat16)
    index = lambda values: torch.tensor([int(v) for v in values], dtype=index_dtype, device="cuda")
    paging = neural.Paging(index(offsets), index(np.concatenate([[0], np.cumsum(pages)])), index(np.arange(sum(pages))),
                           index([k - (n - 1) * page_size for k, n in zip(keys, pages)]))
    q, kc, vc = rand(tokens, heads, 128), rand(sum(pages), page_size, kv_heads, 128), rand(sum(pages), page_size, kv_heads, 128)
    _native.lib().singe_hip_set_paged_attention_splits(3 if case == "shares" else 0)
    _native.lib().singe_hip_set_paged_attention_rows_per_wave(64 if case == "two tiles a wave" else 0)
    try:
        assert route_of(q, kc, vc, paging, neural.AttentionOptions(causal=True)) == {"step": ONE_LAUNCH, "decode": DECODE_KERNELS}.get(case, ROW_TILES)
        poison(((tokens, heads, 128), torch.bfloat16), ((tokens, heads), torch.float32))
        out, lse = neural.paged_attention(q, kc, vc, paging, neural.AttentionOptions(causal=True))
    finally:
        _native.lib().singe_hip_set_paged_attention_splits(0)
        _native.lib().singe_hip_set_paged_attention_rows_per_wave(0)
    assert not out[~mine].any() and torch.isneginf(lse[~mine]).all()
    assert torch.isfinite(out[mine].float()).all() and torch.isfinite(lse[mine]).all()
    assert (out[mine].float().abs().amax(dim=-1) > 0).all()


@pytest.mark.parametrize("dim,dtype", [(16, torch.bfloat16), (32, torch.float16), (48, torch.bfloat16), (64, torch.float16), (80, torch.bfloat16),
                                       (96, torch.float16), (112, torch.bfloat16), (128, torch.float16)])
@pytest.mark.parametrize("case", ["row tiles", "shares", "two tiles a wave", "step", "step of one sequence", "decode", "decode of one sequence", "decode of many sequences"])
def test_rows_no_sequence_owns_at_every_width(case, dim, dtype):
    """(queries, keys) of the sequences, unowned tokens before the first and after the last: also the decode kernels' merges of
    a row's shares, for few of them (more sequences than workers), some, and many (a lone long sequence), and steps in one launch."""
    before, after, sequences = {"step": (3, 4, [(1, 700)] * 3 + [(0, 9)] * 20), "step of one sequence": (2, 1, [(1, 20000)] + [(0, 1)] * 3),
                                "decode": (3, 4, [(1, 1100)] * 46 + [(0, 9)] * 8), "decode of one sequence": (2, 1, [(1, 150000)] + [(0, 1)] * 3),
                                "decode of many sequences": (5, 6, [(1, 60)] * 600 + [(0, 3)] * 11)}.get(case, (3, 300, [(7, 40), (255, 300), (1, 90)]))
    heads, kv_heads, page_size = 8, 2, 16
    query_offsets, page_offsets, table, last, page_count = layout(sequences, page_size)
    tokens = before + query_offsets[-1] + after
    gen = torch.Generator(device="cuda")
    gen.manual_seed(dim)
    rand = lambda *shape: torch.randn(shape, generator=gen, device="cuda").to(dtype)
    index = lambda values: torch.tensor([int(v) for v in values], dtype=torch.int32, device="cuda")
    paging = neural.Paging(index([before + offset for offset in query_offsets]), index(page_offsets), index(table), index(last))
    q, kc, vc = rand(tokens, heads, dim), rand(page_count, page_size, kv_heads, dim), rand(page_count, page_size, kv_heads, dim)
    _native.lib().singe_hip_set_paged_attention_splits(3 if case == "shares" else 0)
    _native.lib().singe_hip_set_paged_attention_rows_per_wave(64 if case == "two tiles a wave" else 32 if case == "row tiles" else 0)
    expected = ROW_TILES if not case.startswith(("step", "decode")) else ONE_LAUNCH if case.startswith("step") and dim % 32 == 0 else DECODE_KERNELS
    try:
        assert route_of(q, kc, vc, paging, neural.AttentionOptions(causal=True)) == expected
        poison(((tokens, heads, dim), dtype), ((tokens, heads), torch.float32))
        out, lse = neural.paged_attention(q, kc, vc, paging, neural.AttentionOptions(causal=True))
    finally:
        _native.lib().singe_hip_set_paged_attention_splits(0)
        _native.lib().singe_hip_set_paged_attention_rows_per_wave(0)
    mine = torch.zeros(tokens, dtype=torch.bool, device="cuda")
    mine[before:tokens - after] = True
    assert not out[~mine].any() and torch.isneginf(lse[~mine]).all()
    assert torch.isfinite(out.float()).all() and torch.isfinite(lse[mine]).all()
    assert (out[mine].float().abs().amax(dim=-1) > 0).all()


STEPS = [
    [(1, 100)], [(1, 3000)], [(1, 16)], [(1, 897), (1, 896), (1, 895)],                        # not shared out, shared out, either side of the line
    [(1, 1), (1, 9000), (1, 0), (1, 33), (0, 500), (1, 64), (1, 65), (1, 4096)],               # one that is far longer, one without keys, one without tokens
    [(2, 700), (1, 100), (0, 90), (3, 2), (0, 40), (0, 16)],                                   # several tokens of a sequence, more of them than keys
    [(0, 300)] * 40 + [(40, 2000), (0, 77)],                                                   # all tokens one sequence's, in several units
    [(1, 37 * i % 700) for i in range(100)],                                                   # more sequences than a wave has lanes
]


@pytest.mark.parametrize("options", [OPTIONS[0], OPTIONS[1], OPTIONS[3], neural.AttentionOptions(causal=True, scale=-0.07, window=1000)])
@pytest.mark.parametrize("heads,kv_heads,page_size,dim,dtype,index_dtype", [
    (32, 8, 16, 128, torch.bfloat16, torch.int64), (16, 1, 32, 64, torch.float16, torch.int32), (6, 2, 64, 96, torch.bfloat16, torch.int32),
    (4, 4, 16, 32, torch.float16, torch.int64), (10, 2, 16, 128, torch.bfloat16, torch.int64)])  # (five heads: threads that merge nothing)
@pytest.mark.parametrize("step", range(len(STEPS)))
def test_decode_steps_in_one_launch(step, heads, kv_heads, page_size, dim, dtype, index_dtype, options):
    run_case(STEPS[step], heads, kv_heads, page_size, options, index_dtype=index_dtype, seed=step, dim=dim, dtype=dtype)


def test_a_decode_step_in_one_launch_replays_over_whatever_its_scratch_holds():
    """Shares tell each other that they are done by words in the scratch: none is taken from an earlier use of it, be that
    another problem's partial rows, bytes of any kind or the same captured launch's last replay."""
    lengths = [3000, 9000, 100, 2000]
    query_offsets, page_offsets, table, last, page_count = layout([(1, n) for n in lengths], 16)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(3)
    q = torch.randn((4, 32, 128), generator=gen, device="cuda").bfloat16()
    kc, vc = (torch.randn((page_count, 16, 8, 128), generator=gen, device="cuda").bfloat16() for _ in range(2))
    index = lambda values: torch.tensor(values, dtype=torch.int64, device="cuda")
    paging = neural.Paging(index(query_offsets), index(page_offsets), index(table), index(last))
    options = neural.AttentionOptions(causal=True)
    status = torch.zeros(1, device="cuda", dtype=torch.int32)
    scratch = torch.empty(8 << 20, device="cuda", dtype=torch.uint8)
    call = lambda: neural.paged_attention(q, kc, vc, paging, options, status=status, check=False, scratch=scratch)
    want, want_lse = call()
    code, reference, reference_lse = oracle.paged_attention_f32(q.float().cpu().numpy(), kc.float().cpu().numpy(), vc.float().cpu().numpy(), query_offsets,
                                                                page_offsets, table, last, scale=None, causal=True, threads=8)
    assert code == 0 and np.abs(want.float().cpu().numpy() - reference).max() <= MAX_ABS and np.abs(want_lse.cpu().numpy() - reference_lse).max() <= LSE_ABS
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        call()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            out, lse = call()
        for turn in range(6):
            if turn % 2 == 1:
                scratch.copy_(torch.randint(0, 256, scratch.shape, generator=gen, device="cuda", dtype=torch.uint8))
            if turn % 3 == 2:
                call()
            q.copy_(torch.randn(q.shape, generator=gen, device="cuda"))
            out.fill_(float("nan"))
            graph.replay()
            fresh, fresh_lse = call()
            stream.synchronize()
            assert torch.equal(out, fresh) and torch.equal(lse, fresh_lse)


@pytest.mark.parametrize("first,count", [(16, 8 << 20), (0, 1 << 18), (16, 100)])
def test_scratch_that_starts_anywhere_or_is_short_serves_a_decode_step(first, count):
    """Off a 256-byte boundary the keys are shared out by the row tiles, as they are where the scratch is too short for the one launch;
    with too little for either the call goes without."""
    query_offsets, page_offsets, table, last, page_count = layout([(1, 3000), (1, 50)], 16)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(5)
    rand = lambda *shape: torch.randn(shape, generator=gen, device="cuda").bfloat16()
    q, kc, vc = rand(2, 32, 128), rand(page_count, 16, 8, 128), rand(page_count, 16, 8, 128)
    index = lambda values: torch.tensor(values, dtype=torch.int32, device="cuda")
    paging = neural.Paging(index(query_offsets), index(page_offsets), index(table), index(last))
    scratch = torch.empty(first + count, device="cuda", dtype=torch.uint8)[first:]
    out, lse = neural.paged_attention(q, kc, vc, paging, neural.AttentionOptions(causal=True), scratch=scratch)
    status, want, want_lse = oracle.paged_attention_f32(q.float().cpu().numpy(), kc.float().cpu().numpy(), vc.float().cpu().numpy(), query_offsets,
                                                        page_offsets, table, last, causal=True, threads=8)
    assert status == 0
    gap = np.abs(out.float().cpu().numpy() - want)
    assert gap.max() <= MAX_ABS and gap.mean() <= MEAN_ABS and np.abs(lse.cpu().numpy() - want_lse).max() <= LSE_ABS
