"""An infinity or a NaN among the values of a key: it reaches the rows that see the key and no others, also where a matrix
product weighs the values of hidden keys by zero.  The ops whose reference walks only a row's own keys: packed 16-bit
prefill and dense f32 attention.  And of paged attention what cache places that belong to no key hold, and keys that other
sequences and kv heads see.

The reference is float64 over each row's visible keys; where it is finite the output is, within the type's rounding of
values up to about 4 (bf16 2^-9, f16 2^-12, f32 sums), and elsewhere the same infinity or NaN."""
import math

import pytest
import torch

from singe_amd import neural
from singe_amd.kernel import attention as A

pytestmark = pytest.mark.gpu

INF, NAN = math.inf, math.nan
TOL = {torch.bfloat16: 2e-2, torch.float16: 4e-3, torch.float32: 2e-5}


def draw(seed, *shape):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed))


def visible_only(q, k, v, first, end, scale):
    """[rows, heads, dim] in float64: row i over keys first[i] .. end[i] - 1."""
    group = q.shape[1] // k.shape[1]
    q, k, v = q.double(), k.double().repeat_interleave(group, 1), v.double().repeat_interleave(group, 1)
    out = torch.zeros_like(q)
    for i, (f, e) in enumerate(zip(first, end)):
        if e > f:
            weights = torch.softmax(torch.einsum("hd,khd->hk", q[i], k[f:e]) * scale, -1)
            out[i] = (weights[:, :, None] * v[f:e].transpose(0, 1)).sum(1)
    return out


def same(out, want, dtype):
    out = out.double().cpu()
    finite = want.isfinite()
    assert ((out[finite] - want[finite]).abs() <= TOL[dtype]).all()
    assert (out.isnan() == want.isnan()).all() and (out[want.isinf()] == want[want.isinf()]).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("dim", [128, 80, 16])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("bad", [INF, -INF, NAN])
def test_packed(dtype, dim, causal, bad):
    heads, kv_heads, lens = 4, 2, [40, 200, 1, 70]
    offsets = [0, 40, 240, 241]
    tokens, scale = sum(lens), dim ** -0.5
    q, k, v = (draw(seed, tokens, h, dim).to(dtype) for seed, h in ((1, heads), (2, kv_heads), (3, kv_heads)))
    v[35, 0, 3] = bad            # inside the last, partial block of the first sequence
    v[40 + 90, 1, dim - 1] = bad  # inside a block that the rows before it share
    v[40 + 199, 0, 0] = bad      # the last key, which the rows past it re-read
    v[240, 1, 5] = bad           # the only key of its sequence
    k[40 + 150, 0] = NAN         # a key of its own: hidden scores weigh nothing
    out, lse = torch.full_like(q, 7.0).cuda(), torch.full((tokens, heads), 7.0, device="cuda")
    index = lambda values: torch.tensor(values, dtype=torch.int32, device="cuda")
    config = A.RaggedKvPrefillAttentionConfig.contiguous(len(lens), tokens, tokens, heads, kv_heads, dim, causal, scale)
    call = A.ragged_kv_prefill_attention_bf16 if dtype == torch.bfloat16 else A.ragged_kv_prefill_attention_f16
    call(None, out, lse, q.cuda(), k.cuda(), v.cuda(), index(lens), index(lens), index(offsets), config)
    first = [start for start, n in zip(offsets, lens) for _ in range(n)]
    end = [start + (i + 1 if causal else n) for start, n in zip(offsets, lens) for i in range(n)]
    same(out, visible_only(q, k, v, first, end, scale), dtype)


@pytest.mark.parametrize("dim", [32, 64, 96, 128])
@pytest.mark.parametrize("batch,heads,length,window", [
    (1, 6, 200, 0), (1, 6, 200, 17),       # 16-row tiles, whose keys several waves share
    (14, 64, 65, 0), (14, 64, 65, 9),      # 32-row tiles, two waves a tile
    (70, 64, 30, 0),                       # 32-row tiles from head_dim 64 on, a wave a tile
])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("bad", [INF, NAN])
def test_dense_f32(dim, batch, heads, length, window, causal, bad):
    scale = dim ** -0.5
    q, k, v = (draw(seed, batch, length, h, dim) for seed, h in ((1, heads), (2, heads // 2), (3, heads // 2)))
    v[:, length // 2, 0, 3] = bad           # inside a block that the rows before it share
    v[:, length - 1, -1, dim - 1] = -bad    # the last key, which the keys past it re-read
    k[:, length // 2 + 3, -1] = NAN
    out = torch.full_like(q, 7.0).cuda()
    config = A.FmhaPrefillConfig.contiguous(batch, length, length, heads, heads // 2, dim, scale, causal)
    A.softcapped_window_attention_f32(None, out, q.cuda(), k.cuda(), v.cuda(), A.SoftcappedWindowAttentionConfig(config, window, None))
    first = [max(0, i - window) if window else 0 for i in range(length)]
    end = [min(length, i + 1 if causal else i + window + 1 if window else length) for i in range(length)]
    for b, of in ((0, slice(0, 2)), (batch - 1, slice(heads - 2, heads))):
        kv = slice(of.start // 2, of.start // 2 + 1)
        same(out[b, :, of], visible_only(q[b, :, of], k[b, :, kv], v[b, :, kv], first, end, scale), torch.float32)


@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("lengths", [None, [70, 150]])
@pytest.mark.parametrize("bad", [INF, NAN])
def test_dense_f32_of_the_tensor_surface(dim, lengths, bad):
    # scaled_dot_product_attention of f32 tensors: a window, and keys past a batch entry's own count
    batch, heads, length, window = 2, 8, 150, 40
    q, k, v = (draw(seed, batch, h, length, dim) for seed, h in ((4, heads), (5, heads), (6, heads)))
    v[:, 0, 60, 1] = bad
    if lengths is None:
        out = neural.attend(q.cuda(), k.cuda(), v.cuda(), None, None, neural.AttentionOptions(causal=True, window=window))
    else:
        v[0, :, lengths[0]:] = bad
        out = neural.attend_padded(q.cuda(), k.cuda(), v.cuda(), torch.tensor(lengths, dtype=torch.int32, device="cuda"))
    for b in range(batch):
        first = [max(0, i + 1 - window) if lengths is None else 0 for i in range(length)]
        end = [i + 1 if lengths is None else lengths[b] for i in range(length)]
        rows = [t[b].transpose(0, 1) for t in (q, k, v)]
        same(out[b].transpose(0, 1), visible_only(*rows, first, end, dim ** -0.5), torch.float32)


def paged(values, dtype, heads, kv_heads, dim, page, sequences, splits, window, key_values=None):
    """The paged op over a cache whose places without a key hold `values` and whose keys are the same whatever that is."""
    counts = [-(-keys // page) for _, keys in sequences]
    pages, tokens = sum(counts), sum(queries for queries, _ in sequences)
    caches = []
    for seed in (1, 2):
        cache, at = torch.full((pages + 1, page, kv_heads, dim), values), 0
        for s, ((_, keys), count) in enumerate(zip(sequences, counts)):
            rows = draw(10 * s + seed, keys, kv_heads, dim)
            hidden = 0 if window is None else max(0, keys - sequences[s][0] + 1 - window) // 64 * 64  # whole tiles that no row sees
            rows[:hidden] = values
            cache[at:at + count].view(count * page, kv_heads, dim)[:keys] = rows
            at += count
        caches.append(cache.to(dtype))
    for where, value in (key_values or {}).items():
        cache, sequence, key, kv_head = where
        place = sum(counts[:sequence]) * page + key
        caches[cache].view(-1, kv_heads, dim)[place, kv_head, dim // 2] = value
    index = lambda numbers: torch.tensor(numbers, dtype=torch.int32, device="cuda")
    sums = lambda numbers: [sum(numbers[:i]) for i in range(len(numbers) + 1)]
    paging = neural.Paging(index(sums([queries for queries, _ in sequences])), index(sums(counts)), index(list(range(pages))),
                           index([keys - (count - 1) * page for (_, keys), count in zip(sequences, counts)]))
    neural._native.lib().singe_hip_set_paged_attention_splits(splits)
    try:
        return neural.paged_attention(draw(3, tokens, heads, dim).to(dtype).cuda(), caches[0].cuda(), caches[1].cuda(), paging,
                                      neural.AttentionOptions(causal=True, window=window))
    finally:
        neural._native.lib().singe_hip_set_paged_attention_splits(0)


# (one to sixteen rows a kv head, which have a loop of their own from pages of sixteen keys up, beside row tiles)
PAGED = [(1, 5), (2, 130), (1, 16), (40, 77), (1, 700), (2, 333), (1, 81)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("heads,kv_heads,dim,page", [(8, 2, 128, 16), (16, 2, 64, 32), (6, 3, 96, 64), (4, 1, 32, 16), (8, 2, 128, 12), (8, 2, 80, 16)])
@pytest.mark.parametrize("splits", [0, 3])
@pytest.mark.parametrize("window", [None, 70])
def test_paged_places_that_belong_to_no_key(dtype, heads, kv_heads, dim, page, splits, window):
    clean, clean_lse = paged(0.0, dtype, heads, kv_heads, dim, page, PAGED, splits, window)
    out, lse = paged(NAN, dtype, heads, kv_heads, dim, page, PAGED, splits, window)
    assert torch.equal(out, clean) and torch.equal(lse, clean_lse) and out.isfinite().all() and lse.isfinite().all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("heads,kv_heads,dim", [(8, 2, 128), (16, 2, 64), (4, 1, 32)])
@pytest.mark.parametrize("splits,cache,bad", [(0, 0, NAN), (0, 1, NAN), (0, 1, INF), (0, 1, -INF), (3, 1, NAN), (3, 1, INF)])
def test_paged_keys_reach_the_rows_that_see_them(dtype, heads, kv_heads, dim, splits, cache, bad):
    # (a share whose sum is a NaN has a log-sum-exp of -inf and is left out by the merge: scores without shares only)
    # keys that every row of their sequence sees: of the last sequences' first and last groups, and of one with row tiles
    places = {(cache, 4, 3, 0): bad, (cache, 6, 79, kv_head := kv_heads - 1): bad, (cache, 3, 20, kv_head): bad}
    clean, _ = paged(0.0, dtype, heads, kv_heads, dim, 16, PAGED, splits, None)
    out, _ = paged(0.0, dtype, heads, kv_heads, dim, 16, PAGED, splits, None, places)
    reached = torch.zeros_like(out, dtype=torch.bool)
    group, start = heads // kv_heads, [sum(queries for queries, _ in PAGED[:s]) for s in range(len(PAGED))]
    for (_, sequence, _, head) in places:
        rows = slice(start[sequence], start[sequence] + PAGED[sequence][0])
        of = slice(head * group, (head + 1) * group)
        reached[rows, of, dim // 2 if cache == 1 else slice(None)] = True
    assert torch.equal(out[~reached], clean[~reached])
    assert (out[reached].isnan() if math.isnan(bad) else out[reached] == bad).all()


# (queries, keys) of a decode step that runs in one launch: sequences that are shared out over several workgroups and ones that
# are not, one without tokens, and one of two tokens, whose first does not see the last key
STEP = [(1, 3100), (1, 50), (0, 20), (2, 1000), (1, 700)]


def decode_step(dtype, heads, kv_heads, dim, scratch, bad):
    """The paged op over STEP with `bad` = {(cache, sequence, key, kv head): value of one element}: what it gives, and what
    float64 gives over the keys that each row sees."""
    page, scale = 16, dim ** -0.5
    counts = [-(-keys // page) for _, keys in STEP]
    tokens, starts = sum(queries for queries, _ in STEP), [sum(counts[:s]) * page for s in range(len(STEP))]
    q = draw(1, tokens, heads, dim).to(dtype)
    caches = [draw(seed, sum(counts) * page, kv_heads, dim).to(dtype) for seed in (2, 3)]
    for (cache, sequence, key, kv_head), value in bad.items():
        caches[cache][starts[sequence] + key, kv_head, dim // 2] = value
    index = lambda numbers: torch.tensor(numbers, dtype=torch.int32, device="cuda")
    sums = lambda numbers: [sum(numbers[:i]) for i in range(len(numbers) + 1)]
    paging = neural.Paging(index(sums([queries for queries, _ in STEP])), index(sums(counts)), index(list(range(sum(counts)))),
                           index([keys - (count - 1) * page for (_, keys), count in zip(STEP, counts)]))
    out, lse = neural.paged_attention(q.cuda(), *(cache.view(-1, page, kv_heads, dim).cuda() for cache in caches), paging,
                                      neural.AttentionOptions(causal=True, scale=scale), scratch=scratch)
    first = [start for (queries, _), start in zip(STEP, starts) for _ in range(queries)]
    end = [start + keys - queries + 1 + i for (queries, keys), start in zip(STEP, starts) for i in range(queries)]
    scores = [torch.einsum("hd,khd->hk", q[t].double(), caches[0][f:e].double().repeat_interleave(heads // kv_heads, 1)) * scale
              for t, (f, e) in enumerate(zip(first, end))]
    want_lse = torch.stack([torch.logsumexp(s, -1) / math.log(2.0) for s in scores])
    # (torch's logsumexp of scores with an infinity is that infinity; the softmax over them is not a number)
    want_lse[torch.stack([(s == INF).any(-1) for s in scores])] = NAN
    return out, lse.double().cpu(), visible_only(q, *caches, first, end, scale), want_lse


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("heads,kv_heads,dim", [(32, 8, 128), (16, 1, 64), (8, 2, 96), (6, 2, 32)])
@pytest.mark.parametrize("scratch", [True, False])
@pytest.mark.parametrize("cache,bad", [(0, NAN), (0, INF), (0, -INF), (1, NAN), (1, INF), (1, -INF)])
def test_a_decode_step_gives_every_row_what_its_keys_hold(dtype, heads, kv_heads, dim, scratch, cache, bad):
    # in the first and in a middle share of a sequence, at its last key, in ones that are not shared out
    # (and at a key that the second of two tokens sees, not the first)
    places = {(cache, 0, 3, 0): bad, (cache, 0, 1700, kv_heads - 1): bad, (cache, 1, 49, 0): bad, (cache, 3, 999, 0): bad, (cache, 4, 64, kv_heads - 1): bad}
    out, lse, want, want_lse = decode_step(dtype, heads, kv_heads, dim, scratch, places)
    same(out, want, dtype)
    assert (lse.isnan() == want_lse.isnan()).all() and ((lse - want_lse).abs()[~want_lse.isnan()] <= 2e-3).all()
