"""A scale of zero (or one whose logits underflow): every visible key weighs the same and a hidden one nothing, so a row is
the mean of the values it sees.  One case for each route whose kernel hides keys before it scales the scores.

Tolerance: a weight of one is exact, a bf16 mean is rounded once (2^-9 of at most about 4)."""
import math

import pytest
import torch

from singe_amd import neural
from singe_amd.kernel import attention as A

pytestmark = pytest.mark.gpu

TOL = 1e-2
SCALES = [0.0, -0.0, 1e-45]


def draw(seed, *shape):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed)).to(torch.bfloat16).cuda()


def means(values, first, end):
    """[rows, kv_heads, dim]: the mean of values[first[i]:end[i]] for every row i, zero where there is none."""
    values = values.float().cpu()
    return torch.stack([values[f:e].mean(0) if e > f else torch.zeros_like(values[0]) for f, e in zip(first, end)])


def near(out, want, group):
    assert (out.float().cpu() - want.repeat_interleave(group, 1)).abs().max().item() <= TOL


@pytest.mark.parametrize("scale", SCALES)
@pytest.mark.parametrize("length,window", [(130, 33), (300, 1), (77, None)])
@pytest.mark.parametrize("dim", [128, 64])
def test_dense(scale, length, window, dim):
    q, k, v = draw(1, 1, 4, length, dim), draw(2, 1, 2, length, dim), draw(3, 1, 2, length, dim)
    out = neural.attend(q, k, v, None, None, neural.AttentionOptions(scale=scale, causal=True, window=window))
    first = [max(0, i + 1 - window) if window else 0 for i in range(length)]
    near(out[0].transpose(0, 1), means(v[0].transpose(0, 1), first, range(1, length + 1)), 2)


@pytest.mark.parametrize("scale", SCALES)
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("dim", [128, 64])
def test_packed(scale, causal, dim):
    lens = [1, 33, 70, 129]
    tokens, offsets = sum(lens), [0, 1, 34, 104]
    q, k, v = draw(4, tokens, 4, dim), draw(5, tokens, 2, dim), draw(6, tokens, 2, dim)
    out, lse = torch.full_like(q, math.nan), torch.full((tokens, 4), math.nan, device="cuda")
    index = lambda values: torch.tensor(values, dtype=torch.int32, device="cuda")
    config = A.RaggedKvPrefillAttentionConfig.contiguous(len(lens), tokens, tokens, 4, 2, dim, causal, scale)
    A.ragged_kv_prefill_attention_bf16(None, out, lse, q, k, v, index(lens), index(lens), index(offsets), config)
    first = [start for start, n in zip(offsets, lens) for _ in range(n)]
    end = [start + (i + 1 if causal else n) for start, n in zip(offsets, lens) for i in range(n)]
    near(out, means(v, first, end), 2)
    want = torch.tensor([math.log(e - f) for f, e in zip(first, end)])[:, None]
    assert (lse.cpu() - want).abs().max().item() <= 1e-5


@pytest.mark.parametrize("scale", SCALES)
@pytest.mark.parametrize("window", [None, 40])
def test_paged(scale, window):
    page, new, keys, dim = 16, [70, 5, 130], [150, 5, 131], 128
    counts = [(n + page - 1) // page for n in keys]
    table = torch.randperm(sum(counts), generator=torch.Generator().manual_seed(7))
    running = lambda values: torch.tensor([0] + values, dtype=torch.int64).cumsum(0).cuda()
    last = torch.tensor([n - (c - 1) * page for n, c in zip(keys, counts)]).cuda()
    q, kc, vc = draw(8, sum(new), 4, dim), draw(9, sum(counts), page, 2, dim), draw(10, sum(counts), page, 2, dim)
    out, _ = neural.paged_attention(q, kc, vc, neural.Paging(running(new), running(counts), table.cuda(), last),
                                    neural.AttentionOptions(scale=scale, causal=True, window=window))
    at, page_at = 0, 0
    for n, held, c in zip(new, keys, counts):
        value = vc.cpu()[table[page_at:page_at + c]].reshape(-1, 2, dim)[:held]
        end = range(held - n + 1, held + 1)
        near(out[at:at + n], means(value, [max(0, e - window) if window else 0 for e in end], end), 2)
        at, page_at = at + n, page_at + c


@pytest.mark.parametrize("scale", SCALES)
def test_block_table(scale):
    block, lens, dim = 16, [37, 130], 128
    counts = [(n + block - 1) // block for n in lens]
    table = torch.zeros((2, max(counts)), dtype=torch.int32)
    table[0, :counts[0]], table[1, :counts[1]] = torch.arange(counts[0]), torch.arange(counts[0], sum(counts))
    q, kc, vc = draw(11, sum(lens), 4, dim), draw(12, sum(counts), block, 2, dim), draw(13, sum(counts), block, 2, dim)
    out, lse = torch.full_like(q, math.nan), torch.full((sum(lens), 4), math.nan, device="cuda")
    index = lambda values: torch.tensor(values, dtype=torch.int32, device="cuda")
    config = A.PagedKvPrefillAttentionConfig.contiguous(2, sum(lens), 4, 2, dim, block, sum(counts), max(counts), True, scale)
    A.paged_kv_prefill_attention_bf16(None, out, lse, q, kc, vc, index(lens), index(lens), index([0, lens[0]]), table.cuda(), config)
    values = vc.reshape(-1, 2, dim)
    for start, first, n in ((0, 0, lens[0]), (lens[0], counts[0] * block, lens[1])):
        near(out[start:start + n], means(values, [first] * n, [first + i + 1 for i in range(n)]), 2)
