"""How the dense, paged and latent kernels cut their work (query tiles to a workgroup, shares of the keys, blocks a window passes
over) against f32 on the CPU, at the edges of tiles, blocks and shares.

Tolerance: a bf16 weight and a bf16 output are each rounded once (2^-9 of the value); outputs of N(0, 1) values stay below
about 4, so single elements are within 4 * 2 * 2^-9 = 1.6e-2."""
import math

import numpy as np
import pytest
import torch

import oracle
from singe_amd import neural

pytestmark = pytest.mark.gpu

TOL = 2e-2


def _inputs(seed, batch, heads, kv_heads, lq, lk, dim, dtype=torch.bfloat16):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    shape = lambda h, n: torch.randn((batch, h, n, dim), generator=gen, device="cuda").to(dtype)
    return shape(heads, lq), shape(kv_heads, lk), shape(kv_heads, lk)


def _reference(q, k, v, causal, window=None, lengths=None, sinks=None):
    """The dense op in f32 on the CPU; a row that sees no key is zero."""
    q, k, v = q.float().cpu(), k.float().cpu(), v.float().cpu()
    group = q.shape[1] // k.shape[1]
    k, v = k.repeat_interleave(group, 1), v.repeat_interleave(group, 1)
    scores = q @ k.transpose(-1, -2).contiguous() / math.sqrt(q.shape[-1])
    i, j = torch.arange(q.shape[2])[:, None], torch.arange(k.shape[2])[None, :]
    hidden = torch.zeros((1, 1, q.shape[2], k.shape[2]), dtype=torch.bool)
    if causal:
        hidden = hidden | (j > i)
    if window is not None:
        hidden = hidden | (j + window <= i)
    if lengths is not None:
        hidden = hidden | (j[None, None] >= torch.tensor(lengths)[:, None, None, None])
    scores = scores.masked_fill(hidden, -math.inf)
    if sinks is not None:
        sink = sinks.float().cpu()[None, :, None, None].expand(scores.shape[0], -1, scores.shape[2], 1)
        return torch.softmax(torch.cat([scores, sink], -1), -1)[..., :-1] @ v
    return torch.nan_to_num(torch.softmax(scores, -1), 0.0) @ v


@pytest.mark.parametrize("dim", [16, 48, 64, 80, 96, 112, 128])
@pytest.mark.parametrize("batch,heads,kv_heads,length,causal,lengths", [
    (1, 8, 2, 300, True, None),                # three tiles, one to a workgroup
    (1, 2, 1, 1100, True, None),               # shares of the keys, an odd count of them for the short rows
    (3, 5, 5, 257, False, [257, 1, 130]),      # a last tile of one row, a batch entry of one key
    (2, 3, 3, 1200, False, [0, 1199]),         # shares, an entry without keys
])
def test_small_dense_launches(dim, batch, heads, kv_heads, length, causal, lengths):
    q, k, v = _inputs(dim + length, batch, heads, kv_heads, length, length, dim)
    if lengths is None:
        out = neural.scaled_dot_product_attention(q, k, v, causal=causal)
    else:
        out = neural.attend_padded(q, k, v, torch.tensor(lengths, dtype=torch.int32, device="cuda"))
    gap = (out.float().cpu() - _reference(q, k, v, causal, lengths=lengths)).abs().max().item()
    assert gap <= TOL, gap


@pytest.mark.parametrize("window", [0, 1, 31, 32, 33, 96, 129, 700])
@pytest.mark.parametrize("dim,length,causal,sinks", [(64, 700, True, True), (128, 333, True, False), (64, 257, False, False), (48, 130, True, True)])
def test_windows_at_block_edges(window, dim, length, causal, sinks):
    q, k, v = _inputs(window + dim, 2, 4, 2, length, length, dim)
    logits = torch.linspace(-1.0, 2.0, 4, device="cuda").to(q.dtype) if sinks else None
    out = neural.attend(q, k, v, None, logits, neural.AttentionOptions(causal=causal, window=window))
    gap = (out.float().cpu() - _reference(q, k, v, causal, window=window, sinks=logits)).abs().max().item()
    assert gap <= TOL, gap


@pytest.mark.parametrize("chunks,chunk,decoding", [
    (2, 512, 62),   # half a whole 256-row tile a sequence: 128-row tiles
    (4, 256, 21),   # 32 tiles, 25 sequences: 256-row tiles
    (4, 256, 22),
    (2, 512, 56),   # 33 tiles, 58 sequences (9 / 16 and a bit): the last on 256-row tiles
    (2, 512, 57),   # 59 sequences: the first on 128-row tiles
    (1, 1025, 62),  # 1024 tokens more than sequences: still 128-row tiles
    (1, 1026, 62),  # 1025: 256-row tiles
])
def test_mixed_steps_either_side_of_the_tile_choice(chunks, chunk, decoding):
    heads, kv_heads, dim, page = 64, 8, 128, 16
    generator = torch.Generator().manual_seed(chunks + decoding)
    new = [chunk] * chunks + [1] * decoding
    keys = [count + int(torch.randint(0, 700, (1,), generator=generator)) for count in new]
    counts = [(k + page - 1) // page for k in keys]
    table = torch.randperm(sum(counts), generator=generator)
    offsets = lambda values: torch.tensor([0] + list(np.cumsum(values)), dtype=torch.int64).cuda()
    last = torch.tensor([k - (c - 1) * page for k, c in zip(keys, counts)], dtype=torch.int64)
    paging = neural.Paging(offsets(new), offsets(counts), table.cuda(), last.cuda())
    draw = lambda *shape: torch.randn(shape, generator=generator).to(torch.bfloat16)
    q, kc, vc = draw(sum(new), heads, dim), draw(sum(counts), page, kv_heads, dim), draw(sum(counts), page, kv_heads, dim)
    out, _ = neural.paged_attention(q.cuda(), kc.cuda(), vc.cuda(), paging, neural.AttentionOptions(causal=True))
    out, at, first = out.float().cpu(), 0, 0
    for count, k, pages in zip(new, keys, counts):
        held = table[first:first + pages]
        rows = q[at:at + count].transpose(0, 1)[None]
        key, value = (c[held].reshape(-1, kv_heads, dim)[:k].transpose(0, 1)[None] for c in (kc, vc))
        # the reference's own mask starts at the first key; a chunk's rows are the last of a causal sequence
        padded = torch.cat([torch.zeros((1, heads, k - count, dim), dtype=rows.dtype), rows], 2)[:, ::7]
        group = heads // kv_heads
        want = _reference(padded, key.repeat_interleave(group, 1)[:, ::7], value.repeat_interleave(group, 1)[:, ::7], True)
        gap = (out[at:at + count, ::7].transpose(0, 1) - want[0, :, k - count:]).abs().max().item()
        assert gap <= TOL, gap
        at, first = at + count, first + pages
