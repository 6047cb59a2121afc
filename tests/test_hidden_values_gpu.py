"""An infinity or a NaN among the values of a key: it reaches the rows that see the key and no others, also where a matrix
product weighs the values of hidden keys by zero.  The ops whose reference walks only a row's own keys: packed 16-bit
prefill and dense f32 attention.

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
