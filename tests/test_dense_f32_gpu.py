"""Dense f32 attention on the GPU against the CPU oracle, through the C ABI.  f32 tolerance: 1e-4."""
import numpy as np
import pytest
import torch

import oracle
from singe_amd import neural
from singe_amd.kernel import attention as A

pytestmark = pytest.mark.gpu

TOL = 1e-4


def test_dense_causal_f32_anchor():
    # batch 1, 8 heads, head_dim 64, seq 512, f32 N(0, 1), scale 1/8, causal, [B, H, L, D] order
    batch, heads, length, dim = 1, 8, 512, 64
    gen = torch.Generator(device="cuda")
    gen.manual_seed(0x51A6E + 1)
    q, k, v = (torch.randn((batch, heads, length, dim), generator=gen, device="cuda") for _ in range(3))
    out = torch.full_like(q, float("nan"))
    config = A.bhsd_config(batch, heads, heads, length, length, dim, 0.125, True)
    A.softcapped_window_attention_f32(None, out, q, k, v, A.SoftcappedWindowAttentionConfig(config))
    torch.cuda.synchronize()
    want = oracle.softcapped_window_attention_f32(q.cpu().numpy(), k.cpu().numpy(), v.cpu().numpy(), batch=batch,
                                                  query_len=length, key_len=length, heads=heads, kv_heads=heads,
                                                  head_dim=dim, scale=0.125, causal=True, threads=8)
    other = oracle.scaled_dot_product_attention_f32(q.cpu().numpy(), k.cpu().numpy(), v.cpu().numpy(), scale=0.125,
                                                    causal=True, threads=8)
    assert np.array_equal(want, other)  # the two CPU surfaces agree bit for bit on this shape
    gap = np.abs(out.cpu().numpy() - want)
    assert gap.max() <= TOL, gap.max()
    out2 = torch.empty_like(q)
    A.fmha_prefill_f32(None, out2, q, k, v, config)
    torch.cuda.synchronize()
    assert torch.equal(out, out2)


@pytest.mark.parametrize("dim", [4, 16, 33, 64, 96, 128, 200])
@pytest.mark.parametrize("causal", [False, True])
def test_prefill_f32_bshd_with_lse(dim, causal):
    batch, lq, lk, heads, kv_heads = 2, 37, 130, 4, 2
    gen = torch.Generator(device="cuda")
    gen.manual_seed(dim)
    q = torch.randn((batch, lq, heads, dim), generator=gen, device="cuda")
    k = torch.randn((batch, lk, kv_heads, dim), generator=gen, device="cuda")
    v = torch.randn((batch, lk, kv_heads, dim), generator=gen, device="cuda")
    out = torch.full_like(q, float("nan"))
    lse = torch.full((batch, heads, lq), float("nan"), device="cuda")
    scale = float(dim) ** -0.5
    A.fmha_prefill_lse_f32(None, out, lse, q, k, v, A.FmhaPrefillConfig.contiguous(batch, lq, lk, heads, kv_heads, dim, scale, causal))
    torch.cuda.synchronize()
    want, want_lse = oracle.fmha_prefill_lse_f32(q.cpu().numpy(), k.cpu().numpy(), v.cpu().numpy(), batch=batch,
                                                 query_len=lq, key_len=lk, heads=heads, kv_heads=kv_heads,
                                                 head_dim=dim, scale=scale, causal=causal, threads=4)
    assert np.abs(out.cpu().numpy() - want).max() <= TOL
    assert np.abs(lse.cpu().numpy() - want_lse).max() <= TOL


@pytest.mark.parametrize("window,cap", [(0, 30.0), (5, None), (16, 2.5)])
def test_softcapped_window_f32(window, cap):
    batch, heads, kv_heads, lq, lk, dim = 1, 4, 2, 70, 70, 32
    gen = torch.Generator(device="cuda")
    gen.manual_seed(7)
    q = torch.randn((batch, heads, lq, dim), generator=gen, device="cuda")
    k = torch.randn((batch, kv_heads, lk, dim), generator=gen, device="cuda")
    v = torch.randn((batch, kv_heads, lk, dim), generator=gen, device="cuda")
    out = torch.full_like(q, float("nan"))
    config = A.bhsd_config(batch, heads, kv_heads, lq, lk, dim, 0.3, True)
    A.softcapped_window_attention_f32(None, out, q, k, v, A.SoftcappedWindowAttentionConfig(config, window, cap))
    torch.cuda.synchronize()
    want = oracle.softcapped_window_attention_f32(q.cpu().numpy(), k.cpu().numpy(), v.cpu().numpy(), batch=batch,
                                                  query_len=lq, key_len=lk, heads=heads, kv_heads=kv_heads, head_dim=dim,
                                                  scale=0.3, causal=True, window_size=window, soft_cap=cap)
    assert np.abs(out.cpu().numpy() - want).max() <= TOL


@pytest.mark.parametrize("cap", [0.0, -2.5, float("inf"), float("nan")])
def test_softcapped_window_f32_refuses_a_cap_that_is_not_positive_and_finite(cap):
    # validate_softcapped_window_attention_config: a cap must be finite and above zero, and is looked at before the window
    from singe_amd import error
    batch, heads, lq, dim = 1, 2, 8, 32
    q = torch.zeros((batch, heads, lq, dim), device="cuda")
    out = torch.zeros_like(q)
    config = A.bhsd_config(batch, heads, heads, lq, lq, dim, 0.3, True)
    with pytest.raises(error.InvalidLength):
        A.softcapped_window_attention_f32(None, out, q, q, q, A.SoftcappedWindowAttentionConfig(config, 2 ** 40, cap))


@pytest.mark.parametrize("dim", [32, 64, 96, 128])
@pytest.mark.parametrize("batch,heads,kv_heads,lq,lk,causal,window", [
    (1, 3, 1, 1, 1, True, 0), (1, 2, 2, 15, 33, False, 0), (2, 2, 1, 17, 16, True, 0), (1, 4, 2, 65, 257, True, 0),  # 16-row tiles
    (1, 2, 1, 100, 90, True, 7), (1, 2, 2, 70, 130, False, 31), (1, 1, 1, 48, 32, False, 3),                        # windows
    (1, 1, 1, 100, 20, True, 9),                                                                                 # rows that see no key
    (3, 64, 32, 33, 70, True, 0), (2, 100, 50, 95, 65, False, 0), (11, 64, 64, 32, 40, True, 5),                    # 32-row tiles
])
def test_prefill_f32_on_the_matrix_cores(dim, batch, heads, kv_heads, lq, lk, causal, window):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(dim + lq)
    q, k, v = (torch.randn((batch, length, h, dim), generator=gen, device="cuda") for length, h in ((lq, heads), (lk, kv_heads), (lk, kv_heads)))
    out = torch.full_like(q, float("nan"))
    config = A.FmhaPrefillConfig.contiguous(batch, lq, lk, heads, kv_heads, dim, -0.2 if window == 31 else dim ** -0.5, causal)
    A.softcapped_window_attention_f32(None, out, q, k, v, A.SoftcappedWindowAttentionConfig(config, window, None))
    torch.cuda.synchronize()
    bhsd = lambda t: np.ascontiguousarray(t.cpu().numpy().transpose(0, 2, 1, 3))
    want = oracle.softcapped_window_attention_f32(bhsd(q), bhsd(k), bhsd(v), batch=batch, query_len=lq, key_len=lk, heads=heads,
                                                  kv_heads=kv_heads, head_dim=dim, scale=config.scale, causal=causal, window_size=window)
    assert np.abs(bhsd(out) - want.reshape(batch, heads, lq, dim)).max() <= TOL
    if window == 0:
        lse = torch.full((batch, heads, lq), float("nan"), device="cuda")
        again = torch.empty_like(out)
        A.fmha_prefill_lse_f32(None, again, lse, q, k, v, config)
        torch.cuda.synchronize()
        _, want_lse = oracle.fmha_prefill_lse_f32(q.cpu().numpy(), k.cpu().numpy(), v.cpu().numpy(), batch=batch, query_len=lq, key_len=lk,
                                                  heads=heads, kv_heads=kv_heads, head_dim=dim, scale=config.scale, causal=causal, threads=4)
        assert torch.equal(out, again) and np.abs(lse.cpu().numpy() - want_lse).max() <= TOL


@pytest.mark.parametrize("window,lengths", [(None, [70, 0, 33]), (5, None), (1, [1, 70, 69])])
@pytest.mark.parametrize("causal", [False, True])
def test_dense_op_f32_on_the_matrix_cores(window, lengths, causal):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(5)
    q, k, v = (torch.randn((3, h, length, 64), generator=gen, device="cuda") for h, length in ((4, 41), (2, 70), (2, 70)))
    options = neural.AttentionOptions(causal=causal, window=window)
    counts = None if lengths is None else torch.tensor(lengths, dtype=torch.int32, device="cuda")
    out = neural.attend(q, k, v, options=options) if counts is None else neural.attend_padded(q, k, v, counts, options)
    torch.cuda.synchronize()
    want = oracle.scaled_dot_product_attention_f32(q.cpu().numpy(), k.cpu().numpy(), v.cpu().numpy(), scale=0.125, causal=causal,
                                                   window=window, key_lengths=lengths)
    assert np.abs(out.cpu().numpy() - want).max() <= TOL


@pytest.mark.parametrize("dim,batch,heads,length,causal,bound", [
    (32, 1, 8, 512, True, 1.40e-7), (64, 1, 8, 512, True, 1.35e-7), (128, 1, 8, 512, True, 1.45e-7),           # 16-row tiles
    (64, 4, 12, 1024, False, 2.05e-7), (96, 4, 12, 1024, False, 2.2e-7), (128, 4, 12, 1024, False, 2.15e-7),   # 32-row tiles
])
def test_matrix_core_sums_are_as_exact_as_the_row_kernels(dim, batch, heads, length, causal, bound):
    # Against float64, relative to the norm.  The row kernel's per-lane sums (head_dim 96: those of the kernel with a wave a
    # row) measured 1.30, 1.23, 1.34, 2.07, 3.7 and 2.2e-7 here; a single chain of products a score and a single one a row's
    # values measured 1.9, 2.4, 3.1, 4.2, 5.5 and 5.8e-7.
    gen = torch.Generator(device="cuda")
    gen.manual_seed(dim)
    q, k, v = (torch.randn((batch, heads, length, dim), generator=gen, device="cuda") for _ in range(3))
    out = torch.full_like(q, float("nan"))
    A.fmha_prefill_f32(None, out, q, k, v, A.bhsd_config(batch, heads, heads, length, length, dim, dim ** -0.5, causal))
    q, k, v, out = (t[-1, :6].double().cpu() for t in (q, k, v, out))
    scores = q @ k.transpose(1, 2).contiguous() * dim ** -0.5
    if causal:
        scores = scores.masked_fill(torch.ones(length, length).triu(1).bool(), -float("inf"))
    want = torch.softmax(scores, -1) @ v
    assert ((out - want).norm() / want.norm()).item() <= bound


@pytest.mark.parametrize("dim", [64, 96, 128])
@pytest.mark.parametrize("batch,heads,lq,lk,causal,window", [
    (32, 64, 33, 70, True, 0),       # a wave a tile (two at head_dim 64: 4096 tiles and more are one), a last tile of one row
    (64, 64, 63, 45, False, 0),
    (90, 64, 20, 31, False, 0),      # a single block of keys
    (6, 32, 33, 100, True, 0),       # four waves a tile, a block each
    (6, 32, 33, 257, False, 0),      # eight waves a tile at head_dim 64, four above; a last block of one key
    (6, 32, 40, 321, False, 90),
    (3, 64, 31, 200, False, 0),      # seven blocks: one of eight waves without any
])
def test_thirty_two_row_tiles_and_their_waves(dim, batch, heads, lq, lk, causal, window):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(dim + lq)
    q, k, v = (torch.randn((batch, h, n, dim), generator=gen, device="cuda") for h, n in ((heads, lq), (heads // 2, lk), (heads // 2, lk)))
    out = torch.full_like(q, float("nan"))
    config = A.bhsd_config(batch, heads, heads // 2, lq, lk, dim, dim ** -0.5, causal)
    lse = None
    if window:
        A.softcapped_window_attention_f32(None, out, q, k, v, A.SoftcappedWindowAttentionConfig(config, window, None))
    else:
        lse = torch.full((batch, heads, lq), float("nan"), device="cuda")
        A.fmha_prefill_lse_f32(None, out, lse, q, k, v, config)
    assert not out.isnan().any()
    i, j = torch.arange(lq)[:, None], torch.arange(lk)[None, :]
    hidden = (j > i if causal else torch.zeros((lq, lk), dtype=torch.bool)) | ((i - j).abs() > window if window else False)
    for b, h in ((0, 0), (0, heads - 1), (batch // 2, 5), (batch - 1, 0), (batch - 1, heads - 1)):
        rows, keys, values = q[b, h].double().cpu(), k[b, h // 2].double().cpu(), v[b, h // 2].double().cpu()
        scores = (rows @ keys.T * dim ** -0.5).masked_fill(hidden, -float("inf"))
        want = torch.softmax(scores, -1) @ values
        assert (out[b, h].double().cpu() - want).abs().max().item() <= 1e-5   # f32 sums of values up to about 4
        if lse is not None:
            assert (lse[b, h].double().cpu() - torch.logsumexp(scores, -1)).abs().max().item() <= 1e-5
