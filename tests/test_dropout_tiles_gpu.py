"""The dropout forward kernel where its own choices change: one, two or four groups of waves per workgroup (by the number of
128-query blocks), tile edges (32 keys, 128 queries), a random stream whose low counter word wraps inside the call, drop
probabilities at the ends of the range.  Rule of the other dropout tests: at most twice the deviation of the 16-bit form."""
import pytest
import torch

from oracle import flash_oracle as FO

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("p,offset", [(0.3, 0), (1e-6, 2 ** 32 - 4096), (0.9, 2 ** 32 - 70000)])
@pytest.mark.parametrize("B,H,Hk,M,N,D,causal", [
    (1, 2, 1, 1, 33, 64, False), (1, 2, 2, 129, 31, 64, True), (2, 3, 3, 127, 128, 128, True),   # four / two groups
    (6, 16, 8, 600, 70, 64, True),     # 480 blocks: two groups
    (6, 16, 16, 800, 65, 64, True),    # 672 blocks: one
    (3, 16, 16, 700, 97, 128, True),   # 288 blocks at head_dim 128: one
    (1, 16, 16, 130, 300, 128, False),
    (1, 24, 8, 1700, 97, 64, True), (1, 20, 20, 1700, 40, 128, True),  # a second round of blocks on some of the CUs
])
def test_dropout_forward_tiles(B, H, Hk, M, N, D, causal, p, offset, gpu_device):
    import flag_attn

    dtype = torch.bfloat16 if (M + D) % 2 else torch.float16
    g = torch.Generator().manual_seed(41)
    q, k, v = (torch.randn(B, h, n, D, generator=g).to(dtype) for h, n in ((H, M), (Hk, N), (Hk, N)))
    dq, dk, dv = (t.to(gpu_device) for t in (q, k, v))
    gen = torch.cuda.default_generators[gpu_device.index or 0]
    gen.manual_seed(99)
    gen.set_offset(offset)
    o, L, _, seed, off = flag_attn.flash_attention(dq, dk, dv, causal, dropout_p=p,
                                                   return_log_normalizer=True, return_seed_offset=True)
    assert (seed, off) == (99, offset)
    mask = flag_attn.testing.recompute_mask(B, H, M, N, p, seed, off, gpu_device).cpu()
    o_ref, L_ref = FO.attention(q, k, v, causal, dropout_p=p, dropout_mask=mask, return_log_normalizer=True, upcast=True)
    yard = FO.max_diff(FO.attention(q, k, v, causal, dropout_p=p, dropout_mask=mask, upcast=False), o_ref)
    got = FO.max_diff(o.cpu(), o_ref)
    assert got <= 2 * yard + 1e-5, (got, yard)
    inf = torch.isinf(L_ref)
    assert torch.equal(torch.isinf(L.cpu()), inf)
    torch.testing.assert_close(L.cpu()[~inf], L_ref[~inf], atol=2e-3, rtol=2e-4)


@pytest.mark.parametrize("B,H,M,N,D,causal", [(1, 2, 129, 200, 64, True), (6, 16, 600, 70, 64, False), (1, 2, 100, 97, 128, False), (3, 16, 700, 97, 128, True)])
@pytest.mark.parametrize("p", [0.3, 0.999])
def test_dropout_forward_keeps_nan(B, H, M, N, D, causal, p, gpu_device):
    """The row sums do not see the dropout mask: a NaN score makes its row NaN, output and log normalizer, also where the
    element is dropped."""
    import flag_attn

    g = torch.Generator().manual_seed(42)
    q, k, v = (torch.randn(B, H, n, D, generator=g).to(torch.float16).to(gpu_device) for n in (M, N, N))
    q[0, 1, M - 2, 3] = float("nan")
    k[B - 1, 0, N // 2, 1] = float("nan")
    o, L, *_ = flag_attn.flash_attention(q, k, v, causal, dropout_p=p, return_log_normalizer=True)
    want = torch.zeros((B, H, M), dtype=torch.bool, device=gpu_device)
    want[0, 1, M - 2] = True
    want[B - 1, 0] = torch.arange(M, device=gpu_device) + (N - M) >= N // 2 if causal else True
    sees = torch.arange(M, device=gpu_device) + (N - M) >= 0 if causal else torch.ones(M, dtype=torch.bool, device=gpu_device)
    assert torch.equal(torch.isnan(L), want) and torch.equal(torch.isneginf(L), ~sees.expand(B, H, M))
    assert torch.equal(torch.isnan(o).all(-1), want) and bool(torch.isfinite(o[~want]).all())


@pytest.mark.parametrize("B,H,M,N,D,causal", [(1, 2, 70, 200, 64, False), (2, 3, 129, 300, 128, True), (6, 16, 1000, 70, 128, True)])
@pytest.mark.parametrize("rise", [0.0, 1.0, -1.0])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_dropout_forward_reference_point(B, H, M, N, D, causal, rise, dtype, gpu_device):
    """Scores whose level rises (falls) by 12 log2 units from one 32-key tile to the next, so that the reference point of a row has to
    move with every tile (stays at the first one); the last shape fills three rounds of 128-query blocks at head_dim 128."""
    import math

    import flag_attn

    g = torch.Generator().manual_seed(43)
    q, k, v = (torch.randn(B, H, n, D, generator=g) for n in (M, N, N))
    q[..., 0] = 4.0
    level = torch.arange(N).div(32, rounding_mode="floor").float() * 12.0 * math.log(2.0) * math.sqrt(D) / 4.0
    k[..., 0] = rise * level
    q, k, v = (t.to(dtype) for t in (q, k, v))
    dq, dk, dv = (t.to(gpu_device) for t in (q, k, v))
    o, L, _, seed, off = flag_attn.flash_attention(dq, dk, dv, causal, dropout_p=0.25, return_log_normalizer=True, return_seed_offset=True)
    mask = flag_attn.testing.recompute_mask(B, H, M, N, 0.25, seed, off, gpu_device).cpu()
    o_ref, L_ref = FO.attention(q, k, v, causal, dropout_p=0.25, dropout_mask=mask, return_log_normalizer=True, upcast=True)
    yard = FO.max_diff(FO.attention(q, k, v, causal, dropout_p=0.25, dropout_mask=mask, upcast=False), o_ref)
    got = FO.max_diff(o.cpu(), o_ref)
    assert got <= 2 * yard + 1e-5, (got, yard)
    inf = torch.isinf(L_ref)
    assert torch.equal(torch.isinf(L.cpu()), inf)
    torch.testing.assert_close(L.cpu()[~inf], L_ref[~inf], atol=2e-3, rtol=2e-4)
