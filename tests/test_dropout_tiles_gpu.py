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
    (3, 16, 16, 1300, 1300, 128, True),  # 528 blocks at head_dim 128, rounds of 5 per head, the third one partial; no row without a key
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
    move with every tile (stays at the first one); the last shape takes one group of waves, four rounds of 128-query blocks."""
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


def _running_maximum_forward(q, k, v, mask, p, causal):
    """(what 32-key tiles, exponentials against the row's maximum so far, P rounded to the inputs' type and unrounded row sums give,
    the exact result), everything else in 64 bits."""
    import math

    dt = q.dtype
    s = q.double() @ k.double().transpose(2, 3) / (math.sqrt(q.shape[-1]) * math.log(2.0))
    m, n = s.shape[-2:]
    if causal:
        s = s.masked_fill(torch.ones(m, n, dtype=torch.bool).triu(n - m + 1), -math.inf)
    ref = (torch.softmax(s * math.log(2.0), -1) * mask) @ v.double() / (1.0 - p)
    top = s.unflatten(-1, (n // 32, 32)).amax(-1).cummax(-1).values.repeat_interleave(32, -1)
    weight, later = torch.exp2(s - top), torch.exp2(top - top[..., -1:])
    o = (weight.to(dt).double() * later * mask) @ v.double() / ((weight * later).sum(-1, keepdim=True) * (1.0 - p))
    return o.to(dt).double(), ref


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("H,M,D,causal", [(2, 1024, 64, True), (4, 512, 64, False), (2, 768, 128, True), (40, 1024, 128, False)])
@pytest.mark.parametrize("std", [1.0, 2.0, 4.0])
def test_dropout_forward_error(std, H, M, D, causal, dtype, gpu_device):
    """The error against 64 bits is that of exponentials against the running maximum, whose largest P of a row is exactly 1.  A 2-norm
    over 10^5 and more roundings repeats itself to 0.5 % (seeds); reference points that lag by 2^8 add 2 to 8 % at std 1, 16 % and more at
    2 and 4.  (4 groups of waves, 2 and 1.)"""
    import flag_attn

    g = torch.Generator().manual_seed(44)
    q, k, v = (torch.randn(1, H, M, D, generator=g) for _ in range(3))
    q, k, v = ((x * f).to(dtype) for x, f in ((q, std), (k, 1.0), (v, 1.0)))
    dq, dk, dv = (t.to(gpu_device) for t in (q, k, v))
    o, _, _, seed, off = flag_attn.flash_attention(dq, dk, dv, causal, dropout_p=0.1, return_log_normalizer=True, return_seed_offset=True)
    mask = flag_attn.testing.recompute_mask(1, H, M, M, 0.1, seed, off, gpu_device).cpu()
    heads = slice(0, 4)
    sim, ref = _running_maximum_forward(q[:, heads], k[:, heads], v[:, heads], mask[:, heads], 0.1, causal)
    got, bound = (o.cpu()[:, heads].double() - ref).norm(), 1.02 * (sim - ref).norm()
    assert got <= bound, (float(got / ref.norm()), float(bound / ref.norm()))
