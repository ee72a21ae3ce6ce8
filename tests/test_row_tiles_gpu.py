"""Short calls on the kernel that takes 32 packed query rows per workgroup (plan_row_tiles): against the oracle, at row tiles that
hold several heads of a group or the end of one, ragged keys, both flags, and with the keys split."""
import pytest
import torch

from oracle import c_oracle as C
from oracle import flash_oracle as FO
from oracle import sage_oracle as O

pytestmark = pytest.mark.gpu

# (batch, heads_q, heads_kv, M, N): one tile and a row; rows of three heads in a tile; the last tile with one row; ragged keys;
# the longest of its range with and without a workspace; fewer queries than keys; more (dense: queries that see no key)
SHAPES = [(1, 2, 2, 33, 64), (2, 6, 2, 11, 130), (1, 8, 1, 37, 200), (3, 4, 4, 65, 65), (1, 2, 2, 256, 256), (1, 8, 8, 1000, 1000),
          (1, 4, 2, 100, 600), (1, 1, 1, 3000, 3000), (1, 4, 2, 200, 130)]


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("b,hq,hkv,m,n", SHAPES)
def test_sage(b, hq, hkv, m, n, causal, d, gpu_device):
    from flag_attn import sage_attention as sa

    g = torch.Generator().manual_seed(m + n)
    dt = torch.bfloat16 if m % 2 else torch.float16
    q, k, v = (torch.randn(b, h, x, d, generator=g).to(dt) for h, x in ((hq, m), (hkv, n), (hkv, n)))
    for layout in ("HND", "NHD"):
        if layout == "NHD":
            q, k, v = (t.transpose(1, 2).contiguous() for t in (q, k, v))
        q8, qs, k8, ks = O.per_block_int8(q, k, tensor_layout=layout)
        o, lse = sa.sage_attention(*(t.to(gpu_device) for t in (q8, k8, v, qs, ks)), tensor_layout=layout, causal=causal,
                                   return_lse=True, output_dtype=torch.float32)
        want, want_lse = C.attention_blockwise(q8, k8, v, qs, ks, layout, causal=causal)
        cos, _, max_abs = O.accuracy_metrics(o.cpu(), want)
        assert cos >= 0.9995 and max_abs <= 2e-2
        torch.testing.assert_close(lse.cpu(), want_lse, atol=2e-3, rtol=1e-4)


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("b,hq,hkv,m,n", SHAPES)
def test_dense(b, hq, hkv, m, n, causal, d, gpu_device):
    import flag_attn

    g = torch.Generator().manual_seed(m + n)
    dt = torch.bfloat16 if m % 2 else torch.float16
    q, k, v = (torch.randn(b, h, x, d, generator=g).to(dt) for h, x in ((hq, m), (hkv, n), (hkv, n)))
    o, lse, *_ = flag_attn.flash_attention(q.to(gpu_device), k.to(gpu_device), v.to(gpu_device), causal, return_log_normalizer=True)
    want, want_lse = FO.attention(q, k, v, causal, return_log_normalizer=True)
    own = FO.attention(q, k, v, causal, upcast=False)
    assert FO.max_diff(o.cpu(), want) <= 2 * FO.max_diff(own, want) + 1e-6  # the reference's own rule
    inf = torch.isinf(want_lse)
    assert torch.equal(torch.isinf(lse.cpu()), inf)
    torch.testing.assert_close(lse.cpu()[~inf], want_lse[~inf], atol=2e-3, rtol=1e-4)
    assert not o.cpu()[inf].any()  # a query that sees no key


def test_more_rows_than_one_head_holds_in_scale_blocks(gpu_device):
    """Row tiles across a head's 128-row scale block and across the heads of a group, every row with a scale of its own size."""
    from flag_attn import sage_attention as sa

    g = torch.Generator().manual_seed(3)
    q, k, v = (torch.randn(1, h, 200, 64, generator=g).to(torch.float16) for h in (6, 2, 2))
    q8, qs, k8, ks = O.per_block_int8(q, k)
    qs = qs * torch.logspace(-1, 0.5, qs.numel()).view(qs.shape)
    ks = ks * torch.logspace(0, -1, ks.numel()).view(ks.shape)
    o, _ = sa.sage_attention(*(t.to(gpu_device) for t in (q8, k8, v, qs, ks)), causal=True, output_dtype=torch.float32)
    want, _ = C.attention_blockwise(q8, k8, v, qs, ks, "HND", causal=True)
    torch.testing.assert_close(o.cpu(), want.float(), rtol=2e-2, atol=2e-3)
