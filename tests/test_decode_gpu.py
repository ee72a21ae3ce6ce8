"""GPU parity of the kernel for few query rows (attn_decode.hip): one or two 32-row tiles that hold the rows of all query
heads of a K/V head.  Sizes at the edges of its tiles: 1, 31..33, 63..64 rows; key counts around 32, 64 and 128 and runs that
end in a ragged tile.  Gates: those of the other attention tests (SageAttention: cosine 0.9995, 2e-2; dense: the
reference's rule, twice the deviation of the 16-bit closed form)."""
import pytest
import torch

from oracle import c_oracle as C
from oracle import flash_oracle as FO
from oracle import sage_oracle as O

pytestmark = pytest.mark.gpu

# (B, Hq, Hkv, M): rows per K/V head = Hq / Hkv * M
ROWS = [(2, 2, 2, 1), (1, 8, 2, 1), (1, 3, 1, 11), (1, 2, 2, 31), (3, 1, 1, 32), (1, 32, 1, 1), (1, 6, 2, 11), (1, 4, 2, 32), (2, 8, 1, 8)]
KEYS = [1, 33, 64, 127, 1000, 4128]


def _qkv(b, hq, hkv, m, n, d, dtype, layout="HND"):
    g = torch.Generator().manual_seed(31)
    q, k, v = (torch.randn(b, h, length, d, generator=g).to(dtype) for h, length in ((hq, m), (hkv, n), (hkv, n)))
    return (q, k, v) if layout == "HND" else tuple(t.transpose(1, 2).contiguous() for t in (q, k, v))


@pytest.mark.parametrize("n", KEYS)
@pytest.mark.parametrize("b,hq,hkv,m", ROWS)
def test_sage_few_rows(b, hq, hkv, m, n, gpu_device):
    from flag_attn import sage_attention as sa

    d, dtype = (64, torch.float16) if (m + n) % 2 else (128, torch.bfloat16)
    layout = "NHD" if hq == 8 else "HND"
    q, k, v = _qkv(b, hq, hkv, m, n, d, dtype, layout)
    q8, qs, k8, ks = O.per_block_int8(q, k, tensor_layout=layout)
    for causal in (False, True):
        if causal and m > n:  # (served as a mask tensor, not by this kernel)
            continue
        for out_dtype in (dtype, torch.float32):
            o, lse = sa.sage_attention(*(t.to(gpu_device) for t in (q8, k8, v, qs, ks)), tensor_layout=layout, causal=causal,
                                       output_dtype=out_dtype, return_lse=True)
            expected, expected_lse = C.attention_blockwise(q8, k8, v, qs, ks, layout, causal=causal)
            cos, _, max_abs = O.accuracy_metrics(o.float().cpu(), expected)
            assert cos >= 0.9995 and max_abs <= 2e-2, (causal, out_dtype, cos, max_abs)
            torch.testing.assert_close(lse.cpu(), expected_lse, atol=2e-3, rtol=1e-4)


@pytest.mark.parametrize("n", KEYS)
@pytest.mark.parametrize("b,hq,hkv,m", ROWS)
def test_dense_few_rows(b, hq, hkv, m, n, gpu_device):
    import flag_attn

    d, dtype = (64, torch.bfloat16) if (m + n) % 2 else (128, torch.float16)
    q, k, v = _qkv(b, hq, hkv, m, n, d, dtype)
    for causal in (False, True):  # (M > N under the causal flag: the first queries see no key)
        o, L, *_ = flag_attn.flash_attention(q.to(gpu_device), k.to(gpu_device), v.to(gpu_device), causal, return_log_normalizer=True)
        o_ref, L_ref = FO.attention(q, k, v, causal, return_log_normalizer=True, upcast=True)
        yard = FO.max_diff(FO.attention(q, k, v, causal, upcast=False), o_ref)
        assert FO.max_diff(o.cpu(), o_ref) <= 2 * yard + 1e-5, (causal, FO.max_diff(o.cpu(), o_ref), yard)
        inf = torch.isinf(L_ref)
        assert torch.equal(torch.isinf(L.cpu()), inf)
        torch.testing.assert_close(L.cpu()[~inf], L_ref[~inf], atol=2e-3, rtol=2e-4)


def test_row_maximum_that_rises_from_run_to_run(gpu_device):
    """Scores that grow along the keys by thousands of log2 units: every tile of a run, and every run, moves the maximum."""
    from flag_attn import sage_attention as sa

    q, k, v = _qkv(1, 8, 2, 1, 2048, 128, torch.float16)
    q8, qs, k8, ks = O.per_block_int8(q, k)
    ks = ks * torch.logspace(0, 3, ks.shape[-1])
    o, lse = sa.sage_attention(*(t.to(gpu_device) for t in (q8, k8, v, qs, ks)), return_lse=True)
    expected, expected_lse = C.attention_blockwise(q8, k8, v, qs, ks)
    cos, _, max_abs = O.accuracy_metrics(o.float().cpu(), expected)
    assert cos >= 0.9995 and max_abs <= 2e-2
    torch.testing.assert_close(lse.cpu(), expected_lse, atol=2e-3, rtol=1e-4)
