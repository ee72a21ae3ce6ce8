"""Rows that lie further apart than 32-bit byte offsets within a tile reach (2^25 elements and more), or in descending
order: the dropout forward (K and V) and the total attention (Q), against contiguous copies."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _far(x):
    """The rows of x [1, 1, L, D], 2^25 + 8 elements apart."""
    step = 2 ** 25 + 8
    big = torch.empty(x.shape[2] * step, dtype=x.dtype, device=x.device)  # (2.7 GB at 40 rows; only the rows are touched)
    return big.as_strided(x.shape, (big.numel(), big.numel(), step, 1)).copy_(x)


def _desc(t, reverse=False):
    """The library's description of t [B, H, L, D]; reverse: its rows in descending order."""
    from flagattention_amd import _lib

    if not reverse:
        return _lib.SageTensor(t.data_ptr(), *t.stride()[:3])
    return _lib.SageTensor(t.data_ptr() + (t.shape[2] - 1) * t.stride(2) * t.element_size(), t.stride(0), t.stride(1), -t.stride(2))


def _params(q, k, v, o, L, causal, desc):
    from flagattention_amd import _lib
    from flagattention_amd.sage_attention._common import DTYPE_CODE

    p = _lib.FlashParams()
    p.q, p.k, p.v, p.out = desc.get("q", _desc(q)), desc.get("k", _desc(k)), desc.get("v", _desc(v)), _desc(o)
    p.log_normalizer = L.data_ptr()
    p.batch, p.heads_q, p.heads_kv, p.qo_len, p.kv_len, p.head_dim = q.shape[0], q.shape[1], k.shape[1], q.shape[2], k.shape[2], q.shape[3]
    p.dtype = p.out_dtype = DTYPE_CODE[q.dtype]
    p.causal, p.sm_scale = int(causal), q.shape[3] ** -0.5
    return p


@pytest.mark.parametrize("D,dtype", [(64, torch.float16), (128, torch.bfloat16)])
@pytest.mark.parametrize("rows", ["far", "descending"])
def test_dropout_forward(rows, D, dtype, gpu_device):
    from flagattention_amd import _lib

    lib, stream = _lib.load(), torch.cuda.current_stream().cuda_stream
    g = torch.Generator().manual_seed(9)
    H, M, N = (1, 130, 40) if rows == "far" else (3, 200, 333)
    q, k, v = (torch.randn(1, H, n, D, generator=g).to(dtype).to(gpu_device) for n in (M, N, N))
    results = []
    for plain in (True, False):
        if rows == "far":
            kk, vv = (k, v) if plain else (_far(k), _far(v))
            desc = {"k": _desc(kk), "v": _desc(vv)}
        else:
            kk, vv = (k.flip(2).contiguous(), v.flip(2).contiguous()) if plain else (k, v)
            desc = {"k": _desc(kk, not plain), "v": _desc(vv, not plain)}
        o, L = torch.empty_like(q), torch.empty((1, H, M), dtype=torch.float32, device=gpu_device)
        _lib.check(lib.sage_flash_attn_fwd_dropout(_params(q, kk, vv, o, L, True, desc), 0.3, 11, 0, stream), "dropout")
        torch.cuda.synchronize()
        results.append((o, L))
    # (contiguous rows may take several groups of waves, whose shares of a row are added in another order: a rounding step of
    # the 16-bit output, fp32 rounding of the normalizer)
    torch.testing.assert_close(results[0][0].float(), results[1][0].float(), atol=1e-2 if dtype == torch.bfloat16 else 2e-3, rtol=1e-2)
    torch.testing.assert_close(results[0][1], results[1][1], atol=1e-5, rtol=1e-5)


@pytest.mark.parametrize("D,dtype", [(64, torch.float16), (128, torch.bfloat16)])
@pytest.mark.parametrize("rows", ["far", "descending"])
def test_total_attention(rows, D, dtype, gpu_device):
    from flagattention_amd import _lib

    lib, stream = _lib.load(), torch.cuda.current_stream().cuda_stream
    g = torch.Generator().manual_seed(10)
    H, M, N = (1, 40, 300) if rows == "far" else (3, 333, 300)
    q, k = (torch.randn(1, H, n, D, generator=g).to(dtype).to(gpu_device) for n in (M, N))
    L = torch.randn(1, H, M, generator=g).to(gpu_device) + 5.0
    results = []
    for plain in (True, False):
        if rows == "far":
            qq = q if plain else _far(q)
            desc = {"q": _desc(qq)}
        else:
            qq = q.flip(2).contiguous() if plain else q
            desc = {"q": _desc(qq, not plain)}
        tot = torch.empty((1, H, N), dtype=torch.float32, device=gpu_device)
        _lib.check(lib.sage_flash_total_attention(_params(qq, k, k, qq, L, True, desc), L.data_ptr(), tot.data_ptr(), stream), "total")
        torch.cuda.synchronize()
        results.append(tot)
    assert torch.equal(results[0], results[1])


def test_python_entry_point(gpu_device):
    import flag_attn

    g = torch.Generator().manual_seed(12)
    q, k, v = (torch.randn(1, 1, n, 64, generator=g).half().to(gpu_device) for n in (40, 300, 300))
    want = flag_attn.flash_attention(q, k, v, True, return_log_normalizer=True, return_total_attention=True)[:3]
    got = flag_attn.flash_attention(_far(q), k, v, True, return_log_normalizer=True, return_total_attention=True)[:3]
    assert all(torch.equal(a, b) for a, b in zip(got, want))
