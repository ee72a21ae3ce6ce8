"""The log-sum-exp that the one-call wrapper returns: base 2 -> natural log with the smoothing's shift, in one pass."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shifted", [False, True])
@pytest.mark.parametrize("n", [1, 255, 256, 257, 100003])
def test_lse_natural(n, shifted, gpu_device):
    from flagattention_amd import _lib

    g = torch.Generator().manual_seed(5)
    lse = 40 * torch.randn(n, generator=g)
    lse[0] = float("-inf")  # (a row that sees no key)
    shift = 10 * torch.randn(n, generator=g)
    buf = torch.full((n + 1,), 7.0, device=gpu_device)
    buf[:n] = lse.to(gpu_device)
    d_shift = shift.to(gpu_device)
    rc = _lib.load().sage_lse_natural(buf.data_ptr(), d_shift.data_ptr() if shifted else None, 0.088, n,
                                      torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    want = lse.double() * torch.log(torch.tensor(2.0, dtype=torch.float64))
    if shifted:
        want += shift.double() * float(torch.tensor(0.088))
    # the product is rounded, then the sum: two roundings of values up to 130
    torch.testing.assert_close(buf[:n].cpu().double(), want, atol=2 * 2**-24 * 256, rtol=0)
    assert float(buf[n]) == 7.0


@pytest.mark.parametrize("layout", ["HND", "NHD"])
def test_wrapper_with_mixed_dtypes(layout, gpu_device):
    """The dot product with the mean comes from torch there, in its own memory order."""
    from flag_attn import sage_attention as sa

    g = torch.Generator().manual_seed(6)
    b, h, hkv, m, n, d = 2, 4, 2, 130, 200, 64
    shape = (lambda x, y: (b, x, y, d)) if layout == "HND" else (lambda x, y: (b, y, x, d))
    q = torch.randn(shape(h, m), generator=g).to(torch.float16).to(gpu_device)
    k = (torch.randn(shape(hkv, n), generator=g) + 1.0).to(torch.bfloat16).to(gpu_device)
    v = torch.randn(shape(hkv, n), generator=g).to(torch.float16).to(gpu_device)
    _, lse = sa.sageattn(q, k, v, tensor_layout=layout, return_lse=True)
    qh, kh = (q, k) if layout == "HND" else (q.transpose(1, 2), k.transpose(1, 2))
    kh = kh.float().repeat_interleave(h // hkv, dim=1)
    want = torch.logsumexp(torch.matmul(qh.float(), kh.transpose(2, 3).contiguous()) * d ** -0.5, dim=-1)
    torch.testing.assert_close(lse, want, atol=3e-2, rtol=0)  # (scores of int8 products: a quantization step of Q and K)
