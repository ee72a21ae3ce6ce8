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


@pytest.mark.parametrize("b,h,hkv,m,n,d,causal,mask", [
    (1, 2, 2, 2048, 2048, 64, False, None),   # whole items or a key split
    (1, 9, 9, 3000, 3000, 128, True, None),   # cut into equal shares
    (1, 32, 8, 1500, 1500, 128, True, None),  # longest first
    (2, 4, 2, 70, 300, 64, True, None),       # 32-row tiles
    (1, 4, 2, 100, 4000, 128, False, None),   # ... and split keys
    (2, 8, 2, 3, 3000, 64, False, None),      # few query rows
    (1, 2, 2, 256, 256, 64, False, torch.bool),
    (1, 2, 2, 300, 304, 64, False, torch.float16),
    (1, 2, 2, 300, 304, 64, True, torch.float32),   # an additive mask with the causal flag
    (1, 2, 2, 100, 112, 64, True, torch.float16),   # ... over two key tiles: the general kernel, and a launch for the log-sum-exp
    (1, 2, 2, 100, 64, 128, True, None),            # more queries than keys: the general kernel
])
def test_attention_writes_what_the_kernel_of_its_own_does(b, h, hkv, m, n, d, causal, mask, gpu_device):
    """The log-sum-exp of every route of the attention launch, with and without a shift, bit for bit."""
    from flagattention_amd import _lib
    from flagattention_amd.sage_attention import attention as A
    from oracle import sage_oracle as O

    g = torch.Generator().manual_seed(n)
    q, k, v = (torch.randn(b, x, y, d, generator=g).to(torch.bfloat16) for x, y in ((h, m), (hkv, n), (hkv, n)))
    q8, qs, k8, ks = O.per_block_int8(q, k)
    args = [t.to(gpu_device) for t in (q8, k8, v, qs, ks)]
    am = None
    if mask is not None:
        keep = torch.rand(1, 1, m, n, generator=g) > 0.3
        am = (keep if mask is torch.bool else torch.zeros(keep.shape, dtype=mask).masked_fill_(~keep, -9.0)).to(gpu_device)
    shift = torch.randn(b, h, m, generator=g).to(gpu_device)
    o2, lse2 = A.forward(*args, attn_mask=am, return_lse=True, causal=causal)
    for s in (None, shift):
        for _ in range(2):  # the second call takes the plan of the first
            o, lse = A._attend(*args, "HND", am, torch.float16, True, None, causal, 0.125, s)
            want = lse2.clone()
            _lib.check(_lib.load().sage_lse_natural(want.data_ptr(), None if s is None else s.data_ptr(), 0.125, want.numel(),
                                                    torch.cuda.current_stream().cuda_stream), "lse")
            torch.cuda.synchronize()
            assert torch.equal(lse, want) and torch.equal(o, o2)
