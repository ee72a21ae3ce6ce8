"""Additive mask tensors together with the causal flag on the pipelined kernel, against the general kernel (the same mask with rows
that cannot be loaded 16 bytes at a time) and against the oracle."""
import ctypes

import pytest
import torch

from flagattention_amd import _lib
from flagattention_amd.sage_attention._common import tensor_desc
from oracle import c_oracle as C

pytestmark = pytest.mark.gpu
KIND = {torch.float16: _lib.MASK_F16, torch.bfloat16: _lib.MASK_BF16, torch.float32: _lib.MASK_F32}


def _launch(q8, qs, k8, ks, v, mask):
    b, h, m, d = q8.shape
    n = k8.shape[2]
    o, lse = torch.empty(q8.shape, device=q8.device), torch.empty(b, h, m, device=q8.device)
    p = _lib.AttnParams()
    p.q, p.k, p.v, p.out = (tensor_desc(t, True) for t in (q8, k8, v, o))
    p.batch, p.heads_q, p.heads_kv, p.qo_len, p.kv_len, p.head_dim = b, h, k8.shape[1], m, n, d
    p.v_dtype = _lib.SAGE_BF16 if v.dtype is torch.bfloat16 else _lib.SAGE_F16
    p.out_dtype, p.mask_kind, p.causal = _lib.SAGE_F32, KIND[mask.dtype], 1
    p.q_scale, p.k_scale, p.lse, p.mask = qs.data_ptr(), ks.data_ptr(), lse.data_ptr(), mask.data_ptr()
    p.mask_stride_b, p.mask_stride_h, p.mask_stride_m, p.mask_stride_n = mask.expand(b, h, m, n).stride()
    _lib.check(_lib.load().sage_attn_fwd(ctypes.byref(p), torch.cuda.current_stream().cuda_stream), "fwd")
    torch.cuda.synchronize()
    return o, lse


def _entries(kind, shape, m, n, dt, g):
    rows, cols = torch.arange(m).view(m, 1) + (n - m), torch.arange(n)
    if kind == "bias":
        x = torch.randn(shape, generator=g)
    elif kind == "padding":
        x = torch.zeros(shape).masked_fill_((cols >= n - n // 3).expand(shape), torch.finfo(dt).min)
    elif kind == "left":  # the first rows see hidden keys only: the keys the causal mask hides from them weigh more
        x = torch.zeros(shape).masked_fill_((cols < n // 3).expand(shape), torch.finfo(dt).min)
    elif kind == "left_inf":
        x = torch.zeros(shape).masked_fill_((cols < n // 3).expand(shape), float("-inf"))
    elif kind == "late":  # entries that outweigh the causal -1e6, and ones around it
        x = torch.randn(shape, generator=g) + (cols % 7 == 3) * (1.0e6 if dt is not torch.float16 else 0.0)
    elif kind == "rising":  # keys a row does not see would raise its reference point
        x = (cols.float() * 0.25).expand(shape).contiguous()
    elif kind == "nan":
        x = torch.randn(shape, generator=g)
        x[..., m // 2, n // 4] = float("nan")
    return x.to(dt)


# (136 keys at head_dim 64, 200 at 128: the fewest tiles that the pipelined kernel serves 16-bit entries with; 200: fp32 ones)
@pytest.mark.parametrize("m,n,d", [(300, 304, 64), (520, 520, 128), (200, 712, 64), (700, 264, 64), (150, 136, 64), (200, 200, 128),
                                   (257, 1000, 128)])
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("kind", ["bias", "padding", "left", "left_inf", "late", "rising", "nan"])
def test_against_the_general_kernel(kind, dt, m, n, d, gpu_device):
    g = torch.Generator().manual_seed(m + n + d)
    b, h, hkv = 2, 4, 2
    q8 = torch.randint(-127, 128, (b, h, m, d), generator=g, dtype=torch.int8)
    k8 = torch.randint(-127, 128, (b, hkv, n, d), generator=g, dtype=torch.int8)
    qs = torch.rand(b, h, -(-m // 128), generator=g) * 2e-3 + 1e-4
    ks = torch.rand(b, hkv, -(-n // 64), generator=g) * 2e-2 + 1e-3
    v = torch.randn(b, hkv, n, d, generator=g).to(torch.bfloat16 if d == 128 else torch.float16)
    x = [t.to(gpu_device) for t in (q8, qs, k8, ks, v)]
    for shape in ((1, h, m, n), (b, 1, m, n), (b, 1, 1, n)):
        if shape[2] == 1 and kind in ("bias", "late", "nan"):
            continue
        mask = _entries(kind, shape, m, n, dt, g).to(gpu_device)
        wide = torch.zeros((*shape[:3], n + 1), dtype=dt, device=gpu_device)[..., :n] if shape[2] > 1 else \
            torch.zeros((*shape[:3], 2 * n), dtype=dt, device=gpu_device)[..., ::2]  # rows 16-byte loads cannot take
        wide.copy_(mask)
        o, lse = _launch(*x, mask)
        o2, lse2 = _launch(*x, wide)
        assert torch.equal(torch.isnan(lse), torch.isnan(lse2)) and torch.equal(torch.isinf(lse), torch.isinf(lse2))
        assert torch.equal(torch.isnan(o), torch.isnan(o2))
        fin = torch.isfinite(lse2)
        if not fin.any():  # (a first tile of -inf alone: NaN rows, as in the reference's arithmetic)
            continue
        assert ((lse - lse2)[fin].abs() <= 4e-3 + 2e-6 * lse2[fin].abs()).all()
        diff = (o - o2).abs().amax(-1)[fin]
        # Rows near -1e6: the scores are multiples of 1 / 16 there in either kernel; two 16-bit roundings of P apart otherwise
        tol = torch.where(lse2[fin].abs() > 1e5, 0.15, 8e-3 if d == 128 else 2e-3)
        assert (diff <= tol * max(1.0, o2[o2.isfinite()].abs().max().item())).all(), diff.max()


@pytest.mark.parametrize("m,n,layout", [(300, 300, "HND"), (130, 515, "NHD")])
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16, torch.float32])
def test_against_the_oracle(dt, m, n, layout, gpu_device):
    from flag_attn import sage_attention as sa
    from oracle import sage_oracle as O

    g = torch.Generator().manual_seed(n)
    q, k, v = (torch.randn(2, h, x, 64, generator=g).to(torch.float16) for h, x in ((4, m), (2, n), (2, n)))
    if layout == "NHD":
        q, k, v = (t.transpose(1, 2).contiguous() for t in (q, k, v))
    q8, qs, k8, ks = O.per_block_int8(q, k, tensor_layout=layout)
    mask = torch.randn(1, 4, m, n, generator=g).to(dt)
    args = [t.to(gpu_device) for t in (q8, k8, v, qs, ks)]
    want, want_lse = C.attention_blockwise(q8, k8, v, qs, ks, layout, attn_mask=mask.float(), causal=True)
    for _ in range(2):
        o, lse = sa.sage_attention(*args, tensor_layout=layout, attn_mask=mask.to(gpu_device), causal=True, return_lse=True,
                                   output_dtype=torch.float32)
        cos, _, max_abs = O.accuracy_metrics(o.cpu(), want)
        assert cos >= 0.9995 and max_abs <= 2e-2
        torch.testing.assert_close(lse.cpu(), want_lse, atol=2e-3, rtol=1e-4)


@pytest.mark.parametrize("m,n,d", [(256, 256, 64), (256, 320, 128), (700, 712, 64)])  # even and odd numbers of steps, a ragged last tile
@pytest.mark.parametrize("dt", [torch.float16, torch.float32])
def test_v_past_the_limit_of_a_block(dt, m, n, d, gpu_device):
    """Inf and NaN in V reach the 128-row blocks that visit their tile and no other: the reference skips tiles that the causal
    mask hides from every row of a block."""
    g = torch.Generator().manual_seed(m + n)
    q8 = torch.randint(-127, 128, (1, 2, m, d), generator=g, dtype=torch.int8)
    k8 = torch.randint(-127, 128, (1, 2, n, d), generator=g, dtype=torch.int8)
    qs = torch.rand(1, 2, -(-m // 128), generator=g) * 2e-3 + 1e-4
    ks = torch.rand(1, 2, -(-n // 64), generator=g) * 2e-2 + 1e-3
    mask = torch.randn(1, 2, m, n, generator=g).to(dt).to(gpu_device)
    wide = torch.zeros(1, 2, m, n + 1, dtype=dt, device=gpu_device)[..., :n]  # rows 16-byte loads cannot take
    wide.copy_(mask)
    for key, bad in ((n - 1, float("inf")), (n - 60, float("nan")), (n - m + 128, float("-inf"))):
        v = torch.randn(1, 2, n, d, generator=g).to(torch.bfloat16 if d == 128 else torch.float16)
        v[:, 0, key, 3] = bad
        x = [t.to(gpu_device) for t in (q8, qs, k8, ks, v)]
        o, lse = _launch(*x, mask)
        o2, lse2 = _launch(*x, wide)
        torch.testing.assert_close(lse, lse2, atol=2e-3, rtol=1e-4)
        assert torch.equal(torch.isfinite(o), torch.isfinite(o2))
        # the first row of the first 128-row block that visits the key's tile
        first = max(0, (key // 64 * 64 - (n - m)) // 128 * 128)
        assert torch.isfinite(o[:, :, :first]).all() and not torch.isfinite(o[:, 0, first:, 3]).any()
        assert torch.isfinite(o[:, 1]).all() and torch.isfinite(o[..., :3]).all()
