"""The quantizer's fused launches at their edges, bit for bit against the oracle: one workgroup per head (up to 256 keys at
head_dim 128, 512 at 64), K blocks that add the chunk partials of the mean themselves (up to 128 chunks), K and Q blocks in one
grid, and the sizes just beyond each."""
import pytest
import torch

from oracle import c_oracle as C

pytestmark = pytest.mark.gpu


def _check(got, want):
    for g, w, name in zip(got, want, ("q_int8", "q_scale", "k_int8", "k_scale")):
        g = g.cpu()
        assert g.shape == w.shape and g.dtype == w.dtype
        assert torch.equal(g.view(torch.int32) if g.dtype == torch.float32 else g, w.view(torch.int32) if w.dtype == torch.float32 else w), name


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("d,n", [(64, 1), (64, 63), (64, 64), (64, 65), (64, 128), (64, 129), (64, 256), (64, 300), (64, 512), (64, 513),
                                 (128, 1), (128, 64), (128, 65), (128, 128), (128, 191), (128, 256), (128, 257), (128, 1024),
                                 (128, 1025), (128, 2048), (64, 2049), (32, 700), (32, 1100), (16, 90), (256, 200)])
def test_smoothing_launch_forms(d, n, dtype, gpu_device):
    from flag_attn import sage_attention as sa
    from flagattention_amd.sage_attention.quant import per_block_int8_smooth_k

    g = torch.Generator().manual_seed(n + d)
    b, hq, hkv, m = 2, 4, 2, max(1, n - 37)
    for layout in ("HND", "NHD"):
        q = torch.randn(b, hq, m, d, generator=g).to(dtype)
        k = (torch.randn(b, hkv, n, d, generator=g) + 3.0 * torch.randn(1, hkv, 1, d, generator=g)).to(dtype)
        k[0, 0, : min(n, 64)] = 0  # a block of zeros (before the mean is taken off)
        if layout == "NHD":
            q, k = q.transpose(1, 2).contiguous(), k.transpose(1, 2).contiguous()
        km = C.k_mean_fixed_order(k, layout)
        want = C.per_block_int8(q, k, km=km, tensor_layout=layout)
        dq, dk = q.to(gpu_device), k.to(gpu_device)
        _check(sa.per_block_int8(dq, dk, tensor_layout=layout, smooth_k=True), want)
        *got, km_got, dot = per_block_int8_smooth_k(dq, dk, tensor_layout=layout, with_q_dot_km=True)
        _check(got, want)
        assert torch.equal(km_got.cpu().view(torch.int16), km.view(torch.int16))
        assert torch.equal(sa.k_mean(dk, layout).cpu().view(torch.int16), km.view(torch.int16))
        qh, kmh = (q, km) if layout == "HND" else (q.transpose(1, 2), km.transpose(1, 2))
        ref = (qh.double() * kmh.double().repeat_interleave(hq // hkv, dim=1)).sum(-1)
        # fp32 sums of d products: each addition rounds once, d roundings of the running sum's magnitude
        bound = d * 2.0 ** -24 * (qh.double().abs() * kmh.double().abs().repeat_interleave(hq // hkv, dim=1)).sum(-1)
        assert bool(((dot.cpu().double() - ref).abs() <= bound + 1e-12).all())


@pytest.mark.parametrize("b,h,n,d", [(1, 2, 2500, 64), (1, 1, 4097, 128), (1, 3, 6001, 64), (1, 6, 8191, 128), (1, 6, 8193, 128),
                                     (1, 33, 3700, 64), (64, 1, 2048, 64), (65, 1, 2048, 64), (90, 1, 2048, 64), (96, 1, 2048, 64),
                                     (1, 24, 2500, 128), (1, 26, 2560, 128), (3, 5, 650, 128)])
def test_mean_added_by_the_k_blocks(b, h, n, d, gpu_device):
    """Each line of the rule and the size beyond it; the same bits as the mean from a launch of its own."""
    from flagattention_amd.sage_attention.quant import per_block_int8_smooth_k

    g = torch.Generator().manual_seed(n)
    k = (torch.randn(b, h, n, d, generator=g) + 2.0).to(torch.bfloat16)
    q = torch.randn(b, h, 70, d, generator=g).to(torch.bfloat16)
    km = C.k_mean_fixed_order(k, "HND")
    want = C.per_block_int8(q, k, km=km, tensor_layout="HND")
    for with_dot in (False, True):
        *got, km_got, dot = per_block_int8_smooth_k(q.to(gpu_device), k.to(gpu_device), tensor_layout="HND", with_q_dot_km=with_dot)
        assert torch.equal(km_got.cpu().view(torch.int16), km.view(torch.int16))
        _check(got, want)
    ref = (q.double() * km.double()).sum(-1)
    bound = d * 2.0 ** -24 * (q.double().abs() * km.double().abs()).sum(-1)  # fp32 sums of d products, one rounding per addition
    assert bool(((dot.cpu().double() - ref).abs() <= bound + 1e-12).all())


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("b,hq,hkv,m,n,d", [(1, 2, 2, 1, 1, 64), (2, 4, 2, 200, 77, 128), (1, 3, 1, 129, 1000, 64),
                                            (4, 32, 8, 2048, 4032, 64), (4, 32, 8, 2048, 4160, 64), (1, 2, 1, 90, 130, 256),
                                            (2, 16, 16, 2000, 2049, 128), (1, 33, 11, 4095, 129, 128), (3, 8, 8, 65, 8191, 32)])
def test_k_and_q_in_one_grid(b, hq, hkv, m, n, d, dtype, gpu_device):
    from flag_attn import sage_attention as sa

    g = torch.Generator().manual_seed(3)
    q, k = torch.randn(b, hq, m, d, generator=g).to(dtype), torch.randn(b, hkv, n, d, generator=g).to(dtype)
    km = k.float().mean(2, keepdim=True).to(dtype)
    for mean in (None, km):
        got = sa.per_block_int8(q.to(gpu_device), k.to(gpu_device), km=None if mean is None else mean.to(gpu_device))
        _check(got, C.per_block_int8(q, k, km=mean))


@pytest.mark.parametrize("layout", ["HND", "NHD"])
@pytest.mark.parametrize("b,hq,hkv,m,n,d", [(1, 16, 4, 2100, 2113, 128), (2, 32, 8, 2047, 2049, 128), (2, 32, 16, 2500, 4100, 64)])
def test_k_and_q_in_one_grid_behind_the_mean(b, hq, hkv, m, n, d, layout, gpu_device):
    """Q blocks that also give q . km, at up to 1024 blocks and beyond: the bits of the K and Q blocks on their own, and the
    same dot products as for one head alone (which is in a smaller grid)."""
    from flagattention_amd.sage_attention.quant import per_block_int8_smooth_k

    g = torch.Generator().manual_seed(4)
    q, k = torch.randn(b, hq, m, d, generator=g).bfloat16(), (torch.randn(b, hkv, n, d, generator=g) + 2.0).bfloat16()
    if layout == "NHD":
        q, k = q.transpose(1, 2).contiguous(), k.transpose(1, 2).contiguous()
    km = C.k_mean_fixed_order(k, layout)
    *got, km_got, dot = per_block_int8_smooth_k(q.to(gpu_device), k.to(gpu_device), tensor_layout=layout, with_q_dot_km=True)
    _check(got, C.per_block_int8(q, k, km=km, tensor_layout=layout))
    assert torch.equal(km_got.cpu().view(torch.int16), km.view(torch.int16))
    if layout == "NHD":
        q, k = q.transpose(1, 2), k.transpose(1, 2)
    h = hq - 1
    *_, one = per_block_int8_smooth_k(q[-1:, h:].contiguous().to(gpu_device), k[-1:, hkv - 1:].contiguous().to(gpu_device), with_q_dot_km=True)
    assert torch.equal(dot[-1, h], one[0, 0])
