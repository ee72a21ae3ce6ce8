"""The total attention kernel at the edges of its tiles: 256 keys per workgroup, 64 per wave, 32 queries per tile, runs of at
least eight query tiles (with and without a workspace: runs or none)."""
import pytest
import torch

from oracle import flash_oracle as FO

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,dtype", [(64, torch.float16), (128, torch.bfloat16)])
@pytest.mark.parametrize("M,N", [(1, 1), (31, 257), (33, 64), (65, 255), (97, 513), (520, 320), (1055, 300), (300, 1055)])
def test_total_attention_tile_edges(M, N, D, dtype, gpu_device):
    import flag_attn
    from flagattention_amd import _lib
    from flagattention_amd.sage_attention._common import DTYPE_CODE, tensor_desc

    B, Hq, Hk = 2, 4, 2
    g = torch.Generator().manual_seed(5)
    q, k, v = (torch.randn(B, h, n, D, generator=g).to(dtype) for h, n in ((Hq, M), (Hk, N), (Hk, N)))
    dq, dk, dv = (t.to(gpu_device) for t in (q, k, v))
    lib = _lib.load()
    for causal in (False, True):
        o, L, tot, *_ = flag_attn.flash_attention(dq, dk, dv, causal, return_log_normalizer=True, return_total_attention=True)
        _, _, want = FO.attention(q, k, v, causal, return_total_attention=True, upcast=True)
        _, _, want_16 = FO.attention(q, k, v, causal, return_total_attention=True, upcast=False)
        # the reference's rule: at most twice the deviation of the 16-bit closed form
        assert FO.max_diff(tot.cpu(), want) <= 2 * FO.max_diff(want_16, want) + 1e-5, causal
        # one run over all queries (no workspace): the same terms added in another order.  A key's sum has at most M terms
        # of at most 1, so either order is within M * 2^-24 of the exact sum per term added
        p = _lib.FlashParams()
        p.q, p.k = tensor_desc(dq, True), tensor_desc(dk, True)
        p.batch, p.heads_q, p.heads_kv, p.qo_len, p.kv_len, p.head_dim = B, Hq, Hk, M, N, D
        p.dtype, p.causal, p.sm_scale = DTYPE_CODE[dtype], int(causal), D ** -0.5
        assert (lib.sage_flash_total_attention_workspace_bytes(p) > 0) == (M >= 512)
        one = torch.empty_like(tot)
        _lib.check(lib.sage_flash_total_attention(p, L.data_ptr(), one.data_ptr(), torch.cuda.current_stream().cuda_stream), "total")
        torch.cuda.synchronize()
        torch.testing.assert_close(one, tot, rtol=2 * M * 2.0 ** -24, atol=1e-6)
