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


@pytest.mark.parametrize("where", ["query_nan", "query_inf", "key_nan", "normalizer_nan"])
@pytest.mark.parametrize("M,N,causal", [(600, 700, False), (600, 700, True), (700, 600, True), (33, 65, True), (2100, 2100, True)])
def test_total_attention_keeps_nan(M, N, causal, where, gpu_device):
    """A query whose log normalizer is NaN makes the sums of all keys it sees NaN, and no other: with runs of the queries and
    without, also where the causal limit runs through a tile."""
    import flag_attn
    from flagattention_amd import _lib
    from flagattention_amd.sage_attention._common import DTYPE_CODE, tensor_desc

    B, H, D = 1, 2, 64
    g = torch.Generator().manual_seed(6)
    q, k, v = (torch.randn(B, H, n, D, generator=g).to(torch.bfloat16).to(gpu_device) for n in (M, N, N))
    row = M // 2 + 5
    if where == "key_nan":
        k[0, 1, N // 3, 0] = float("nan")
    elif where != "normalizer_nan":
        q[0, 1, row, 0] = float(where[6:])
    _, L, tot, *_ = flag_attn.flash_attention(q, k, v, causal, return_log_normalizer=True, return_total_attention=True)
    if where == "normalizer_nan":
        L[0, 1, row] = float("nan")
    sees = torch.ones(M, N, dtype=torch.bool, device=gpu_device)
    if causal:
        sees = torch.arange(N, device=gpu_device)[None, :] <= torch.arange(M, device=gpu_device)[:, None] + (N - M)
    bad = torch.zeros(M, dtype=torch.bool, device=gpu_device)
    bad[row] = True
    if where == "key_nan":
        bad = sees[:, N // 3]
    want = torch.zeros((B, H, N), dtype=torch.bool, device=gpu_device)
    want[0, 1] = sees[bad].any(0)
    assert torch.equal(torch.isnan(L)[0, 1], bad)
    lib = _lib.load()
    p = _lib.FlashParams()
    p.q, p.k = tensor_desc(q, True), tensor_desc(k, True)
    p.batch, p.heads_q, p.heads_kv, p.qo_len, p.kv_len, p.head_dim = B, H, H, M, N, D
    p.dtype, p.causal, p.sm_scale = DTYPE_CODE[torch.bfloat16], int(causal), D ** -0.5
    one, runs = torch.empty_like(tot), torch.empty_like(tot)
    stream = torch.cuda.current_stream().cuda_stream
    _lib.check(lib.sage_flash_total_attention(p, L.data_ptr(), one.data_ptr(), stream), "total")
    need = lib.sage_flash_total_attention_workspace_bytes(p)
    ws = torch.empty(max(need, 16), dtype=torch.uint8, device=gpu_device)
    _lib.check(lib.sage_flash_total_attention_ws(p, L.data_ptr(), runs.data_ptr(), ws.data_ptr(), ws.numel(), stream), "total")
    torch.cuda.synchronize()
    for got in (one, runs) if where == "normalizer_nan" else (tot, one, runs):
        assert torch.equal(torch.isnan(got), want) and bool(torch.isfinite(got[~want]).all())


@pytest.mark.parametrize("B,H,Hk,M,N,D,causal", [
    (1, 2, 2, 1024, 1024, 64, True),     # runs of the fewest tiles, a different number for every key block
    (1, 3, 1, 700, 2300, 128, True),     # fewer queries than keys: every block is seen by the last queries
    (1, 2, 2, 2300, 700, 64, True),      # more: the first queries see no key
    (2, 4, 4, 3000, 2900, 64, False),    # long runs
])
def test_total_attention_runs(B, H, Hk, M, N, D, causal, gpu_device):
    """Runs of different numbers per key block against one run per block (no workspace)."""
    import flag_attn
    from flagattention_amd import _lib
    from flagattention_amd.sage_attention._common import tensor_desc

    g = torch.Generator().manual_seed(M)
    q, k, v = (torch.randn(B, h, n, D, generator=g).to(torch.float16).to(gpu_device) for h, n in ((H, M), (Hk, N), (Hk, N)))
    o, L, tot, *_ = flag_attn.flash_attention(q, k, v, causal, return_log_normalizer=True, return_total_attention=True)
    p = _lib.FlashParams()
    p.q, p.k, p.v, p.out = (tensor_desc(t, True) for t in (q, k, v, o))
    p.batch, p.heads_q, p.heads_kv, p.qo_len, p.kv_len, p.head_dim = B, H, Hk, M, N, D
    p.dtype = p.out_dtype = _lib.SAGE_F16
    p.causal, p.sm_scale = int(causal), D ** -0.5
    lib = _lib.load()
    assert lib.sage_flash_total_attention_workspace_bytes(p) > 0
    one = torch.empty_like(tot)
    _lib.check(lib.sage_flash_total_attention(p, L.data_ptr(), one.data_ptr(), torch.cuda.current_stream().cuda_stream), "total")
    torch.cuda.synchronize()
    torch.testing.assert_close(tot, one, rtol=1e-5, atol=1e-5)  # (fp32 sums of the same terms in another order)
    seen = int((~torch.isinf(L)).sum())
    assert abs(tot.sum().item() - seen) <= 2e-3 * seen
