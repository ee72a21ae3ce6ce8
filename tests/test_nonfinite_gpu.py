"""A NaN or an infinity in Q or K makes the rows that see it NaN, output and log-sum-exp alike, whether a launch is whole or
leaves partial results in a workspace that a second kernel combines."""
import ctypes
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

# (batch, heads_q, heads_kv, M, N, D, causal)
SHAPES = [
    (8, 32, 8, 1, 8192, 128, False),    # few query rows, four runs of the keys
    (1, 8, 8, 1, 8192, 64, False),      # ... many runs, which eight groups of threads per row share
    (1, 32, 32, 1, 8192, 64, False),    # ... a run for each of the groups
    (1, 8, 2, 5, 3000, 128, True),
    (1, 4, 2, 300, 4096, 64, True),     # keys of a 256-row block split
    (1, 2, 2, 20, 4096, 128, False),
    (1, 9, 9, 3000, 3000, 128, True),   # launch cut into equal shares
    (1, 33, 33, 2100, 2100, 64, False),
]


def _launch(lib, kind, p, workspace, device):
    stream = torch.cuda.current_stream().cuda_stream
    need = getattr(lib, f"sage_{kind}_workspace_bytes")(ctypes.byref(p))
    assert need > 0, "this shape was meant to leave partial results"
    if workspace:
        ws = torch.empty(need, dtype=torch.uint8, device=device)
        rc = getattr(lib, f"sage_{kind}_ws")(ctypes.byref(p), ws.data_ptr(), need, stream)
    else:
        rc = getattr(lib, f"sage_{kind}")(ctypes.byref(p), stream)
    assert rc == 0, lib.sage_hip_last_error()
    torch.cuda.synchronize()


def _check(results, want, empty=None):
    """``want`` [B, H, M]: the rows that are NaN in every channel and in the log-sum-exp; all others are finite, but for the
    log-sum-exp of ``empty`` ones, whose scores are all -inf."""
    for workspace, (o, lse) in enumerate(results):
        infinite = want if empty is None else want | empty
        for got, expected in ((torch.isnan(lse), want), (~torch.isfinite(lse), infinite), (torch.isnan(o).all(-1), want),
                              (~torch.isfinite(o).all(-1), want)):
            wrong = (got != expected).nonzero()
            assert not len(wrong), (f"workspace {workspace}: {len(wrong)} rows", wrong[:4].tolist(), wrong[-4:].tolist())


def _sees(m, n, key, causal, device):
    """[M]: which queries see key ``key``."""
    return torch.arange(m, device=device) + (n - m) >= key if causal else torch.ones(m, dtype=torch.bool, device=device)


@pytest.mark.parametrize("where", ["query_nan", "query_inf", "key_nan"])
@pytest.mark.parametrize("b,h,hkv,m,n,d,causal", SHAPES)
def test_dense_rows(b, h, hkv, m, n, d, causal, where, gpu_device):
    from flagattention_amd import _lib
    from flagattention_amd.sage_attention._common import DTYPE_CODE, tensor_desc

    g = torch.Generator().manual_seed(3)
    q, k, v = (torch.randn(b, x, y, d, generator=g).to(torch.bfloat16).to(gpu_device) for x, y in ((h, m), (hkv, n), (hkv, n)))
    want = torch.zeros((b, h, m), dtype=torch.bool, device=gpu_device)
    if where == "key_nan":
        k[0, hkv - 1, 100, 7] = float("nan")
        want[0, (hkv - 1) * (h // hkv):] = _sees(m, n, 100, causal, gpu_device)
    else:
        row = m // 2
        q[0, 1, row, 5] = float("nan" if where == "query_nan" else "inf")
        want[0, 1, row] = True
    lib = _lib.load()
    results = []
    for workspace in (False, True):
        o, lse = torch.empty_like(q), torch.empty((b, h, m), dtype=torch.float32, device=gpu_device)
        p = _lib.FlashParams()
        p.q, p.k, p.v, p.out = (tensor_desc(t, True) for t in (q, k, v, o))
        p.log_normalizer = lse.data_ptr()
        p.batch, p.heads_q, p.heads_kv, p.qo_len, p.kv_len, p.head_dim, p.causal = b, h, hkv, m, n, d, causal
        p.dtype = p.out_dtype = DTYPE_CODE[torch.bfloat16]
        p.sm_scale = d ** -0.5
        _launch(lib, "flash_attn_fwd", p, workspace, gpu_device)
        results.append((o, lse))
    _check(results, want)


@pytest.mark.parametrize("where", ["query_scale", "key_scale"])
@pytest.mark.parametrize("b,h,hkv,m,n,d,causal", SHAPES)
def test_quantized_rows(b, h, hkv, m, n, d, causal, where, gpu_device):
    """An infinite scale, as the quantizer gives a block that holds an infinity: scores of +inf or (product 0) NaN make their
    rows NaN, a score of -inf is a key of weight 0."""
    from flag_attn import sage_attention as sa
    from flagattention_amd import _lib
    from flagattention_amd.sage_attention._common import DTYPE_CODE, tensor_desc

    g = torch.Generator().manual_seed(4)
    q, k, v = (torch.randn(b, x, y, d, generator=g).to(torch.bfloat16).to(gpu_device) for x, y in ((h, m), (hkv, n), (hkv, n)))
    q8, qs, k8, ks = sa.per_block_int8(q, k)
    want = torch.zeros((b, h, m), dtype=torch.bool, device=gpu_device)
    keys = torch.arange(n, device=gpu_device)
    sees = keys[None, :] <= torch.arange(m, device=gpu_device)[:, None] + (n - m) if causal else torch.ones((m, n), dtype=torch.bool, device=gpu_device)
    rows = torch.ones(m, dtype=torch.bool, device=gpu_device)
    if where == "key_scale":
        heads = range((hkv - 1) * (h // hkv), h)
        ks[0, hkv - 1, 1] = float("inf")  # keys 64 to 127
        sees = sees & (keys >= 64) & (keys < 128)
    else:
        heads = [1]
        qs[0, 1, 0] = float("inf")  # queries 0 to 127
        rows[128:] = False
    for head in heads:
        dot = q8[0, head].float() @ k8[0, head // (h // hkv)].float().T
        want[0, head] = rows & ((dot >= 0) & sees).any(1)
    assert bool(want.any())
    empty = torch.zeros_like(want)
    if where == "query_scale":  # (the first queries under the causal flag see few keys)
        empty[0, 1] = rows & ~want[0, 1]
    lib = _lib.load()
    results = []
    for workspace in (False, True):
        o, lse = torch.empty_like(q), torch.empty((b, h, m), dtype=torch.float32, device=gpu_device)
        p = _lib.AttnParams()
        p.q, p.k, p.v, p.out = (tensor_desc(t, True) for t in (q8, k8, v, o))
        p.q_scale, p.k_scale, p.lse = qs.data_ptr(), ks.data_ptr(), lse.data_ptr()
        p.batch, p.heads_q, p.heads_kv, p.qo_len, p.kv_len, p.head_dim, p.causal = b, h, hkv, m, n, d, causal
        p.v_dtype = p.out_dtype = DTYPE_CODE[torch.bfloat16]
        _launch(lib, "attn_fwd", p, workspace, gpu_device)
        results.append((o, lse))
    _check(results, want, empty)


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("mask_dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_additive_mask_rows_that_meet_hidden_tiles_first(mask_dtype, d, gpu_device):
    """A sliding window as an additive mask of the type's lowest value: the first tiles hide every key of a row while other
    rows of its wave already see some."""
    from flag_attn import sage_attention as sa
    from oracle import sage_oracle as O

    g = torch.Generator().manual_seed(5)
    n = 768
    q, k, v = (torch.randn(1, 2, n, d, generator=g).to(torch.bfloat16) for _ in range(3))
    q8, qs, k8, ks = O.per_block_int8(q, k)
    rows, cols = torch.arange(n).view(n, 1), torch.arange(n)
    keep = ((cols <= rows) & (cols > rows - 100)).view(1, 1, n, n)
    mask = torch.zeros(keep.shape, dtype=mask_dtype).masked_fill_(~keep, torch.finfo(mask_dtype).min)
    o, lse = sa.sage_attention(*(t.to(gpu_device) for t in (q8, k8, v, qs, ks)), attn_mask=mask.to(gpu_device), return_lse=True)
    # (float64: hidden scores lie beyond the exponent's range there too)
    sc = qs.double().repeat_interleave(128, -1)[..., :n, None] * ks.double().repeat_interleave(64, -1)[..., None, :n]
    s = (q8.double() @ k8.double().transpose(-1, -2)) * sc
    s = s.masked_fill(~keep, float("-inf"))
    want = torch.softmax(s * math.log(2.0), -1) @ v.double()
    torch.testing.assert_close(o.double().cpu(), want, rtol=2e-2, atol=2e-2)
    torch.testing.assert_close(lse.double().cpu(), torch.logsumexp(s * math.log(2.0), -1) / math.log(2.0), rtol=1e-4, atol=2e-3)


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("n", [2112, 2112 + 40])  # 33 steps of 64 keys, an odd number; a ragged last one
def test_a_nan_query_leaves_its_neighbours_alone(n, causal, d, gpu_device):
    """A NaN query row makes every step of its wave look too large, the padding step after an odd number included: the other
    rows of the wave have to come out as without it."""
    import flag_attn
    from oracle import flash_oracle as FO

    g = torch.Generator().manual_seed(n)
    q, k, v = (torch.randn(1, 16, x, d, generator=g).to(torch.float16) for x in (n, n, n))
    bad = [3, 70, n - 5]
    q_nan = q.clone()
    q_nan[:, :, bad] = float("nan")
    o, lse, *_ = flag_attn.flash_attention(q_nan.to(gpu_device), k.to(gpu_device), v.to(gpu_device), causal, return_log_normalizer=True)
    want, want_lse = FO.attention(q[:, :2], k[:, :2], v[:, :2], causal, return_log_normalizer=True)
    keep = [i for i in range(n) if i not in bad]
    torch.testing.assert_close(lse.cpu()[:, :2, keep], want_lse[:, :, keep], atol=2e-3, rtol=1e-4)
    torch.testing.assert_close(o.cpu()[:, :2, keep].float(), want[:, :, keep].float(), atol=4e-3, rtol=1e-2)
    assert torch.isnan(o[:, :, bad]).all() and torch.isnan(lse[:, :, bad]).all()


@pytest.mark.parametrize("mask_dtype", [torch.float16, torch.float32])
def test_a_nan_mask_entry_leaves_its_neighbours_alone(mask_dtype, gpu_device):
    from flag_attn import sage_attention as sa
    from oracle import sage_oracle as O

    g = torch.Generator().manual_seed(2)
    n = 320
    q, k, v = (torch.randn(1, 2, n, 64, generator=g).to(torch.float16) for _ in range(3))
    args = [t.to(gpu_device) for t in O.per_block_int8(q, k)]
    mask = torch.randn(1, 2, n, n, generator=g).to(mask_dtype).to(gpu_device)
    o, lse = sa.sage_attention(args[0], args[2], v.to(gpu_device), args[1], args[3], attn_mask=mask, return_lse=True)
    mask[0, :, 100, 7] = float("nan")
    o_nan, lse_nan = sa.sage_attention(args[0], args[2], v.to(gpu_device), args[1], args[3], attn_mask=mask, return_lse=True)
    rows = [i for i in range(n) if i != 100]
    torch.testing.assert_close(lse_nan[:, :, rows], lse[:, :, rows], atol=2e-3, rtol=1e-4)
    torch.testing.assert_close(o_nan[:, :, rows].float(), o[:, :, rows].float(), atol=4e-3, rtol=1e-2)
    assert torch.isnan(o_nan[:, :, 100]).all() and torch.isnan(lse_nan[:, :, 100]).all()
