"""GPU parity of the launches that are cut into equal shares of their steps, and of the causal launches that hand out
q-blocks longest first: odd and even numbers of q-blocks, ragged tiles, more and fewer queries than keys, rows that see
no key, both head_dims."""
import ctypes

import pytest
import torch

from oracle import c_oracle as C
from oracle import flash_oracle as FO
from oracle import sage_oracle as O

pytestmark = pytest.mark.gpu


def _run(lib, p, kind, workspace, device):
    stream = torch.cuda.current_stream().cuda_stream
    need = getattr(lib, f"sage_{kind}_workspace_bytes")(ctypes.byref(p))
    if workspace:
        ws = torch.full((need,), 0xFF, dtype=torch.uint8, device=device)  # (NaN wherever nothing is written)
        rc = getattr(lib, f"sage_{kind}_ws")(ctypes.byref(p), ws.data_ptr(), need, stream)
    else:
        rc = getattr(lib, f"sage_{kind}")(ctypes.byref(p), stream)
    assert rc == 0, lib.sage_hip_last_error()
    torch.cuda.synchronize()
    return need


# (heads_q, heads_kv, M, N, D, causal, whether the launch is cut)
SHAPES = [
    (9, 9, 3000, 3000, 128, True, True),      # twelve q-blocks, ragged last tile
    (6, 2, 3400, 3400, 64, True, True),       # fourteen, grouped heads
    (10, 10, 1200, 2905, 128, True, True),    # fewer queries than keys, an odd number of q-blocks
    (33, 33, 2100, 2100, 64, False, True),    # 297 q-blocks, cut nearly once each
    (5, 1, 14000, 1531, 128, False, True),    # 275 q-blocks: one round and a bit, ragged last tile
    (36, 36, 1100, 1100, 128, True, False),   # longest first: five q-blocks, heads not a multiple of eight
    (40, 8, 1025, 1025, 64, True, False),     # ... a multiple of eight, one row in the last q-block
]


@pytest.mark.parametrize("h,hkv,m,n,d,causal,cut", SHAPES)
def test_sage_shares(h, hkv, m, n, d, causal, cut, gpu_device):
    from flagattention_amd import _lib
    from flagattention_amd.sage_attention.attention import DTYPE_CODE, tensor_desc

    g = torch.Generator().manual_seed(31)
    q, k, v = (torch.randn(1, x, y, d, generator=g).to(torch.bfloat16) for x, y in ((h, m), (hkv, n), (hkv, n)))
    host = O.per_block_int8(q, k)
    q8, qs, k8, ks, dv = (t.to(gpu_device) for t in (*host, v))
    lib = _lib.load()
    res = []
    for workspace in (True, False):
        o = torch.empty(q8.shape, dtype=torch.bfloat16, device=gpu_device)
        lse = torch.empty((1, h, m), dtype=torch.float32, device=gpu_device)
        p = _lib.AttnParams()
        p.q, p.k, p.v, p.out = (tensor_desc(t, True) for t in (q8, k8, dv, o))
        p.q_scale, p.k_scale, p.lse = qs.data_ptr(), ks.data_ptr(), lse.data_ptr()
        p.batch, p.heads_q, p.heads_kv, p.qo_len, p.kv_len, p.head_dim, p.causal = 1, h, hkv, m, n, d, causal
        p.v_dtype = p.out_dtype = DTYPE_CODE[torch.bfloat16]
        need = _run(lib, p, "attn_fwd", workspace and cut, gpu_device)
        share = 2 * 256 * (d + 1) * 4
        assert (need % share == 0 and 0 < need // share <= 256) if cut else need == 0
        res.append((o, lse))
    # the keys of a row grouped in another way: a 16-bit output may move by a rounding step, the row sums are those of rounded P
    torch.testing.assert_close(res[0][0].float(), res[1][0].float(), atol=4e-3, rtol=1e-2)
    torch.testing.assert_close(res[0][1], res[1][1], atol=2e-3, rtol=1e-4)
    # the oracle on the first and the last K/V head (the gates of the unsplit tests)
    per = h // hkv
    for j in sorted({0, hkv - 1}):
        a = slice(j * per, j * per + 1)
        kv = slice(j, j + 1)
        ref, ref_lse = C.attention_blockwise(host[0][:, a], host[2][:, kv], v[:, kv], host[1][:, a], host[3][:, kv], "HND", causal=causal)
        cos, _, max_abs = O.accuracy_metrics(res[0][0][:, a].float().cpu(), ref)
        assert cos >= 0.9995 and max_abs <= 2e-2
        torch.testing.assert_close(res[0][1][:, a].cpu(), ref_lse, atol=2e-3, rtol=1e-4)


@pytest.mark.parametrize("h,hkv,m,n,d,causal,cut", SHAPES + [
    (6, 6, 5000, 3000, 128, True, True),   # more queries than keys: the first seven q-blocks see no key, the next one in part
    (24, 24, 900, 700, 64, True, False),   # ... longest first
])
def test_flash_shares(h, hkv, m, n, d, causal, cut, gpu_device):
    from flagattention_amd import _lib
    from flagattention_amd.sage_attention._common import DTYPE_CODE, tensor_desc

    g = torch.Generator().manual_seed(32)
    q, k, v = (torch.randn(1, x, y, d, generator=g).to(torch.float16) for x, y in ((h, m), (hkv, n), (hkv, n)))
    dq, dk, dv = q.to(gpu_device), k.to(gpu_device), v.to(gpu_device)
    lib = _lib.load()
    res = []
    for workspace in (True, False):
        o = torch.empty_like(dq)
        L = torch.empty((1, h, m), dtype=torch.float32, device=gpu_device)
        p = _lib.FlashParams()
        p.q, p.k, p.v, p.out = (tensor_desc(t, True) for t in (dq, dk, dv, o))
        p.log_normalizer = L.data_ptr()
        p.batch, p.heads_q, p.heads_kv, p.qo_len, p.kv_len, p.head_dim, p.causal = 1, h, hkv, m, n, d, causal
        p.dtype = p.out_dtype = DTYPE_CODE[torch.float16]
        p.sm_scale = d ** -0.5
        need = _run(lib, p, "flash_attn_fwd", workspace and cut, gpu_device)
        share = 2 * 256 * (d + 1) * 4
        assert (need % share == 0 and 0 < need // share <= 256) if cut else need == 0
        res.append((o, L))
    torch.testing.assert_close(res[0][0].float(), res[1][0].float(), atol=2e-3, rtol=1e-2)
    inf = torch.isinf(res[1][1])
    assert torch.equal(torch.isinf(res[0][1]), inf)
    torch.testing.assert_close(res[0][1][~inf], res[1][1][~inf], atol=2e-3, rtol=2e-4)
    per = h // hkv
    for j in sorted({0, hkv - 1}):  # the reference's own rule on one head
        a, kv = slice(j * per, j * per + 1), slice(j, j + 1)
        ref, _ = FO.attention(q[:, a], k[:, kv], v[:, kv], causal, return_log_normalizer=True, upcast=True)
        yard = FO.max_diff(FO.attention(q[:, a], k[:, kv], v[:, kv], causal, upcast=False), ref)
        assert FO.max_diff(res[0][0][:, a].cpu(), ref) <= 2 * yard + 1e-5
