"""Tiles left out under a mask tensor that the heads share (csrc/mask_scan.hip): the launch with the scan (workspace given) against
the one that visits every tile (no workspace), and against the oracle's arithmetic through the latter's own tests."""
import ctypes
import math

import pytest
import torch

from flagattention_amd import _lib
from flagattention_amd.sage_attention import attention as A
from flagattention_amd.sage_attention._common import tensor_desc

gpu = pytest.mark.gpu
KIND = {torch.bool: _lib.MASK_BOOL, torch.float16: _lib.MASK_F16, torch.bfloat16: _lib.MASK_BF16, torch.float32: _lib.MASK_F32}


def _params(q8, qs, k8, ks, v, mask, o, lse, kind, hnd):
    p = _lib.AttnParams()
    p.q, p.k, p.v, p.out = (tensor_desc(t, hnd) for t in (q8, k8, v, o))
    if hnd:
        (b, h, m, d), (_, hkv, n, _) = q8.shape, k8.shape
    else:
        (b, m, h, d), (_, n, hkv, _) = q8.shape, k8.shape
    p.batch, p.heads_q, p.heads_kv, p.qo_len, p.kv_len, p.head_dim = b, h, hkv, m, n, d
    code = {torch.float16: _lib.SAGE_F16, torch.bfloat16: _lib.SAGE_BF16, torch.float32: _lib.SAGE_F32}
    p.v_dtype, p.out_dtype, p.mask_kind = code[v.dtype], code[o.dtype], kind
    p.q_scale, p.k_scale, p.lse = qs.data_ptr(), ks.data_ptr(), lse.data_ptr()
    mask = mask.expand(b, h, m, n)
    p.mask = mask.data_ptr()
    p.mask_stride_b, p.mask_stride_h, p.mask_stride_m, p.mask_stride_n = mask.stride()
    return p


def _inputs(b, h, hkv, m, n, d, dt, hnd, scale=1.0):
    g = torch.Generator().manual_seed(3 * n + m)
    dev = "cuda:0"

    def t(heads, length):
        return torch.randint(-127, 128, (b, heads, length, d) if hnd else (b, length, heads, d), generator=g, dtype=torch.int8).to(dev)

    q8, k8 = t(h, m), t(hkv, n)
    qs = (torch.rand(b, h, -(-m // 128), generator=g) * 2e-3 * scale + 1e-4).to(dev)
    ks = (torch.rand(b, hkv, -(-n // 64), generator=g) * 2e-2 + 1e-3).to(dev)
    v = torch.randn(k8.shape, generator=g).to(dt).to(dev)
    return q8, qs, k8, ks, v


def _mask(kind, dt, b, m, n):
    """Masks shared by the heads."""
    dev = "cuda:0"
    g = torch.Generator().manual_seed(n)
    cols, rows = torch.arange(n), torch.arange(m).view(m, 1) + (n - m)
    lengths = torch.tensor([n // 2 + 3 + 70 * i for i in range(b)]).view(b, 1, 1, 1)
    if kind == "padding":
        keep = (cols < lengths).expand(b, 1, 1, n)
    elif kind == "causal_padding":
        keep = (cols < lengths) & (cols <= rows)
    elif kind == "left":  # left padding under the causal mask: the first rows see no key
        keep = (cols >= n - lengths) & (cols <= rows)
    elif kind == "window":
        keep = ((cols <= rows) & (cols > rows - 100)).view(1, 1, m, n)
    elif kind == "holes":  # any pattern, some 64-key columns of tiles hidden
        keep = (torch.rand(b, 1, m, n, generator=g) < 0.3) & ((cols // 64) % 3 != 1)
    elif kind == "none":
        keep = torch.zeros(1, 1, m, n, dtype=torch.bool)
    elif kind == "all":  # nothing hidden; one row of all takes one key away in two tiles, the ragged last one is left whole
        keep = torch.ones(1, 1, m, n, dtype=torch.bool)
        keep[0, 0, m - 1, 70] = keep[0, 0, 5, 200] = False
    elif kind == "slope":  # a steep linear bias, no hidden keys
        return (-(rows - cols).abs().float() * 3.0).view(1, 1, m, n).to(dt).to(dev)
    if dt is torch.bool:
        return keep.contiguous().to(dev)
    low = -float("inf") if kind == "holes" else torch.finfo(dt).min
    return torch.zeros(keep.shape, dtype=dt).masked_fill_(~keep, low).to(dev)


def _both(q8, qs, k8, ks, v, mask, hnd, out_dt=torch.float32):
    """(o, lse) with the scan, (o, lse) of the launch that visits every tile."""
    lib, res = _lib.load(), []
    b, h = (q8.shape[0], q8.shape[1]) if hnd else (q8.shape[0], q8.shape[2])
    m = q8.shape[2] if hnd else q8.shape[1]
    stream = torch.cuda.current_stream().cuda_stream
    for scan in (True, False):
        o, lse = torch.empty(q8.shape, dtype=out_dt, device=q8.device), torch.empty(b, h, m, device=q8.device)
        p = _params(q8, qs, k8, ks, v, mask, o, lse, KIND[mask.dtype], hnd)
        if scan:
            nbytes = lib.sage_attn_fwd_workspace_bytes(ctypes.byref(p))
            assert nbytes > 0
            ws = torch.full((nbytes,), 0x7f, dtype=torch.uint8, device=q8.device)
            _lib.check(lib.sage_attn_fwd_ws(ctypes.byref(p), ws.data_ptr(), nbytes, stream), "ws")
        else:
            _lib.check(lib.sage_attn_fwd(ctypes.byref(p), stream), "fwd")
        torch.cuda.synchronize()
        res.append((o, lse))
    return res


def _check(res, dt):
    (o, lse), (o_all, lse_all) = res
    # NaN, infinities and empty rows in the same places
    assert torch.equal(torch.isnan(o), torch.isnan(o_all)) and torch.equal(torch.isnan(lse), torch.isnan(lse_all))
    assert torch.equal(torch.isinf(lse), torch.isinf(lse_all))
    fin = torch.isfinite(o_all)
    # The same scores and the same P up to the reference point of a row (which rounds P to 16 bits at another place): one
    # unit of the 16-bit type per term at most
    eps = 2.0 ** -8 if dt is torch.bfloat16 else 2.0 ** -11
    assert (o - o_all)[fin].abs().max().item() <= 4 * eps * o_all[fin].abs().max().item() if fin.any() else True
    lf = torch.isfinite(lse_all)
    if lf.any():  # (fully hidden rows: lse near the type's lowest value)
        assert ((lse - lse_all)[lf].abs() <= 2 * eps + 1e-6 * lse_all[lf].abs()).all()


# b, h, hkv, m, n, d, hnd: few q-blocks, whose tiles are split over runs (a ragged last tile; more than 64 tiles, two per bit; fewer
# tiles than a run of each); more q-blocks than compute units, unsplit (29 tiles: from 28 on every kind of mask is scanned)
SHAPES = [(2, 4, 2, 300, 3072, 64, True), (2, 2, 2, 600, 1608, 128, False), (1, 4, 1, 300, 4304, 64, True), (1, 2, 1, 7, 2000, 64, True),
          (3, 48, 2, 520, 1800, 64, True)]


@gpu
@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("mask_dt", [torch.bool, torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("kind", ["padding", "causal_padding", "left", "window", "holes", "none", "slope"])
def test_scan_changes_nothing(shape, mask_dt, kind):
    b, h, hkv, m, n, d, hnd = shape
    if mask_dt is torch.bool and (kind == "slope" or n % 16):
        pytest.skip("not a bool mask the kernel stages as it is")
    dt = torch.bfloat16 if d == 128 else torch.float16
    x = _inputs(b, h, hkv, m, n, d, dt, hnd)
    mask = _mask(kind, mask_dt, b, m, n)
    _check(_both(*x, mask, hnd), dt)


@gpu
@pytest.mark.parametrize("shape", [(2, 4, 2, 300, 3072, 64, True), (3, 48, 2, 520, 1808, 64, True)])
@pytest.mark.parametrize("mask_dt", [torch.bool, torch.float16, torch.float32])
@pytest.mark.parametrize("kind", ["padding", "causal_padding", "slope", "all"])
def test_what_the_scan_finds(kind, mask_dt, shape):
    """The scan's results as it leaves them in the workspace, and that the rule of the attention kernel, applied to them here,
    leaves out every tile that padding or the causal mask hides from a whole q-block.  Where the largest entry of a tile is 0 its sign
    tells whether the tile is whole and every entry a zero of either sign (bool: visible): +0 for those, -0 for the others."""
    if mask_dt is torch.bool and kind == "slope":
        pytest.skip("not a bool mask")
    b, h, hkv, m, n, d, hnd = shape
    q8, qs, k8, ks, v = _inputs(b, h, hkv, m, n, d, torch.float16, hnd)
    v[1, 0, n - 1, 3], v[0, 1, 70, 9] = float("inf"), float("nan")
    mask = _mask(kind, mask_dt, b, m, n)
    if mask_dt is not torch.bool and kind != "slope":
        mask = torch.where((mask == 0) & (torch.arange(n, device=mask.device) % 3 == 0), torch.full_like(mask, -0.0), mask)
    o, lse = torch.empty(q8.shape, device=q8.device), torch.empty(b, h, m, device=q8.device)
    p = _params(q8, qs, k8, ks, v, mask, o, lse, KIND[mask_dt], hnd)
    lib = _lib.load()
    nbytes = lib.sage_attn_fwd_workspace_bytes(ctypes.byref(p))
    ws = torch.full((nbytes,), 0x7f, dtype=torch.uint8, device=q8.device)
    _lib.check(lib.sage_attn_fwd_ws(ctypes.byref(p), ws.data_ptr(), nbytes, torch.cuda.current_stream().cuda_stream), "ws")
    torch.cuda.synchronize()
    nk, mb, rows = -(-n // 64), mask.shape[0] if mask.stride(0) or mask.shape[0] == 1 else 1, m if p.mask_stride_m else 1
    strips = -(-rows // 16)
    f = ws[: nbytes // 4 * 4].view(torch.float32)
    top, low = f[: mb * strips * nk].view(mb, strips, nk), f[mb * strips * nk: mb * strips * (nk + 1)].view(mb, strips)
    odd = f[mb * strips * (nk + 1): mb * strips * (nk + 1) + b * hkv * nk].view(torch.int32).view(b, hkv, nk)
    e = torch.zeros(mask.shape, device=mask.device).masked_fill_(~mask, float("-inf")) if mask_dt is torch.bool else mask.float()
    e = torch.nn.functional.pad(e[:mb, 0, :rows], (0, nk * 64 - n), value=float("-inf"))
    e = torch.nn.functional.pad(e, (0, 0, 0, strips * 16 - rows), mode="replicate") if strips * 16 > rows else e
    tiles = e.view(mb, strips, 16, nk, 64).amax((2, 4))
    if mask_dt is not torch.bool and n % 64:
        tiles[..., -1].clamp_(min=-1.0e6)
    assert torch.equal(top, tiles) and torch.equal(low, e.view(mb, strips, 16, -1).amax(-1).amin(-1))
    unchanged, zero = (e == 0).view(mb, strips, 16, nk, 64).all(4).all(2), tiles == 0
    assert torch.equal(torch.signbit(top)[zero], ~unchanged[zero])
    assert bool(unchanged.any()) == (kind != "slope") and (bool((zero & ~unchanged).any()) or kind in ("padding", "slope"))
    bad = ~torch.isfinite(torch.nn.functional.pad(v, (0, 0, 0, nk * 64 - n)).view(b, hkv, nk, 64 * d)).all(-1)
    assert torch.equal(odd != 0, bad)
    # the rule: 256-row q-blocks, the largest scales and sums of |q| of the call (a bound above that of every block)
    bound = 256 * ks.max() * (q8.float().abs().sum(-1).amax() * qs.max())
    per = 16 if p.mask_stride_m else 1
    blocks = [slice(i, i + per) for i in range(0, strips, per)]
    left = torch.stack([top[:, s].amax(1) < (0.0 if mask_dt is torch.bool else low[:, s].amin(1, keepdim=True)) - 150.0 - bound for s in blocks], 1)
    hidden = torch.stack([tiles[:, s].amax(1) < -1e4 for s in blocks], 1)
    assert torch.equal(left, hidden) if kind != "slope" else not hidden.any()
    assert left.float().mean() > {"padding": 0.3, "causal_padding": 0.3, "slope": 0.0, "all": -1.0}[kind]


@gpu
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("mask_dt", [torch.bool, torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n", [832, 896, 800])
@pytest.mark.parametrize("rows", ["all", "one"])
def test_tiles_that_the_mask_leaves_as_they_are(rows, n, mask_dt, d):
    """No tile is hidden, one entry changes a score: in every tile it is found where it is (waves of other rows take the steps
    without entries before it, that wave up to it: odd and even numbers of them), and the results are those of the full walk bit for
    bit.  The first mask of each changes nothing at all (additive: zeros of both signs)."""
    b, h, m = 2, 48, 768
    dt = torch.float16 if mask_dt is torch.float16 else torch.bfloat16
    x = _inputs(b, h, 2, m, n, d, dt, True)
    zero = torch.ones(b, 1, m, n, dtype=torch.bool, device="cuda:0") if mask_dt is torch.bool else torch.zeros(b, 1, m, n, dtype=mask_dt, device="cuda:0")
    if mask_dt is not torch.bool:
        zero[:, :, ::3] = -0.0
    plain = None
    for t in [None, *range(n // 64), (n - 1) // 64]:
        mask = zero.clone()
        if t is not None:
            where = (1, 0, slice(None) if rows == "all" else 300 + 7 * t, 64 * t + (5 * t + 3) % 32)
            mask[where] = False if mask_dt is torch.bool else 9.0
        (o, lse), (o_all, lse_all) = _both(*x, mask, True)
        assert torch.equal(o, o_all) and torch.equal(lse, lse_all), t
        if t is None:
            plain = lse
        elif mask_dt is not torch.bool:
            assert (lse[1, :, where[2]] > plain[1, :, where[2]]).any() and torch.equal(lse[0], plain[0])


@gpu
@pytest.mark.parametrize("mask_dt", [torch.bool, torch.bfloat16, torch.float16])
def test_scan_nonfinite(mask_dt):
    """Inf / NaN in V under hidden keys, in a block scale, in a mask entry; scales so large that no entry hides a key."""
    b, h, hkv, m, n, d = 2, 2, 2, 512, 2560, 64
    mask = _mask("causal_padding", mask_dt, b, m, n)
    for what in ("v_inf", "v_nan", "ks_nan", "ks_inf", "qs_nan", "large", "entry"):
        q8, qs, k8, ks, v = _inputs(b, h, hkv, m, n, d, torch.float16, True, scale=1e4 if what == "large" else 1.0)
        mk = mask.clone()
        if what == "v_inf":
            v[0, 1, n - 2, 5] = float("inf")
        elif what == "v_nan":
            v[1, 0, n - 70, 9] = float("nan")
        elif what == "ks_nan":
            ks[0, 1, -1] = float("nan")
        elif what == "ks_inf":
            ks[1, 1, -2] = float("inf")
        elif what == "qs_nan":
            qs[0, 0, 1] = float("nan")
        elif what == "entry":
            if mask_dt is torch.bool:
                continue
            mk[0, 0, 300, 100] = float("nan")
            mk[1, 0, 30, 2500] = float("inf")
        res = _both(q8, qs, k8, ks, v, mk, True)
        if what == "large":  # (exponents of thousands: P is 0 or 1, the rounding of the exponent shows)
            assert torch.equal(torch.isnan(res[0][0]), torch.isnan(res[1][0]))
            continue
        _check(res, torch.float16)


@gpu
@pytest.mark.parametrize("sign", [1, -1])
@pytest.mark.parametrize("mask_dt", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("d", [64, 128])
def test_scores_that_outweigh_their_entries(d, mask_dt, sign):
    """Tiles of entries of -296 that a good part of a row's weight lies in all the same.  sign 1: scores of 150 there and -150
    elsewhere, 0.99 of the difference that the bound on the scores allows.  sign -1: scores of 300 there by negative block
    scales on negative products, -1.5 elsewhere."""
    b, h, m, n = 1, 2, 256, 3072
    dev, dt = "cuda:0", torch.bfloat16 if d == 128 else torch.float16
    q8, qs, k8, ks, v = _inputs(b, h, h, m, n, d, dt, True)
    q8.fill_(127)
    k8.fill_(-127)
    ks.fill_(1e-2 if sign > 0 else 1e-4)
    qs.fill_(150.0 / (127 * 127 * d) / 1e-2)
    mask = torch.zeros(1, 1, m, n, dtype=mask_dt, device=dev)
    for tile in (5, 30, 31, 47):
        keys = slice(64 * tile, 64 * tile + 64)
        mask[..., keys] = -296.0
        if sign > 0:
            k8[:, :, keys] = 127
        else:
            ks[..., tile] = -2e-2
    o, lse = _both(q8, qs, k8, ks, v, mask, True)[0]
    sc = qs.double().repeat_interleave(128, -1)[..., None] * ks.double().repeat_interleave(64, -1)[..., None, :]
    s = (q8.double() @ k8.double().transpose(-1, -2).contiguous()) * sc + mask.double()
    p = torch.softmax(s * math.log(2.0), -1)
    assert p[..., 320:384].sum(-1).min() > 0.1
    # An exponent is off by 2e-4 at most (the scale times 1.5 * 2^23 is near 3700: half of its unit, 1.2e-4; scores near 300: 3e-5 for
    # each of two roundings), P by 1.4e-4 of itself and half a unit of the 16-bit type; twice that for the ratio of two sums
    unit = 2.0 ** -8 if dt is torch.bfloat16 else 2.0 ** -11
    torch.testing.assert_close(o.double(), p @ v.double(), rtol=0, atol=(2.8e-4 + unit) * v.abs().max().item())
    torch.testing.assert_close(lse.double(), torch.logsumexp(s * math.log(2.0), -1) / math.log(2.0), rtol=0, atol=2e-4 + unit)


@gpu
def test_scan_through_the_public_call_and_a_graph():
    from flag_attn import sage_attention as sa

    b, h, m, n, d = 2, 4, 300, 3072, 64
    q8, qs, k8, ks, v = _inputs(b, h, h, m, n, d, torch.bfloat16, True)
    for dt in (torch.bool, torch.bfloat16, torch.float32):
        mask = _mask("causal_padding", dt, b, m, n)
        want = _both(q8, qs, k8, ks, v, mask, True, torch.bfloat16)[1][0]
        for _ in range(2):  # the second call takes the plan of the first
            o, _l = sa.sage_attention(q8, k8, v, qs, ks, attn_mask=mask, output_dtype=torch.bfloat16)
            torch.testing.assert_close(o, want, rtol=2e-2, atol=2e-2)
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            og, _l = sa.sage_attention(q8, k8, v, qs, ks, attn_mask=mask, output_dtype=torch.bfloat16)
        other = _mask("padding", dt, b, m, n).expand(b, 1, m, n).contiguous()
        for i in range(3):  # the scan is part of the graph: it sees what the mask holds when the graph runs
            if i == 2:
                mask.copy_(other)
                want = _both(q8, qs, k8, ks, v, mask, True, torch.bfloat16)[1][0]
            og.zero_()
            g.replay()
            torch.cuda.synchronize()
            torch.testing.assert_close(og, want, rtol=2e-2, atol=2e-2)


@gpu
def test_scan_follows_the_reference_for_bool_masks():
    """A row without any visible key in the 128 x 64 tiles its block visits; blocks of 128 rows of one workgroup that visit
    different tiles (attn_qk_int8_per_block.py:33-36)."""
    from oracle import c_oracle as C

    b, h, m, n, d = 1, 2, 768, 2048, 64
    q8, qs, k8, ks, v = _inputs(b, h, h, m, n, d, torch.float16, True)
    mask = torch.zeros(1, 1, m, n, dtype=torch.bool)
    mask[..., :128, 64:256] = True
    mask[..., 40:50, :] = False     # rows without a visible key in a visited tile
    mask[..., 128:256, 512:576] = True
    mask[..., 300:, 100:700] = torch.rand(m - 300, 600, generator=torch.Generator().manual_seed(1)) < 0.5
    o, lse = A.forward(q8, k8, v, qs, ks, attn_mask=mask.cuda(), output_dtype=torch.float32, return_lse=True)
    want, want_lse = C.attention_blockwise(q8.cpu(), k8.cpu(), v.cpu(), qs.cpu(), ks.cpu(), "HND", attn_mask=mask)
    torch.testing.assert_close(o.cpu(), want.float(), rtol=2e-2, atol=2e-2)
    torch.testing.assert_close(lse.cpu(), want_lse, rtol=1e-4, atol=2e-3)
