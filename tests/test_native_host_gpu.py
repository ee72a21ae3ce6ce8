"""Calls whose shape has been seen before take the native host side (csrc/host.cpp): the same results as the first call of
that shape, bit for bit, and everything its key does not cover goes back to the Python checks."""
import threading

import pytest
import torch

pytestmark = pytest.mark.gpu


def _qkv(seed, dev, b=1, h=4, hkv=2, m=77, n=130, d=64, dtype=torch.float16):
    g = torch.Generator().manual_seed(seed)
    return tuple(torch.randn(b, x, s, d, generator=g).to(dtype).to(dev) for x, s in ((h, m), (hkv, n), (hkv, n)))


def _calls(sa, flag_attn, q, k, v, mask):
    q8, qs, k8, ks = sa.per_block_int8(q, k, smooth_k=True)
    plain = sa.per_block_int8(q, k)
    km = sa.per_block_int8(q, k, km=k.mean(dim=2, keepdim=True))
    out = [q8, qs, k8, ks, *plain, *km]
    for kw in ({}, {"return_lse": True, "output_dtype": torch.float32}, {"attn_mask": mask}, {"causal": True}):
        out += list(sa.sage_attention(q8, k8, v, qs, ks, **kw))
    out += [flag_attn.flash_attention(q, k, v), *flag_attn.flash_attention(q, k, v, True, return_log_normalizer=True)[:2]]
    out += list(sa.sageattn(q, k, v, return_lse=True))
    return out


def test_repeated_shapes_give_the_first_call_s_results(gpu_device):
    import flag_attn
    from flag_attn import sage_attention as sa
    from flagattention_amd import _lib

    mask = torch.rand(1, 1, 77, 128, generator=torch.Generator().manual_seed(1)).to(gpu_device) > 0.3
    a, b = _qkv(1, gpu_device, n=128), _qkv(2, gpu_device, n=128)
    first_a = [t.clone() for t in _calls(sa, flag_attn, *a, mask)]
    assert _lib.host().flash(*a, False, None, False) is not None  # (the shape is known now)
    second_b = [t.clone() for t in _calls(sa, flag_attn, *b, mask)]
    again_a = _calls(sa, flag_attn, *a, mask)
    assert all(x.shape == y.shape and x.stride() == y.stride() and torch.equal(x, y) for x, y in zip(first_a, again_a))
    # other inputs of the same shape, in threads of their own (each with a plan table of its own) and on their own streams
    results = {}

    def work(name, args):
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            for _ in range(3):
                results[name] = _calls(sa, flag_attn, *args, mask)
        s.synchronize()

    torch.cuda.synchronize()
    threads = [threading.Thread(target=work, args=(name, args)) for name, args in (("a", a), ("b", b))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert all(torch.equal(x, y) for x, y in zip(results["a"], first_a)) and all(torch.equal(x, y) for x, y in zip(results["b"], second_b))


def test_what_the_key_does_not_cover_is_checked_again(gpu_device):
    import flag_attn
    from flag_attn import sage_attention as sa
    from flagattention_amd import _lib

    q, k, v = _qkv(3, gpu_device)
    want = flag_attn.flash_attention(q, k, v)
    host = _lib.host()
    assert host.flash(q, k, v, False, None, False) is not None
    with pytest.raises(NotImplementedError, match="forward only"):
        flag_attn.flash_attention(q.clone().requires_grad_(), k, v)
    # the same shape and strides, but rows that are not 16-byte aligned: the library refuses them, as on a first call
    shifted = torch.empty(q.numel() + 8, dtype=q.dtype, device=gpu_device)[1:1 + q.numel()].view(q.shape).copy_(q)
    assert shifted.stride() == q.stride() and host.flash(shifted, k, v, False, None, False) is None
    with pytest.raises(_lib.SageHipError, match="aligned"):
        flag_attn.flash_attention(shifted, k, v)
    assert torch.equal(flag_attn.flash_attention(q, k, v), want)
    assert host.flash(q, k[:, :, :100], v[:, :, :100], False, None, False) is None
    assert host.flash(q.cpu(), k, v, False, None, False) is None
    with pytest.raises(RuntimeError):
        flag_attn.flash_attention(q.cpu(), k, v)
    q8, qs, k8, ks = sa.per_block_int8(q, k)
    o, _ = sa.sage_attention(q8, k8, v, qs, ks)
    with pytest.raises(ValueError, match="q_scale"):
        sa.sage_attention(q8, k8, v, qs[..., :0], ks)
    with pytest.raises(ValueError, match="maxnreg"):
        sa.sage_attention(q8, k8, v, qs, ks, maxnreg=0)
    with pytest.raises(ValueError, match="layout"):
        sa.sage_attention(q8, k8, v, qs, ks, "HDN")
    # a mask of a known shape whose contents change, and one of the same shape that has to be staged first
    mask = torch.ones(1, 1, 77, 144, dtype=torch.bool, device=gpu_device)[..., :130]
    for _ in range(2):
        assert torch.equal(sa.sage_attention(q8, k8, v, qs, ks, attn_mask=mask)[0], sa.sage_attention(q8, k8, v, qs, ks, attn_mask=mask.clone())[0])


@pytest.mark.parametrize("first", [True, False])  # whether the captured call is the first of its shape (the Python side) or not
def test_a_captured_graph_owns_its_scratch_memory(gpu_device, first):
    """The partial results of a captured call lie in memory that no other tensor gets while the graph lives, also when later
    calls on the capture stream need more of it; every replay gives the eager result and touches nothing else."""
    import flag_attn
    from flag_attn import sage_attention as sa
    from flagattention_amd import _lib

    n = 1030 if first else 1040
    q, k, v = _qkv(5, gpu_device, m=40, n=n, d=128)
    big = _qkv(6, gpu_device, h=16, hkv=16, m=256, n=4096, d=128)

    def run():
        q8, qs, k8, ks = sa.per_block_int8(q, k, smooth_k=True)
        return [*sa.sage_attention(q8, k8, v, qs, ks, return_lse=True), flag_attn.flash_attention(q, k, v)]

    side = torch.cuda.Stream()
    with torch.cuda.stream(side):  # scratch memory of the capture stream from before the capture
        for other in (big if not first else _qkv(7, gpu_device, m=40, n=1100, d=128),):
            sa.sageattn(*other)
            flag_attn.flash_attention(*other)
        if not first:
            run()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        captured = run()
    want = [t.clone() for t in run()]
    assert _lib.host().flash(q, k, v, False, None, False) is not None
    with torch.cuda.stream(side):
        flag_attn.flash_attention(*_qkv(8, gpu_device, h=32, hkv=32, m=512, n=8192, d=128))
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        kept = [torch.full((1 << s,), 7, dtype=torch.uint8, device=gpu_device) for s in (16, 18, 20, 20, 22, 24)]
    for rep in range(3):
        for t in captured:
            t.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(captured, want)), f"replay {rep}"
        assert all(bool((t == 7).all()) for t in kept), f"replay {rep} wrote to another tensor"


def test_shapes_that_return_stay_known(gpu_device):
    """A hundred shapes that come once each, as the keys of a growing cache do, do not push out the plan of a shape that is
    used between them; plans that are not used go."""
    import flag_attn
    from flagattention_amd import _lib

    host = _lib.host()
    q, k, v = _qkv(9, gpu_device, m=1, n=400)
    kept, first = (q, k[:, :, :290], v[:, :, :290]), (q, k[:, :, :300], v[:, :, :300])
    flag_attn.flash_attention(*kept)
    for n in range(300, 400):
        flag_attn.flash_attention(q, k[:, :, :n], v[:, :, :n])
        assert host.flash(*kept, False, None, False) is not None, n
    assert host.flash(q, k[:, :, :399], v[:, :, :399], False, None, False) is not None
    assert host.flash(*first, False, None, False) is None


def test_the_python_side_alone_gives_the_same_results(gpu_device, monkeypatch):
    import flag_attn
    from flag_attn import sage_attention as sa
    from flagattention_amd import _lib

    mask = torch.rand(1, 1, 77, 128, generator=torch.Generator().manual_seed(1)).to(gpu_device) > 0.3
    q, k, v = _qkv(10, gpu_device, n=128)
    for _ in range(2):
        want = _calls(sa, flag_attn, q, k, v, mask)
    monkeypatch.setattr(_lib, "_host_module", _lib._PythonHost)
    for _ in range(2):
        got = _calls(sa, flag_attn, q, k, v, mask)
        assert all(x.shape == y.shape and x.stride() == y.stride() and torch.equal(x, y) for x, y in zip(want, got))
