"""Masks that have to be staged (copied into padded rows) show their present contents on every call: after writes that the
tensor object does not record, in captured graphs, and as inference tensors."""
import pytest
import torch


def _masks(m, n, dev):
    """(mask, causal flag) per kind of staging; n is not a multiple of 16 bytes of entries."""
    g = torch.Generator().manual_seed(7)
    keep = torch.rand(1, 1, m, n, generator=g) > 0.4
    keep[..., 0] = True  # (no query without a key)
    bias = torch.randn(1, 2, m, n, generator=g)
    return {"bool": (keep.to(dev), False), "bool_causal": (keep.to(dev), True), "fp16": (bias.half().to(dev), False), "fp32": (bias.to(dev), False)}


def _flip(mask):
    """Other contents, written where the mask's version counter does not see it."""
    if mask.dtype == torch.bool:
        mask.data[..., 1:].logical_not_()
    else:
        mask.data.neg_()


KINDS = ["bool", "bool_causal", "fp16", "fp32"]


@pytest.mark.parametrize("kind", KINDS)
def test_contents_are_copied_on_every_call(kind):
    from flagattention_amd.sage_attention import attention as A

    mask, causal = _masks(9, 37, "cpu")[kind]
    dev = torch.device("cpu")

    def staged(mask):
        if mask.dtype == torch.bool:
            return A._staged_cached(mask, 2, 2, 9, 37, causal, dev, 0).tensor
        return A._staged_additive_cached(mask, 2, 2, 9, 37, dev, 0)

    def want():
        w = mask.expand(2, 2, 9, 37)
        return w & (torch.arange(37)[None, :] <= torch.arange(9)[:, None] + 28) if causal else w

    A._STAGED.clear()
    first = staged(mask)
    assert torch.equal(first, want())
    version = mask._version
    _flip(mask)
    assert mask._version == version
    assert torch.equal(staged(mask), want())
    if mask.is_floating_point():
        mask.requires_grad_()
        assert not staged(mask).requires_grad
        mask = mask.detach()
    with torch.inference_mode():
        fresh = mask.clone()  # (a tensor without a version counter)
        assert torch.equal(staged(fresh), want())
    assert torch.equal(staged(fresh), want())  # ... whose buffer is filled again outside inference mode
    A._STAGED.clear()


def _inputs(dev, m, n):
    from flag_attn import sage_attention as sa

    g = torch.Generator().manual_seed(8)
    q, k, v = (torch.randn(1, 2, x, 64, generator=g).half().to(dev) for x in (m, n, n))
    q8, qs, k8, ks = sa.per_block_int8(q, k)
    return lambda mask, causal: sa.sage_attention(q8, k8, v, qs, ks, attn_mask=mask, causal=causal, return_lse=True)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", KINDS)
def test_unrecorded_writes_are_seen(kind, gpu_device):
    run = _inputs(gpu_device, 300, 501)
    mask, causal = _masks(300, 501, gpu_device)[kind]
    results = []
    for _ in range(3):
        results.append(run(mask, causal))
        assert all(torch.equal(a, b) for a, b in zip(results[-1], run(mask.clone(), causal)))
        _flip(mask)
    assert not torch.equal(results[0][0], results[1][0]) and torch.equal(results[0][0], results[2][0])


@pytest.mark.gpu
@pytest.mark.parametrize("warm", [True, False])  # whether a call on the capture stream has staged the mask before
@pytest.mark.parametrize("kind", KINDS)
def test_a_captured_graph_stages_its_mask(kind, warm, gpu_device):
    """Every replay shows the mask's contents at that time, in memory of the graph's own; an eager call after the capture
    does not depend on a replay."""
    run = _inputs(gpu_device, 300, 501)
    mask, causal = _masks(300, 501, gpu_device)[kind]
    other = _masks(300, 499, gpu_device)[kind][0]
    run_other = _inputs(gpu_device, 300, 499)
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        run_other(other, causal)
        if warm:
            run(mask, causal)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        captured = run(mask, causal)
    with torch.cuda.stream(side):
        eager = run(mask, causal)
    torch.cuda.synchronize()
    assert all(torch.equal(a, b) for a, b in zip(eager, run(mask.clone(), causal)))
    for rep in range(4):
        if rep % 2:
            _flip(mask)
        with torch.cuda.stream(side):
            run_other(other, causal)  # another mask staged on the capture stream, and memory like the staged masks' taken
            kept = [torch.full((x,), 3, dtype=torch.uint8, device=gpu_device) for x in (300 * 512, 300 * 1008, 600 * 1008, 600 * 2016)]
        for t in captured:
            t.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(captured, run(mask.clone(), causal))), f"replay {rep}"
        assert all(bool((t == 3).all()) for t in kept), f"replay {rep} wrote to another tensor"
