"""What the differentiable wrapper keeps of its mask and of its backward metadata, and when it looks at them."""
import pytest
import torch

from sparseattention_amd import compute_backward_metadata, sparse_attention_trainable, workloads as W

pytestmark = pytest.mark.gpu
B, H, S, D = 2, 3, 256, 64


def case(gpu):
    q, k, v = (t.requires_grad_(True) for t in W.qkv(B, H, S, D, torch.bfloat16, seed=3, device=gpu))
    return q, k, v, torch.ones(S, S, dtype=torch.bool, device=gpu).tril(), torch.randn_like(q)


@pytest.mark.parametrize("dims", [2, 4])
@pytest.mark.parametrize("listed", [False, True])
def test_hooks_see_the_mask_as_it_was_passed(gpu, dims, listed):
    q, k, v, mask, do = case(gpu)
    if dims == 4:
        mask = mask[None, None]
    bmd = compute_backward_metadata(mask.expand(B, H, S, S)) if listed else None
    seen = []

    def pack(t):
        seen.append((t.dtype, tuple(t.shape)))
        return t.cpu()

    with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t.to(gpu)):
        o = sparse_attention_trainable(q, k, v, mask, 128, 64, None, bmd)
    assert [shape for dtype, shape in seen if dtype == torch.bool] == [tuple(mask.shape)]
    got = torch.autograd.grad(o, (q, k, v), do)
    want = torch.autograd.grad(sparse_attention_trainable(q, k, v, mask, 128, 64), (q, k, v), do)
    assert all(torch.equal(a, b) for a, b in zip(got, want))


def test_metadata_is_looked_at_in_the_backward(gpu):
    q, k, v, mask, do = case(gpu)
    other = compute_backward_metadata(mask[:128, :128].expand(B, H, 128, 128))  # of other sizes
    with torch.no_grad():  # nothing to differentiate: never looked at
        want = sparse_attention_trainable(q, k, v, mask, 128, 64)
        assert torch.equal(sparse_attention_trainable(q, k, v, mask, 128, 64, None, other), want)
    o = sparse_attention_trainable(q, k, v, mask, 128, 64, None, other)
    with pytest.raises(ValueError):
        torch.autograd.grad(o, (q, k, v), do)
    # counts changed in place between the two are checked against the tiles there are
    bmd = compute_backward_metadata(mask.expand(B, H, S, S))
    o = sparse_attention_trainable(q, k, v, mask, 128, 64, None, bmd)
    bmd.by_key.unmasked_lens.fill_(S)
    with pytest.raises(ValueError):
        torch.autograd.grad(o, (q, k, v), do)


def test_trace(gpu):
    """A trace keeps the call itself, so that other inputs and their gradients go through it."""
    q, k, v, mask, do = case(gpu)
    bmd = compute_backward_metadata(mask.expand(B, H, S, S))
    call = lambda *t: sparse_attention_trainable(*t, mask, 128, 64, None, bmd)  # noqa: E731
    traced = torch.jit.trace(call, (q, k, v))
    other = tuple(t.requires_grad_(True) for t in W.qkv(B, H, S, D, torch.bfloat16, seed=4, device=gpu))
    want = call(*other)
    for _ in range(2):
        got = traced(*other)
        assert torch.equal(got, want)
        grads = torch.autograd.grad(got, other, do)
        assert all(torch.equal(a, b) for a, b in zip(grads, torch.autograd.grad(want, other, do, retain_graph=True)))
