"""What the differentiable wrapper hands to hooks on saved tensors: its inputs and results, not the lists of its metadata."""
import pytest
import torch

from sparseattention_amd import compute_backward_metadata, compute_mask_kernel, sparse_attention_trainable, workloads as W

pytestmark = pytest.mark.gpu


def test_hooks_see_inputs_and_results_only(gpu):
    B, H, S, D = 1, 2, 256, 64
    q, k, v = (t.requires_grad_(True) for t in W.qkv(B, H, S, D, torch.bfloat16, seed=3, device=gpu))
    mask = torch.ones(S, S, dtype=torch.bool, device=gpu).tril()[None, None].expand(B, H, S, S)
    md, bmd = compute_mask_kernel(mask, 128, 64), compute_backward_metadata(mask)
    seen = []

    def pack(t):
        seen.append((t.dtype, tuple(t.shape)))
        return t.cpu()

    with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t.to(gpu)):
        o = sparse_attention_trainable(q, k, v, None, 128, 64, md, bmd)
    rows = [(torch.bfloat16, (B, H, S, D))] * 4
    assert sorted(map(str, seen)) == sorted(map(str, rows + [(torch.float32, (B, H, S))]))
    do = torch.randn_like(o)
    got = torch.autograd.grad(o, (q, k, v), do)
    want = torch.autograd.grad(sparse_attention_trainable(q, k, v, None, 128, 64, md, bmd), (q, k, v), do)
    assert all(torch.equal(a, b) for a, b in zip(got, want))
