"""The gradient passes as one launch: tile counts that are no multiple of eight, passes of unequal length, and every source of
the PARTIAL tiles' mask entries."""
import pytest
import torch

from sparseattention_amd import BackwardMetadata, compute_backward_metadata, compute_mask_kernel, sparse_attention, sparse_attention_backward

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,tol", [(torch.bfloat16, 2e-2), (torch.float16, 4e-3)])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("B,H,Sq,Sk", [(1, 1, 128, 128), (1, 1, 128, 1152), (1, 3, 896, 128), (3, 3, 384, 640)])
def test_passes_of_every_length(gpu, dtype, tol, D, B, H, Sq, Sk):
    g = torch.Generator().manual_seed(Sq + Sk)
    q, k, v, do = (torch.randn(B, H, S, D, generator=g).to(gpu, dtype) for S in (Sq, Sk, Sk, Sq))
    mask = torch.rand(B, 1, Sq, Sk, generator=g) < 0.6
    mask[..., : Sk // 2] = True             # FULL tiles
    mask[:, :, Sq // 2:, Sk // 4: Sk // 2] = False  # EMPTY ones
    mask[0, 0, 3] = False                   # a query without a key
    mask[0, 0, :, 5] = False                # a key without a query
    mask = mask.to(gpu).expand(B, H, Sq, Sk)
    o, lse = sparse_attention(q, k, v, mask, 128, 64, return_lse=True)
    packed = sparse_attention_backward(do, q, k, v, o, lse, None, compute_backward_metadata(mask))

    q32, k32, v32 = (t.float().requires_grad_(True) for t in (q, k, v))
    s = (q32 @ k32.transpose(-1, -2).contiguous()) * D ** -0.5
    p = torch.softmax(s.masked_fill(~mask, float("-inf")), -1).nan_to_num()
    (p @ v32).backward(do.float())
    for got, t in zip(packed, (q32, k32, v32)):
        assert torch.isfinite(got).all()
        assert float((got.float() - t.grad.nan_to_num()).abs().max()) <= tol * max(1.0, float(t.grad.nan_to_num().abs().max()))

    # the mask entries from the bool tensors, and packed for one side only: the same gradients bit for bit
    plain = compute_backward_metadata(mask, pack_partial=False)
    by_query = compute_mask_kernel(mask, 128, 64, pack_partial=True)
    one_sided = BackwardMetadata(by_query, plain.by_key, plain.transposed_mask)
    for other in (plain, one_sided):
        again = sparse_attention_backward(do, q, k, v, o, lse, mask, other)
        assert all(torch.equal(a, b) for a, b in zip(packed, again))
