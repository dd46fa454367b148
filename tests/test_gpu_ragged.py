"""Forward on a tile grid larger than its tensors, and head dims between the kernels': nothing is padded in memory."""
import pytest
import torch

from sparseattention_amd import compute_mask_kernel, select_tiling, sparse_attention, sparse_attention_tiled

pytestmark = pytest.mark.gpu


def inside(B, H, S, D, dtype, seed, device):
    """[B,H,S,D] with NaN before and behind every row and every plane: what a read outside the tensor would bring in."""
    g = torch.Generator().manual_seed(seed)
    big = torch.full((B, H, S + 7, 2 * D), float("nan"))
    big[:, :, 3:3 + S, :D] = torch.randn(B, H, S, D, generator=g)
    return big.to(device, dtype)[:, :, 3:3 + S, :D]


def reference(q, k, v, mask):
    s = (q.double() @ k.double().transpose(-1, -2).contiguous()) * q.shape[-1] ** -0.5
    s = s.masked_fill(~mask, float("-inf"))
    return torch.nan_to_num(torch.softmax(s, -1)) @ v.double(), torch.logsumexp(s, -1)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,H,Sq,Sk,D,BQ,BK,qo,ko", [
    (2, 3, 299, 299, 80, 128, 64, 0, 0),
    (1, 2, 129, 515, 128, 128, 32, 0, 0),     # one row in the last Q tile, three keys in the last KV tile
    (1, 2, 100, 200, 64, 64, 16, 63, 15),     # a grid that starts as far off the tensors as it can
    (1, 1, 33, 65, 8, 32, 128, 0, 0),         # the smallest head dim
    (1, 3, 250, 130, 120, 128, 256, 5, 200),  # a KV tile wider than the keys, and most of it in front of them
    (1, 2, 31, 1, 40, 32, 32, 1, 31),         # one key
])
def test_tiled_forward_without_padding(gpu, dtype, B, H, Sq, Sk, D, BQ, BK, qo, ko):
    q, k, v = (inside(B, H, S, D, dtype, i, gpu) for i, S in enumerate((Sq, Sk, Sk)))
    g = torch.Generator().manual_seed(9)
    i, j = torch.arange(Sq)[:, None], torch.arange(Sk)[None, :]
    mask = ((torch.rand(B, 1, Sq, Sk, generator=g) < 0.8) | (j % 64 < 20)) & (j <= i + Sk // 2)
    mask[0, 0, Sq // 2] = False
    mask = mask.to(gpu).expand(B, H, Sq, Sk)
    t = select_tiling(mask, candidates=((BQ, BK),), offsets=((qo, ko),))
    assert (t.q_offset, t.k_offset) == (qo, ko)
    o, lse = sparse_attention_tiled(q, k, v, t, return_lse=True)
    assert o.shape == q.shape and lse.shape == (B, H, Sq)
    want, want_lse = reference(q, k, v, mask)
    tol = 2e-2 if dtype == torch.bfloat16 else 4e-3
    assert float((o.double() - want).abs().max()) <= tol
    live = torch.isfinite(want_lse)
    assert torch.equal(torch.isfinite(lse), live)
    assert float((lse.double() - want_lse)[live].abs().max()) <= 6e-3 + 2 ** -9 * 6
    assert torch.equal(o, sparse_attention_tiled(q, k, v, t))


@pytest.mark.parametrize("D", [16, 72, 96, 104])
def test_head_dims_between_the_kernels(gpu, D):
    B, H, S = 2, 2, 256
    q, k, v = (inside(B, H, S, D, torch.bfloat16, 20 + i, gpu) for i in range(3))
    mask = torch.rand(S, S, generator=torch.Generator().manual_seed(D)) < 0.5
    mask[:, :64] = True
    mask = mask.to(gpu)[None, None].expand(B, H, S, S)
    o = sparse_attention(q, k, v, mask, 64, 32, compute_mask_kernel(mask, 64, 32))
    want, _ = reference(q, k, v, mask)
    assert o.shape == q.shape and float((o.double() - want).abs().max()) <= 2e-2
    # through padding, as without the packed tiles
    p = sparse_attention(q, k, v, mask, 64, 32, compute_mask_kernel(mask, 64, 32, pack_partial=False))
    assert torch.equal(o, p)


@pytest.mark.parametrize("Sk", [257, 299])
def test_tensors_with_fewer_keys_than_the_mask(gpu, Sk):
    """Keys that the mask has and the tensors do not are keys of zeros."""
    B, H, S, D, qo, ko = 1, 2, 300, 80, 3, 5
    q, k, v = (inside(B, H, n, D, torch.bfloat16, 30 + i, gpu) for i, n in enumerate((S, Sk, Sk)))
    t = select_tiling(torch.ones(B, H, S, S, dtype=torch.bool, device=gpu), candidates=((64, 32),), offsets=((qo, ko),))
    Pq, Pk = t.padded_mask.shape[-2:]
    pad = torch.nn.functional.pad
    want = sparse_attention(pad(q, (0, 0, qo, Pq - qo - S)), *(pad(x, (0, 0, ko, Pk - ko - Sk)) for x in (k, v)), t.padded_mask,
                            64, 32, t.metadata)[:, :, qo:qo + S]
    assert torch.equal(sparse_attention_tiled(q, k, v, t), want)
