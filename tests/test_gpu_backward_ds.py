"""The backward whose dQ comes from stored dS (D = 128, packed tiles, 512 key tiles and more): masks with blocks no pass visits,
a query without a key and a key without a query, one group of planes and several."""
import math

import pytest
import torch

from sparseattention_amd import compute_backward_metadata, compute_mask_kernel, sparse_attention, sparse_attention_backward
from sparseattention_amd import _native

pytestmark = pytest.mark.gpu


def _poison(nbytes, gpu):
    """Leaves NaN patterns in the memory that the next workspace of this size is taken from."""
    torch.full((nbytes,), 0xFF, dtype=torch.uint8, device=gpu)


def _rel(a, b):
    return float((a.double() - b.double()).norm() / b.double().norm())


# Outputs of a correct backward are within 3.2e-3 (bf16) and 3.8e-4 (fp16) of float64 in the relative 2-norm; twice that.
@pytest.mark.parametrize("dtype,tol", [(torch.bfloat16, 6.4e-3), (torch.float16, 8e-4)])
@pytest.mark.parametrize("B,H,Sq,Sk", [(2, 32, 1024, 1024), (1, 57, 128, 1152), (4, 128, 128, 128)])
def test_gradients_against_float64(gpu, dtype, tol, B, H, Sq, Sk):
    assert _native.load().sa_bwd_workspace_bytes_ex(B, H, Sq, Sk, 128) > B * H * Sq * Sk * 2
    g = torch.Generator().manual_seed(Sq + Sk)
    q, k, v, do = (torch.randn(B, H, S, 128, generator=g).to(gpu, dtype) for S in (Sq, Sk, Sk, Sq))
    mask = torch.rand(B, 1, Sq, Sk, generator=g) < 0.6
    mask[..., : Sk // 2] = True                       # FULL tiles
    mask[:, :, Sq // 2:, Sk // 4: Sk // 2] = False    # EMPTY ones
    mask[:, :, :64, Sk - 128:] = False                # empty for the key pass, half of a PARTIAL tile for the query pass
    mask[0, 0, 3] = False                             # a query without a key
    mask[0, 0, :, 5] = False                          # a key without a query
    mask = mask.to(gpu).expand(B, H, Sq, Sk)
    o, lse = sparse_attention(q, k, v, mask, 128, 64, return_lse=True)
    bmd = compute_backward_metadata(mask)
    _poison(_native.load().sa_bwd_workspace_bytes_ex(B, H, Sq, Sk, 128), gpu)
    got = sparse_attention_backward(do, q, k, v, o, lse, None, bmd)

    q64, k64, v64 = (t.double().requires_grad_(True) for t in (q, k, v))
    s = (q64 @ k64.transpose(-1, -2).contiguous()) * 128 ** -0.5
    (torch.softmax(s.masked_fill(~mask, float("-inf")), -1).nan_to_num() @ v64).backward(do.double())
    for x, t in zip(got, (q64, k64, v64)):
        assert torch.isfinite(x).all()
        assert _rel(x, t.grad.nan_to_num()) <= tol


def test_planes_in_groups(gpu):
    """9 planes of 512 MiB of dS: groups of five and four through one workspace, against the passes that store nothing."""
    B, H, S = 1, 9, 16384
    assert 5 * S * S * 2 <= _native.load().sa_bwd_workspace_bytes_ex(B, H, S, S, 128) <= 5 * S * S * 2 + B * H * S * 8 + 1024
    g = torch.Generator(device=gpu).manual_seed(1)
    q, k, v, do = (torch.randn(B, S, H, 128, device=gpu, generator=g, dtype=torch.bfloat16).transpose(1, 2) for _ in range(4))
    i = torch.arange(S, device=gpu)
    mask = ((i[None] <= i[:, None]) & (i[:, None] - i[None] < 300))[None, None].expand(B, H, S, S)
    o, lse = sparse_attention(q, k, v, mask, 128, 64, compute_mask_kernel(mask, 128, 64), return_lse=True)
    _poison(5 * S * S * 2 + B * H * S * 8, gpu)
    got = sparse_attention_backward(do, q, k, v, o, lse, None, compute_backward_metadata(mask))
    want = sparse_attention_backward(do, q, k, v, o, lse, mask, compute_backward_metadata(mask, pack_partial=False))
    for x, y in zip(got, want):
        assert torch.isfinite(x).all()
        assert _rel(x, y) <= 6.4e-3


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_past_the_caches_or_through_them(gpu, dtype):
    """33 planes of 32 MiB of dS: more than 1 GiB in one group, which goes past the caches from the last plane on, or in groups of
    seventeen and sixteen, which do not.  The same bits."""
    B, H, S, D = 1, 33, 4096, 128
    lib, st, plane = _native.load(), _native.strides, S * S * 2
    g = torch.Generator(device=gpu).manual_seed(2)
    q, k, v, do = (torch.randn(B, H, S, D, device=gpu, generator=g, dtype=dtype) for _ in range(4))
    i = torch.arange(S, device=gpu)
    mask = ((i[None] <= i[:, None]) & (i[:, None] - i[None] < 900))[None, None].expand(B, H, S, S)
    o, lse = sparse_attention(q, k, v, mask, 128, 64, return_lse=True)
    bmd = compute_backward_metadata(mask)
    lists, packs = [], []
    for md in (bmd.by_query, bmd.by_key):
        for t in (md.unmasked_kv_ids, md.unmasked_lens, md.masked_kv_ids, md.masked_lens):
            lists += [t.data_ptr(), st(t.stride())]
        packs += [md.packed_masks.data_ptr(), st(md.packed_masks.stride()[:2])]

    def gradients(planes):
        nbytes = lib.sa_bwd_workspace_bytes_within(B, H, S, S, D, planes * plane + B * H * S * 8 + 1024)
        assert planes * plane < nbytes <= planes * plane + B * H * S * 8 + 1024
        out, ws = [torch.full_like(t, float("nan")) for t in (q, k, v)], torch.full((nbytes,), 0xFF, dtype=torch.uint8, device=gpu)
        tensors = [x for t in (q, k, v, o, do, lse, *out) for x in (t.data_ptr(), st(t.stride()))]
        _native.check(lib.sa_sparse_attention_bwd(*tensors, None, None, None, None, *packs, *lists, ws.data_ptr(), nbytes, B, H, S, S, D,
                                                  _native.SA_DTYPE_BF16 if dtype == torch.bfloat16 else _native.SA_DTYPE_FP16,
                                                  D ** -0.5 / math.log(2), torch.cuda.current_stream().cuda_stream))
        torch.cuda.synchronize()
        return out

    want = gradients(33)
    assert not any(torch.isnan(t).any() for t in want)
    assert all(torch.equal(a, b) for a, b in zip(gradients(17), want))


@pytest.mark.parametrize("B,H,Sq,Sk", [(2, 8, 384, 4096), (9, 8, 128, 1024), (11, 8, 256, 768), (16, 8, 384, 512), (8, 8, 1152, 1024),
                                         (3, 12, 384, 1920), (1, 4, 128, 16384)])
def test_planes_of_an_xcd_side_by_side(gpu, B, H, Sq, Sk):
    """Two, nine, eleven (one by one), sixteen (by eights) and eight planes to an XCD; last blocks of 32 workgroups that are not full; planes
    shared by two XCDs."""
    test_gradients_against_float64(gpu, torch.bfloat16, 6.4e-3, B, H, Sq, Sk)
