"""Lists walked in two halves by one workgroup: at most as many Q tiles as compute units and more than half as many."""
import pytest
import torch

from sparseattention_amd import _native, compute_mask_kernel, sparse_attention, workloads as W
from sparseattention_amd.mask_utils import MaskMetadata

pytestmark = pytest.mark.gpu


def exact(q, k, v, mask):
    s = (q.double() @ k.double().transpose(-1, -2).contiguous()) * q.shape[-1] ** -0.5
    s = s.masked_fill(~mask, float("-inf"))
    lse = torch.logsumexp(s, -1)
    return torch.exp(s - lse.masked_fill(lse.isinf(), 0.0)[..., None]) @ v.double(), lse


@pytest.mark.parametrize("dtype,B,H,Sq,Sk,D,BQ,BK", [
    (torch.bfloat16, 1, 32, 1024, 3136, 128, 128, 64),  # 256 Q tiles, the shortest rows
    (torch.bfloat16, 3, 43, 128, 3200, 128, 128, 128),  # 129 Q tiles, an odd number of planes, 25 entries of two chunks
    (torch.float16, 1, 13, 640, 1088, 64, 64, 32),      # 130 Q tiles
    (torch.float16, 2, 33, 256, 3104, 128, 128, 32),    # a last chunk that is not full
    (torch.bfloat16, 1, 3, 4096, 2048, 64, 64, 1024),   # fewer entries than chunks
    (torch.bfloat16, 2, 3, 1920, 1216, 128, 64, 64),    # 180 Q tiles of 64 rows at D = 128, 19 chunks
    (torch.float16, 1, 17, 1024, 3168, 64, 128, 32),    # 136 Q tiles of 128 rows at D = 64
])
@pytest.mark.parametrize("packed", [True, False])
def test_halves_against_float64(gpu, dtype, B, H, Sq, Sk, D, BQ, BK, packed):
    assert _native.load().sa_fwd_split_workspace_bytes(B, H, Sq, Sk, D, BQ, BK, {torch.bfloat16: 0, torch.float16: 1}[dtype]) == 0
    q, _, _ = W.qkv(B, H, Sq, D, dtype, seed=1, device=gpu)
    assert _native.host().forward_lists(q, Sk, BQ, BK, None) == "halves"
    _, k, v = W.qkv(B, H, Sk, D, dtype, seed=2, device=gpu)
    g = torch.Generator(device=gpu).manual_seed(BK)
    nq, nk = Sq // BQ, Sk // BK
    # tiles empty, full or of coin flips; lists grow with the Q tile from one entry to all that there are (too short for halves, odd
    # numbers of chunks), the last Q tile of plane 0 attends to none where there is another
    kind = torch.randint(0, 3, (B, 1, nq, nk), device=gpu, generator=g)
    reach = torch.tensor([nk if nq == 1 else 1 + (nk - 1) * t // (nq - 1) for t in range(nq)], device=gpu)
    kind[:, :, torch.arange(nk, device=gpu)[None, :] >= reach[:, None]] = 0
    if nq > 1:
        kind[0, :, -1] = 0
    kind[-1, :, 0, 0] = 2
    up = kind.repeat_interleave(BQ, 2).repeat_interleave(BK, 3)
    mask = (up == 2) | ((up == 1) & (torch.rand(B, 1, Sq, Sk, device=gpu, generator=g) < 0.5))
    mask[0, :, 5] = False
    me = mask.expand(B, H, Sq, Sk)
    md = compute_mask_kernel(me, BQ, BK, pack_partial=packed)
    o, lse = sparse_attention(q, k, v, me, BQ, BK, mask_metadata=md, return_lse=True)
    again, _ = sparse_attention(q, k, v, me, BQ, BK, mask_metadata=md, return_lse=True)
    assert torch.equal(o, again)
    live = mask.any(-1).expand(B, H, Sq)
    assert torch.equal(torch.isfinite(lse), live) and (o[~live] == 0).all()
    for b in range(B):
        want, want_lse = exact(q[b, :3], k[b, :3], v[b, :3], mask[b])
        want = torch.where(live[b, :3, :, None], want, 0.0)
        # P and the output are rounded to 8 (bf16) or 11 bits: half a unit of each, and as much of the scaled queries
        eps = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
        err = (o[b, :3].double() - want).norm() / want.norm().clamp(min=1e-30)
        assert err <= 2 * eps, float(err)
        if live[b, :3].any():
            assert (lse[b, :3] - want_lse)[live[b, :3]].abs().max() <= 16 * eps


# (tiles in 1/256 of the compute units: lists that differ in length finish sooner in parts than in halves there, and were shared before)
@pytest.mark.parametrize("tiles,chunks,D,BQ", [(136, 73, 128, 128), (136, 96, 64, 128), (176, 128, 128, 128), (192, 192, 128, 128), (224, 80, 64, 128),
                                               (240, 256, 128, 128), (255, 96, 128, 128), (256, 97, 128, 128), (256, 256, 64, 128),
                                               (136, 97, 64, 64), (170, 97, 128, 64), (224, 128, 128, 64), (240, 256, 128, 64), (255, 97, 128, 64)])
def test_long_uneven_lists_are_shared(gpu, tiles, chunks, D, BQ):
    cus = torch.cuda.get_device_properties(gpu).multi_processor_count
    if cus % 256:
        pytest.skip("the numbers are those of 256 compute units")
    lib = _native.load()
    assert lib.sa_fwd_split_workspace_bytes(1, tiles * cus // 256, BQ, 64 * chunks, D, BQ, 64, 0) > 0


@pytest.mark.parametrize("D,BQ", [(128, 128), (64, 128), (128, 64), (64, 64)])
def test_infinite_values_that_lists_name(gpu, D, BQ):
    """An infinity or a NaN in V reaches its column of the result whichever half holds it, and no other column."""
    B, H, Sk, BK = 1, 32, 3200, 64
    Sq = 8 * BQ
    q, _, _ = W.qkv(B, H, Sq, D, torch.bfloat16, seed=5, device=gpu)
    _, k, v = W.qkv(B, H, Sk, D, torch.bfloat16, seed=6, device=gpu)
    mask = torch.ones(B, 1, Sq, Sk, dtype=torch.bool, device=gpu)
    mask[..., : BQ + 5, 2 * Sk // 3:] = False  # (rows that attend to none of the second infinity)
    me = mask.expand(B, H, Sq, Sk)
    want, _ = exact(q[0], k[0], v[0], mask[0])
    v[..., 70, 3], v[..., -70, 9] = float("inf"), float("-inf")  # (the first half's, the second half's)
    v[..., 300, 17], v[..., -300, 31] = float("nan"), float("nan")
    assert _native.host().forward_lists(q, Sk, BQ, BK, None) == "halves"
    o = sparse_attention(q, k, v, me, BQ, BK, mask_metadata=compute_mask_kernel(me, BQ, BK))[0].double()
    # (where a tile is listed, the keys of it that a row does not attend to have a weight of 0: 0 times these is NaN)
    far = slice(2 * BQ, Sq)
    assert torch.isposinf(o[..., 3]).all() and torch.isneginf(o[:, far, 9]).all()
    assert torch.isnan(o[..., 17]).all() and torch.isnan(o[:, far, 31]).all()
    near = slice(0, BQ)  # (their lists end before the second ones)
    assert torch.isfinite(o[:, near, 9]).all() and torch.isfinite(o[:, near, 31]).all()
    rest = [d for d in range(D) if d not in (3, 9, 17, 31)]
    assert ((o[..., rest] - want[..., rest]).norm() / want[..., rest].norm()) <= 2.0 ** -7


def test_halves_with_infinite_values_and_entries_out_of_range(gpu):
    """What a list does not name does not reach the result; an entry outside K leaves other Q tiles alone and is left out."""
    B, H, Sq, Sk, D, BQ, BK = 1, 32, 1024, 3200, 128, 128, 64
    q, _, _ = W.qkv(B, H, Sq, D, torch.bfloat16, seed=3, device=gpu)
    _, k0, v0 = W.qkv(B, H, Sk, D, torch.bfloat16, seed=4, device=gpu)
    k, v = k0.clone(), v0.clone()
    k[:, :, :64] = float("nan")
    v[:, :, :64] = float("inf")
    mask = torch.zeros(1, 1, Sq, Sk, dtype=torch.bool, device=gpu)
    for t in range(Sq // BQ):  # lists of 2 .. 44 entries, none of them the first
        mask[..., BQ * t:BQ * (t + 1), 64:64 * (6 * t + 3)] = True
    me = mask.expand(B, H, Sq, Sk)
    md = compute_mask_kernel(me, BQ, BK)
    o = sparse_attention(q, k, v, me, BQ, BK, mask_metadata=md)
    want, _ = exact(q[0, :3, :, :], k[0, :3, 64:], v[0, :3, 64:], mask[0, :, :, 64:])
    assert torch.isfinite(o).all() and ((o[0, :3].double() - want).norm() / want.norm()) <= 2.0 ** -7
    ids = md.unmasked_kv_ids.clone()
    ids[..., 7, 2], ids[..., 7, 6] = Sk // BK, -1
    bad = MaskMetadata(ids, md.unmasked_lens.clone(), md.masked_kv_ids, md.masked_lens, md.packed_masks)
    from sparseattention_amd.mask_utils import validation_key
    bad._validated_for = validation_key(bad, Sk, BK)  # (past the wrapper's own check)
    got = sparse_attention(q, k0, v0, me, BQ, BK, mask_metadata=bad)  # (such an entry's keys are read as the first ones)
    assert torch.equal(got[:, :, :7 * BQ], o[:, :, :7 * BQ])
    left = mask[0, :, 7 * BQ:].clone()
    left[..., 64 * 3:64 * 4] = left[..., 64 * 7:64 * 8] = False
    want, _ = exact(q[0, :3, 7 * BQ:], k[0, :3, 64:], v[0, :3, 64:], left[..., 64:])
    assert ((got[0, :3, 7 * BQ:].double() - want).norm() / want.norm()) <= 2.0 ** -7
