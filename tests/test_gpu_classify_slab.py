"""Classification, lists and packed tiles of slabs of megabytes in one launch: rows whose last 16-byte pieces fill a column block or
part of one, with and without a second block to a wave, Q tiles that are no multiple of the rows in flight, planes of their own and
shared ones, rows apart in memory, and both sides of the rule's edges."""
import pytest
import torch

from sparseattention_amd import compute_mask_kernel

pytestmark = pytest.mark.gpu

# (distinct batches, distinct heads, nQ, BQ, Sk, BK, columns between rows)
CASES = [(1, 1, 128, 72, 8192, 64, 8192), (1, 2, 64, 67, 8208, 16, 8208), (2, 1, 64, 128, 8192 + 96, 32, 8192 + 96),
         (1, 1, 130, 33, 16384 + 16, 16, 16384 + 512), (1, 1, 128, 24, 32768 - 128, 128, 32768), (1, 1, 128, 17, 32768 + 1024, 1024, 32768 + 1024),
         (1, 1, 127, 72, 8192, 64, 8192), (1, 1, 128, 72, 8176, 16, 8176), (1, 1, 128, 64, 8192, 64, 8192),   # the three-launch and the small form
         (1, 1, 128, 17, 32784, 16, 32784)]                                                                    # more tiles than LDS holds


@pytest.mark.parametrize("uB,uH,nQ,BQ,Sk,BK,pitch", CASES)
def test_lists_and_bits(gpu, uB, uH, nQ, BQ, Sk, BK, pitch):
    g = torch.Generator(device=gpu).manual_seed(BQ * Sk + BK)
    nK, Sq = Sk // BK, nQ * BQ
    u = torch.rand(uB, uH, nQ, 1, nK, 1, generator=g, device=gpu)
    dense = torch.rand(uB, uH, nQ, BQ, nK, BK, generator=g, device=gpu) < 0.5
    tiles = torch.where(u < 0.3, dense, u < 0.6)
    for only, value in ((0.6, True), (0.8, False)):                       # FULL but for one entry, empty but for one
        one = (u > only) & (u < only + 0.1)
        where = torch.randint(BQ * BK, (uB, uH, nQ, 1, nK, 1), generator=g, device=gpu)
        at = torch.arange(BQ, device=gpu).view(BQ, 1, 1) * BK + torch.arange(BK, device=gpu) == where
        tiles = torch.where(one, at != value, tiles)
    del dense
    store = torch.zeros(uB, uH, Sq, pitch, dtype=torch.bool, device=gpu)
    store[..., :Sk] = tiles.reshape(uB, uH, Sq, Sk)
    got = compute_mask_kernel(store[..., :Sk].expand(2, 2, Sq, Sk), BQ, BK)
    some, every = tiles.any(5).any(3), tiles.all(5).all(3)
    ids = torch.arange(nK, device=gpu, dtype=torch.int32)
    for wanted, lens, lists in ((every, got.unmasked_lens, got.unmasked_kv_ids), (some & ~every, got.masked_lens, got.masked_kv_ids)):
        n = wanted.sum(-1, dtype=torch.int32)
        assert torch.equal(lens, n.expand(2, 2, nQ))
        in_order = torch.where(wanted, ids, nK).sort(-1).values.int()
        assert torch.equal(torch.where(ids < n[..., None], lists, nK), in_order.expand(2, 2, nQ, nK))
    if BQ * BK % 8 == 0 and got.packed_masks is not None:
        packed = got.packed_masks[:uB, :uH].reshape(uB, uH, nQ, nK, BQ, BK // 8, 1)
        bits = (packed >> torch.arange(8, dtype=torch.uint8, device=gpu)) & 1
        slots = in_order.clamp(max=nK - 1).long().view(uB, uH, nQ, nK, 1, 1).expand(uB, uH, nQ, nK, BQ, BK)
        want = tiles.transpose(3, 4).gather(3, slots)
        used = (ids < n[..., None]).view(uB, uH, nQ, nK, 1, 1)
        assert torch.equal(bits.reshape(uB, uH, nQ, nK, BQ, BK).bool() & used, want & used)
