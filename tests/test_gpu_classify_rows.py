"""Classification, lists and packed tiles in one launch: rows of every length a wave instruction shares out, one row to many, the
edges of the rule that chooses it, masks that differ per batch and head, and the masks it does not take."""
import pytest
import torch

from sparseattention_amd import compute_mask_kernel, compute_mask_slow

pytestmark = pytest.mark.gpu


def _unpack(packed, BQ, BK):
    bits = (packed.cpu()[..., None] >> torch.arange(8, dtype=torch.uint8)) & 1
    return bits.reshape(*packed.shape[:-1], BQ, BK).bool()


def _check(mask, gpu_mask, BQ, BK):
    B, H, Sq, Sk = mask.shape
    got, want = compute_mask_kernel(gpu_mask, BQ, BK), compute_mask_slow(mask, BQ, BK)
    assert torch.equal(got.unmasked_lens.cpu(), want.unmasked_lens) and torch.equal(got.masked_lens.cpu(), want.masked_lens)
    tiles = mask.reshape(B, H, Sq // BQ, BQ, Sk // BK, BK).transpose(3, 4)
    bits = _unpack(got.packed_masks, BQ, BK)
    gf, wf, gp, wp = (t.cpu() for t in (got.unmasked_kv_ids, want.unmasked_kv_ids, got.masked_kv_ids, want.masked_kv_ids))
    for b in range(B):
        for h in range(H):
            for i in range(Sq // BQ):
                nf, np_ = int(want.unmasked_lens[b, h, i]), int(want.masked_lens[b, h, i])
                assert torch.equal(gf[b, h, i, :nf], wf[b, h, i, :nf]) and torch.equal(gp[b, h, i, :np_], wp[b, h, i, :np_])
                assert torch.equal(bits[b, h, i, :np_], tiles[b, h, i][wp[b, h, i, :np_].long()])


# (B, H, distinct heads, Sq, Sk, BQ, BK)
CASES = [(1, 1, 1, 1, 16, 1, 16), (2, 3, 1, 2, 32, 1, 16), (1, 2, 2, 3, 96, 3, 32), (4, 2, 1, 1, 2048, 1, 64), (1, 1, 1, 2, 32768, 2, 16),
         (2, 1, 1, 5, 1040, 5, 16), (1, 2, 2, 64, 512, 32, 512), (1, 1, 1, 128, 1024, 128, 1024), (2, 2, 2, 384, 384, 128, 64),
         (1, 3, 1, 256, 1152, 128, 128), (1, 1, 1, 128, 1088, 128, 64),     # the last past 128 KiB with one workgroup
         (1, 1, 1, 1, 32784, 1, 16)]                                         # more tiles than LDS holds


@pytest.mark.parametrize("B,H,uH,Sq,Sk,BQ,BK", CASES)
def test_lists_and_bits(gpu, B, H, uH, Sq, Sk, BQ, BK):
    g = torch.Generator().manual_seed(Sq * Sk + BK)
    u = torch.rand(B, uH, Sq // BQ, Sk // BK, generator=g).repeat_interleave(BQ, 2).repeat_interleave(BK, 3)
    mask = torch.where(u < 0.4, torch.rand(B, uH, Sq, Sk, generator=g) < 0.5, u < 0.7)
    _check(mask.expand(B, H, Sq, Sk), mask.to(gpu).expand(B, H, Sq, Sk), BQ, BK)


def test_rows_off_their_alignment(gpu):
    wide = torch.rand(1, 1, 64, 528, generator=torch.Generator().manual_seed(0)) < 0.5
    for first in (1, 8, 16):
        part = wide[..., first: first + 256]
        _check(part, wide.to(gpu)[..., first: first + 256], 32, 32)
