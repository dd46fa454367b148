"""The two tilings of a backward from one launch, against a launch for each (whole numbers and bytes: equal)."""
import pytest
import torch

from sparseattention_amd import MaskTerm, block_term, causal_term, compute_backward_metadata_terms, compute_mask_terms

pytestmark = pytest.mark.gpu


# (grids of different height, so that workgroups of the larger one have no tile in the other; with and without a plane per batch element)
@pytest.mark.parametrize("B,H,Sq,Sk", [(1, 1, 128, 128), (3, 2, 256, 1152), (2, 3, 1152, 384)])
@pytest.mark.parametrize("kind", ["causal", "documents", "one row of documents", "documents and prefix"])
def test_both_tilings(gpu, B, H, Sq, Sk, kind):
    g = torch.Generator().manual_seed(Sq + Sk)
    dq = dk = None
    terms = [causal_term(offset=Sk - Sq, same_doc=kind != "causal")]
    if kind != "causal":
        n = 1 if kind == "one row of documents" else B
        dq, dk = (torch.randint(0, 5, (n, S), generator=g, dtype=torch.int32).sort(-1).values.to(gpu) for S in (Sq, Sk))
        if n == 1:
            dq, dk = dq[0], dk[0]
    if kind == "documents and prefix":
        terms += [block_term((0, 70), (0, 100)), MaskTerm(back=9, ahead=40)]
    got = compute_backward_metadata_terms(terms, B, H, Sq, Sk, dq, dk, device=gpu)
    want = (compute_mask_terms(terms, B, H, Sq, Sk, 128, 64, dq, dk, device=gpu),
            compute_mask_terms([t.transposed() for t in terms], B, H, Sk, Sq, 128, 64, dk, dq, device=gpu))
    for a, b in zip((got.by_query, got.by_key), want):
        for x, y in ((a.unmasked_lens, b.unmasked_lens), (a.masked_lens, b.masked_lens)):
            assert torch.equal(x, y) and x.stride() == y.stride()
        at = torch.arange(a.masked_kv_ids.shape[-1], device=gpu)
        full, part = at < b.unmasked_lens[..., None], at < b.masked_lens[..., None]
        assert torch.equal(a.unmasked_kv_ids[full], b.unmasked_kv_ids[full])
        assert torch.equal(a.masked_kv_ids[part], b.masked_kv_ids[part])
        assert torch.equal(a.packed_masks[part], b.packed_masks[part])
