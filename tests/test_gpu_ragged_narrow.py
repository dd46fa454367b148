"""Ragged tensors whose head dim is at most three quarters of the kernel's 128: the last quarter takes no part.  Every shape of workgroup
and chunk, head dims up to the line and past it."""
import pytest
import torch

from sparseattention_amd import select_tiling, sparse_attention_tiled
from test_gpu_ragged import inside, reference

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [72, 88, 96, 104])
@pytest.mark.parametrize("BQ,BK,dtype", [(32, 16, torch.bfloat16), (64, 32, torch.float16), (64, 128, torch.bfloat16), (128, 16, torch.float16),
                                         (128, 32, torch.bfloat16), (128, 64, torch.float16)])
def test_against_the_definition(gpu, D, BQ, BK, dtype):
    B, H, Sq, Sk = 2, 2, 165, 421
    q, k, v = (inside(B, H, S, D, dtype, 30 + i, gpu) for i, S in enumerate((Sq, Sk, Sk)))
    mask = torch.rand(B, 1, Sq, Sk, generator=torch.Generator().manual_seed(D + BK)) < 0.6
    mask[..., 128:256] = True
    mask[..., 256:320] = False
    mask[0, 0, 7] = False
    mask = mask.to(gpu).expand(B, H, Sq, Sk)
    o, lse = sparse_attention_tiled(q, k, v, select_tiling(mask, candidates=((BQ, BK),)), return_lse=True)
    want, want_lse = reference(q, k, v, mask)
    # as for the other head dims: a result's own rounding and that of P, values up to 4
    assert float((o.double() - want).abs().max()) <= (2e-2 if dtype == torch.bfloat16 else 4e-3)
    live = torch.isfinite(want_lse)
    assert torch.equal(torch.isfinite(lse), live)
    assert float((lse.double() - want_lse)[live].abs().max()) <= 6e-3 + 2 ** -9 * 6
