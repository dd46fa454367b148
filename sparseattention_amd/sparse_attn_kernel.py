"""Block-sparse attention forward (replaces the reference's ``sparseattention/sparse_attn_kernel.py``).

The steps of a call - checks, outputs, strides, launch - are native (csrc/host_ops.cpp); here is what a caller sees and
what sizes without a kernel need around it."""
from __future__ import annotations

import torch

from . import _native
from .mask_utils import MaskMetadata, Tiling, compute_mask_kernel, compute_mask_terms_backward, validation_key

_DTYPES = {torch.bfloat16: _native.SA_DTYPE_BF16, torch.float16: _native.SA_DTYPE_FP16}


def _pad_mask(mask: torch.Tensor, q_multiple: int, k_multiple: int) -> torch.Tensor:
    """``mask`` [B,H,Sq,Sk] with all-False rows and columns added up to multiples of the two numbers; only the
    distinct planes of a broadcast view are copied."""
    B, H, Sq, Sk = mask.shape
    if Sq % q_multiple == 0 and Sk % k_multiple == 0:
        return mask
    distinct = mask[: 1 if mask.stride(0) == 0 else B, : 1 if mask.stride(1) == 0 else H]
    padded = torch.nn.functional.pad(distinct, (0, -Sk % k_multiple, 0, -Sq % q_multiple), value=False)
    return padded.expand(B, H, *padded.shape[2:])


def _same_device(ref: torch.Tensor, **tensors) -> None:
    """Every tensor whose data pointer goes to a kernel must live where ``ref`` lives: a host pointer (or one of
    another GPU) in any slot would be a memory fault on the device, where the reference raises a Python error."""
    for name, t in tensors.items():
        if t is not None and t.device != ref.device:
            raise ValueError(f"{name} is on {t.device}, expected {ref.device} (every tensor argument must be on q's device)")


def validate_metadata(md: MaskMetadata, Sk: int, BLOCK_K: int) -> None:
    """Raise ValueError unless the lists can address K and V: ``0 <= lens``, ``unmasked_lens + masked_lens <= Sk/BLOCK_K``
    and ``0 <= ids[..., :len] < Sk/BLOCK_K`` (the reference guards its loads with ``kv_offset < SEQLEN_K``,
    sparse_attn_kernel.py:35,39,60).  Plain torch on the tensors' own device; reads two flags back, so it synchronises.
    The wrappers run it once per metadata object that did not come from this package's own preprocessing; the kernels
    additionally clamp counts and skip indices out of range, so unchecked metadata cannot fault either."""
    nK = Sk // BLOCK_K
    bad = []
    fl, pl = md.unmasked_lens, md.masked_lens
    if bool(((fl < 0) | (pl < 0) | (fl.to(torch.int64) + pl.to(torch.int64) > nK)).any()):
        bad.append(f"counts outside [0, {nK}] or unmasked_lens + masked_lens > {nK}")
    for name, ids, lens in (("unmasked_kv_ids", md.unmasked_kv_ids, fl), ("masked_kv_ids", md.masked_kv_ids, pl)):
        if ids.shape[-1] != nK:
            bad.append(f"{name} has {ids.shape[-1]} slots per Q tile, expected {nK}")
            continue
        live = torch.arange(nK, device=ids.device) < lens[..., None]
        if bool((live & ((ids < 0) | (ids >= nK))).any()):
            bad.append(f"{name}[..., :len] holds tile indices outside [0, {nK})")
    if bad:
        raise ValueError("mask_metadata does not fit Sk=%d, BLOCK_K=%d: %s" % (Sk, BLOCK_K, "; ".join(bad)))


def _checked_metadata(md: MaskMetadata, Sk: int, BLOCK_K: int) -> None:
    """validate_metadata once per (object, tiling, state of its list tensors); metadata made by compute_mask_kernel /
    compute_mask_terms is trusted (marked there), so the usual call path never synchronises.  Lists edited in place
    afterwards, or an object whose tensors were exchanged (dataclasses.replace, copy), are checked again."""
    key = validation_key(md, Sk, BLOCK_K)
    if getattr(md, "_validated_for", None) == key:
        return
    validate_metadata(md, Sk, BLOCK_K)
    try:
        md._validated_for = key
    except AttributeError:  # the reference's own dataclass, say: a carrier without the field is checked every time
        pass


_KERNEL_BLOCK_Q = (128, 64, 32, 256)  # in order of preference when the caller's size is not one of them


def kernel_tiles(Sq: int, Sk: int, D: int, BLOCK_Q: int, BLOCK_K: int):
    """The tile sizes the forward runs a request for ``BLOCK_Q`` x ``BLOCK_K`` tiles with: the same pair when the
    kernels tile by it (BLOCK_Q 32/64/128/256 — 64/128 at head dim 256 —, BLOCK_K a power of two >= 16), else the
    nearest pair they have that divides Sq and Sk, or None when there is none.  The reference takes any sizes its
    compiler accepts (sparse_attn_kernel.py:149-185); the result does not depend on them."""
    BLOCK_Q, BLOCK_K = int(BLOCK_Q), int(BLOCK_K)
    ok_k = BLOCK_K >= 16 and BLOCK_K & (BLOCK_K - 1) == 0 and Sk % BLOCK_K == 0
    if Sq < 32:  # the few-rows kernels: one Q tile of all rows, KV tiles of 16 keys or more, head dims up to 128
        if D > 128:
            return None
        if ok_k:
            return Sq, BLOCK_K
        return next(((Sq, bk) for bk in (32, 64) if Sk % bk == 0), None)
    ok_q = [b for b in _KERNEL_BLOCK_Q if Sq % b == 0 and (D <= 128 or b in (64, 128))]  # (D above 128 runs as 256)
    if not ok_q:
        return None
    bq = BLOCK_Q if BLOCK_Q in ok_q else ok_q[0]
    if ok_k:
        return bq, BLOCK_K
    return next(((bq, bk) for bk in (32, 64, 16) if Sk % bk == 0), None)


def sparse_attention(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, mask: torch.Tensor | None, BLOCK_Q, BLOCK_K,
                     mask_metadata: MaskMetadata | None = None, *, return_lse: bool = False, kernel: str | None = None):
    """softmax(q kᵀ / sqrt(D) + (mask ? 0 : -inf)) v, skipping KV tiles the mask empties.

    Signature and meaning follow sparse_attn_kernel.py:149-185: ``q`` [B,H,Sq,D], ``k``/``v``
    [B,H,Sk,D] (bf16, fp16, or float32 on kernels that compute in float32 throughout; on a
    ROCm GPU), ``mask`` bool broadcastable to [B,H,Sq,Sk] with
    True = attend, tile sizes ``BLOCK_Q`` x ``BLOCK_K``, and optionally the metadata from
    :func:`compute_mask_kernel` so that preprocessing is paid once for many calls.
    Returns ``o`` with q's shape, dtype and strides; with ``return_lse=True`` (not in the reference, which drops
    the row statistics after the division at sparse_attn_kernel.py:144) the pair ``(o, lse)`` where ``lse``
    [B,H,Sq] float32 is the log of the row's softmax denominator, -inf for rows that attend to nothing.
    ``mask`` may be None when ``mask_metadata`` carries ``packed_masks`` (the kernels then read no mask tensor), which
    is how masks given by a formula run (:func:`compute_mask_terms`).
    ``kernel`` (not in the reference, whose one kernel Triton autotunes at the first call, sparse_attn_kernel.py:66-72):
    "default" = two workgroups per compute unit, 64 keys per step (the list of a Q tile shared by several workgroups
    where there are too few Q tiles to fill the device); "short" = the form for masks that leave a Q tile
    few KV tiles (three workgroups per compute unit, 32 keys per step; bf16/fp16, D = 128, BLOCK_Q = 128, packed
    PARTIAL tiles, ``mask_metadata.list_stats`` with no list above 256 entries); None / "auto" = "short" when the
    metadata carries ``list_stats`` (``compute_mask_kernel(..., list_stats=True)``) that say the lists are short,
    else "default".  "rotated" = the default kernel with the FULL entries of Q tile qt walked from a start that depends
    on qt (for sliding windows; "auto" takes it when ``mask_metadata.list_rotation`` says so).  All agree within rounding.
    """
    BLOCK_Q, BLOCK_K = int(BLOCK_Q), int(BLOCK_K)
    kernel = "auto" if kernel is None else kernel
    out = _native.host().forward(q, k, v, mask, BLOCK_Q, BLOCK_K, mask_metadata, return_lse, kernel)
    if out is not None:
        return out
    # Sizes the kernels do not tile by (everything else about the arguments has been checked).
    B, H, Sq, D = q.shape
    Sk = k.shape[-2]
    if mask is not None:
        mask = mask.expand(B, H, Sq, Sk)
    tiles = kernel_tiles(Sq, Sk, D, BLOCK_Q, BLOCK_K)
    row_multiple = 32 if D <= 128 else 64  # the smallest Q tile the kernels have
    if tiles is None and mask is not None and Sq % row_multiple and Sq % BLOCK_Q == 0 and Sk % BLOCK_K == 0:
        # A row count that no Q tile of the kernels divides (48, 80, ...; fewer than 32 rows at a head dim the few-rows
        # kernels do not have): zero rows are added to q and all-False rows to the mask, and their (zero) output rows
        # dropped again.  Nothing is kept between calls on this path.
        pad = -Sq % row_multiple
        padded_tiles = kernel_tiles(Sq + pad, Sk, D, BLOCK_Q, BLOCK_K)
        if padded_tiles is not None:
            out = sparse_attention(torch.nn.functional.pad(q, (0, 0, 0, pad)), k, v, _pad_mask(mask, row_multiple, 1),
                                   *padded_tiles, return_lse=return_lse)
            return (out[0][:, :, :Sq].contiguous(), out[1][:, :, :Sq].contiguous()) if return_lse \
                else out[:, :, :Sq].contiguous()
    # The sizes only say how the mask is cut up, not what is computed, so the mask is classified again at sizes the
    # kernels have; the lists are kept on the caller's metadata.
    # what the reference asserts (mask_utils.py:89-90)
    assert Sq % BLOCK_Q == 0 and Sk % BLOCK_K == 0, \
        f"Sq={Sq} / Sk={Sk} must be multiples of BLOCK_Q={BLOCK_Q} / BLOCK_K={BLOCK_K}"
    if tiles is None or mask is None:
        raise ValueError(f"sparse_attention: no kernel tiles for BLOCK_Q={BLOCK_Q}, BLOCK_K={BLOCK_K} at Sq={Sq}, "
                         f"Sk={Sk}, D={D}" + ("" if tiles is None else " without a mask tensor to classify again"))
    again = getattr(mask_metadata, "_retiled", None)
    if again is None or again[0] != (tiles, mask.data_ptr(), tuple(mask.stride()), mask._version):
        again = ((tiles, mask.data_ptr(), tuple(mask.stride()), mask._version),
                 compute_mask_kernel(mask, *tiles, pack_partial=None if Sq >= 32 else False))
        if mask_metadata is not None:
            mask_metadata._retiled = again
    return _native.host().forward(q, k, v, mask, *tiles, again[1], return_lse, kernel)


def sparse_attention_tiled(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, tiling: Tiling, *, return_lse: bool = False):
    """:func:`sparse_attention` on the tile grid chosen by :func:`sparseattention_amd.select_tiling`: q, k, v get
    ``q_offset`` / ``k_offset`` zero rows in front (and zero rows at the end up to whole tiles), which the padded mask
    lets nothing attend to or from, and the rows of the result that belong to the caller's queries are returned.  With
    both offsets 0 and sizes that are whole tiles this is sparse_attention itself.  In bf16 and fp16 with packed tiles,
    BLOCK_Q up to 128 and head dims that are multiples of 8 up to 128 the kernel leaves the rows out that do not exist;
    otherwise, and for k and v of fewer keys than the mask, it costs a copy of q, k, v."""
    Sq, Sk = q.shape[-2], k.shape[-2]
    Pq, Pk = tiling.padded_mask.shape[-2:]
    qo, ko = tiling.q_offset, tiling.k_offset
    if not (qo + Sq <= Pq and ko + Sk <= Pk):
        raise ValueError(f"tiling for a mask of {Pq - qo}x{Pk - ko} or smaller, got Sq={Sq}, Sk={Sk}")
    # (the kernel reads no key that the tensors do not have, so it needs a mask that has none there either; with fewer keys
    # than the mask the missing ones are zeros, as below)
    if (qo, Pq, ko, Pk) != (0, Sq, 0, Sk) and Sk == tiling.Sk:
        out = _native.host().forward_tiled(q, k, v, tiling.BLOCK_Q, tiling.BLOCK_K, qo, ko, Pq, Pk, tiling.metadata, return_lse)
        if out is not None:
            return out
    pad = torch.nn.functional.pad
    qp = q if (qo, Pq) == (0, Sq) else pad(q, (0, 0, qo, Pq - qo - Sq))
    kp = k if (ko, Pk) == (0, Sk) else pad(k, (0, 0, ko, Pk - ko - Sk))
    vp = v if (ko, Pk) == (0, Sk) else pad(v, (0, 0, ko, Pk - ko - Sk))
    out = sparse_attention(qp, kp, vp, tiling.padded_mask, tiling.BLOCK_Q, tiling.BLOCK_K, tiling.metadata,
                           return_lse=return_lse)
    if (qo, Pq) == (0, Sq):
        return out
    if return_lse:
        return out[0][:, :, qo:qo + Sq].contiguous(), out[1][:, :, qo:qo + Sq].contiguous()
    return out[:, :, qo:qo + Sq].contiguous()


def sparse_attention_decode(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, mask: torch.Tensor | None, BLOCK_K,
                            mask_metadata: MaskMetadata | None = None, num_splits: int = 0, *,
                            return_lse: bool = False):
    """:func:`sparse_attention` for Sq <= 32 query rows (decode, speculative or chunked-prefill tails), BLOCK_Q = Sq.

    The reference lists decode kernels as future work (README.md:65); the result is defined by its forward
    (sparse_attn_kernel.py:149-185) called with ``BLOCK_Q = Sq``.  Every (b, h) has one Q tile, so its list of KV
    tiles is cut into ``num_splits`` ranges (0: chosen from the shape and the device) that run in parallel and are
    merged afterwards.  ``mask_metadata``: from ``compute_mask_kernel(mask, Sq, BLOCK_K)``; when it carries
    ``packed_masks`` (the default there) the kernels read those bits and ``mask`` may be None (at BLOCK_K = 16 with an odd
    number of query rows the bool mask is read instead).  ``return_lse``: as in :func:`sparse_attention`.
    """
    return _native.host().decode(q, k, v, mask, int(BLOCK_K), mask_metadata, int(num_splits), return_lse)


class BackwardMetadata:
    """Tile lists the backward pass walks: of the mask per 128 queries (KV tiles of 64 keys) and of the transposed
    mask per 128 keys (tiles of 64 queries).  Built once per mask by :func:`compute_backward_metadata`.

    When both lists carry ``packed_masks`` (the PARTIAL tiles at one bit per entry), the backward reads those and
    neither the mask nor its transposed copy, so both bool tensors can be released after this preprocessing.

    Lists put together by the caller need not agree with each other: dQ follows ``by_query`` alone, dK and dV ``by_key``.
    Lists of one mask from the functions below are known to agree (``_agreeing``: their tensors with the addresses and
    in-place versions they had) until they are edited or replaced, and then dQ may be made from the dS of the pass over the keys."""

    def __init__(self, by_query: MaskMetadata, by_key: MaskMetadata, transposed_mask: torch.Tensor | None = None):
        self.by_query = by_query
        self.by_key = by_key
        #: bool [B,H,Sk,Sq], the mask transposed as a tensor of its own (distinct planes, expanded), or None
        self.transposed_mask = transposed_mask
        self._agreeing = None

    def __getstate__(self):
        return {**self.__dict__, "_agreeing": None}  # (addresses and versions are this process's own)


def _of_one_mask(bmd: BackwardMetadata) -> BackwardMetadata:
    """Notes that both lists of ``bmd``, with packed tiles, were made from one mask."""
    bmd._agreeing = _native.host().of_one_mask(bmd.by_query, bmd.by_key)
    return bmd


def compute_backward_metadata(mask: torch.Tensor, pack_partial: bool = True) -> BackwardMetadata:
    """``mask``: bool [B,H,Sq,Sk] (broadcast views are fine).  Sq and Sk that are not multiples of 128 are taken up to
    the next one with rows and columns that attend to nothing, as :func:`sparse_attention_backward` does with its
    tensors.

    ``pack_partial``: bit-pack the PARTIAL tiles of both tilings (2 * Sq*Sk/8 bytes per distinct plane at most) and
    drop the transposed copy; otherwise keep that copy (Sq*Sk bytes per distinct plane) for the key passes."""
    if mask.dim() != 4:
        raise ValueError("mask must be [B,H,Sq,Sk] (broadcast views are fine)")
    mask = _pad_mask(mask, 128, 128)
    # the transposed mask as a tensor of its own, distinct planes only, so that its classification reads rows
    B, H = mask.shape[:2]
    distinct = mask[: 1 if mask.stride(0) == 0 else B, : 1 if mask.stride(1) == 0 else H]
    transposed = distinct.transpose(-1, -2).contiguous().expand(B, H, mask.shape[3], mask.shape[2])
    bmd = BackwardMetadata(compute_mask_kernel(mask, 128, 64, pack_partial=pack_partial),
                           compute_mask_kernel(transposed, 128, 64, pack_partial=pack_partial),
                           None if pack_partial else transposed)
    return _of_one_mask(bmd) if pack_partial else bmd


def compute_backward_metadata_terms(terms, B: int, H: int, Sq: int, Sk: int, doc_q=None, doc_k=None,
                                    device=None) -> BackwardMetadata:
    """:func:`compute_backward_metadata` for a mask given by terms (:func:`compute_mask_terms`): both tilings with
    their packed PARTIAL tiles, the key-major one from the transposed terms, so that
    ``sparse_attention_backward(..., mask=None, bwd_metadata=...)`` runs without any mask tensor."""
    return _of_one_mask(BackwardMetadata(*compute_mask_terms_backward(terms, B, H, Sq, Sk, doc_q, doc_k, device), None))


def sparse_attention_backward(do: torch.Tensor, q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, o: torch.Tensor,
                              lse: torch.Tensor, mask: torch.Tensor | None,
                              bwd_metadata: BackwardMetadata | None = None):
    """Gradients (dq, dk, dv) of :func:`sparse_attention` for the upstream gradient ``do``.

    The reference has no backward pass (README.md:65 lists it as future work); this differentiates its forward
    (sparse_attn_kernel.py:149-185).  ``o`` and ``lse`` come from ``sparse_attention(..., return_lse=True)`` with the
    same inputs.  bf16/fp16; the kernels have D = 64 and 128 and tile by 128 rows, other head dims up to 128 and
    other Sq, Sk are padded here (zero columns; rows that attend to nothing).  The backward tiles the mask its own way
    (128 x 64 both ways), whatever BLOCK_Q / BLOCK_K the forward used.  ``mask`` may be None when ``bwd_metadata``
    carries the packed PARTIAL tiles of both tilings.
    """
    grads = _native.host().backward(do, q, k, v, o, lse, mask, bwd_metadata)
    if grads is not None:
        return grads
    # The kernels tile by 128 rows both ways: zero rows (lse = -inf: rows that attended to nothing) and mask rows and
    # columns that attend to nothing are added, and the gradients of the added rows dropped.
    B, H, Sq, _ = q.shape
    Sk = k.shape[-2]
    rows = lambda t, n: torch.nn.functional.pad(t, (0, 0, 0, -n % 128))  # noqa: E731
    dq, dk, dv = sparse_attention_backward(
        rows(do, Sq), rows(q, Sq), rows(k, Sk), rows(v, Sk), rows(o, Sq),
        torch.nn.functional.pad(lse, (0, -Sq % 128), value=float("-inf")),
        None if mask is None else _pad_mask(mask.expand(B, H, Sq, Sk), 128, 128), bwd_metadata)
    return dq[:, :, :Sq].contiguous(), dk[:, :, :Sk].contiguous(), dv[:, :, :Sk].contiguous()


class _SparseAttentionFunction(torch.autograd.Function):
    @staticmethod
    def forward(ctx, q, k, v, mask, BLOCK_Q, BLOCK_K, mask_metadata, bwd_metadata):
        o, lse = sparse_attention(q, k, v, mask, BLOCK_Q, BLOCK_K, mask_metadata, return_lse=True)
        ctx.save_for_backward(q, k, v, o, lse, mask)
        ctx.bwd_metadata = bwd_metadata
        return o

    @staticmethod
    def backward(ctx, do):
        q, k, v, o, lse, mask = ctx.saved_tensors
        dq, dk, dv = sparse_attention_backward(do, q, k, v, o, lse, mask, ctx.bwd_metadata)
        return dq, dk, dv, None, None, None, None, None


def sparse_attention_trainable(q, k, v, mask, BLOCK_Q, BLOCK_K, mask_metadata: MaskMetadata | None = None,
                               bwd_metadata: BackwardMetadata | None = None) -> torch.Tensor:
    """:func:`sparse_attention` as a differentiable torch function (gradients for q, k, v through
    :func:`sparse_attention_backward`)."""
    out = _native.host().trainable(q, k, v, mask, int(BLOCK_Q), int(BLOCK_K), mask_metadata, bwd_metadata)
    if out is None:  # sizes that the wrappers pad or tile anew, and under torch.jit.trace
        out = _SparseAttentionFunction.apply(q, k, v, mask, BLOCK_Q, BLOCK_K, mask_metadata, bwd_metadata)
    return out


def merge_attention_parts(o_parts: torch.Tensor, lse_parts: torch.Tensor, return_lse: bool = False):
    """Merge attention results computed over disjoint key ranges of the same queries.

    ``o_parts`` [n,B,H,Sq,D] (bf16/fp16) and ``lse_parts`` [n,B,H,Sq] (float32) as returned, per key range, by
    ``sparse_attention(..., return_lse=True)``: ``o = Σ_i exp(lse_i − lse) o_i`` with ``lse = logsumexp_i lse_i``.
    This is the exchange a key-axis sharding of the forward ends with (no counterpart in the reference).
    """
    if o_parts.dim() != 5 or lse_parts.shape != o_parts.shape[:4] or lse_parts.dtype != torch.float32:
        raise ValueError("o_parts must be [n,B,H,Sq,D] and lse_parts float32 [n,B,H,Sq]")
    if o_parts.dtype not in _DTYPES or not o_parts.is_cuda:
        raise TypeError("o_parts must be a bfloat16 or float16 tensor on a ROCm GPU")
    _same_device(o_parts, lse_parts=lse_parts)
    n, B, H, Sq, D = o_parts.shape
    if o_parts.stride(-1) != 1 or o_parts.data_ptr() % 16 or any(s % 8 for s in o_parts.stride()[:-1]):
        o_parts = o_parts.contiguous()
    o = torch.empty(B, H, Sq, D, dtype=o_parts.dtype, device=o_parts.device)
    lse = torch.empty(B, H, Sq, dtype=torch.float32, device=o_parts.device) if return_lse else None
    S = _native.strides
    with torch.cuda.device(o_parts.device):
        rc = _native.load().sa_merge_attention_parts(
            o_parts.data_ptr(), S(o_parts.stride()), lse_parts.data_ptr(), S(lse_parts.stride()),
            o.data_ptr(), S(o.stride()), lse.data_ptr() if return_lse else None, S(lse.stride()) if return_lse else None,
            n, B, H, Sq, D, _DTYPES[o_parts.dtype], torch.cuda.current_stream(o_parts.device).cuda_stream)
    _native.check(rc)
    return (o, lse) if return_lse else o


def sparse_attention_kv_split(q, k, v, mask, BLOCK_Q, BLOCK_K, num_splits: int, return_lse: bool = False):
    """:func:`sparse_attention` with the key axis cut into ``num_splits`` equal ranges, each run as a forward of
    its own (own tile lists) and merged by :func:`merge_attention_parts`: what one device per range would do.
    Useful on one device when there are too few Q tiles to fill it (a few hundred query rows against long keys)."""
    B, H, Sq, D = q.shape
    Sk = k.shape[-2]
    if Sk % (num_splits * BLOCK_K):
        raise ValueError(f"Sk ({Sk}) must be a multiple of num_splits * BLOCK_K ({num_splits} * {BLOCK_K})")
    mask = mask.expand(B, H, Sq, Sk)
    step = Sk // num_splits
    o_parts = torch.empty(num_splits, B, H, Sq, D, dtype=q.dtype, device=q.device)
    lse_parts = torch.empty(num_splits, B, H, Sq, dtype=torch.float32, device=q.device)
    for i in range(num_splits):
        sl = slice(i * step, (i + 1) * step)
        o_parts[i], lse_parts[i] = sparse_attention(q, k[:, :, sl], v[:, :, sl], mask[..., sl], BLOCK_Q, BLOCK_K,
                                                    return_lse=True)
    return merge_attention_parts(o_parts, lse_parts, return_lse)
