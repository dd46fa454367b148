"""Arguments of sa_mask_classify_terms_pair, refused on the host before any launch (no GPU needed)."""
import ctypes

from sparseattention_amd import _native

FAKE = 0x1000  # never dereferenced
S3 = _native.strides((0, 0, 1))
I4 = _native.strides((0, 0, 2, 1))


def test_a_pair_of_masks_by_terms_is_checked_call_by_call():
    class Call(ctypes.Structure):
        _fields_ = [("terms", ctypes.c_void_p), ("n_terms", ctypes.c_int), ("doc_q", ctypes.c_void_p), ("dqs", ctypes.c_void_p),
                    ("doc_k", ctypes.c_void_p), ("dks", ctypes.c_void_p)] + \
                   [(n, ctypes.c_int) for n in ("B", "H", "Sq", "Sk", "BQ", "BK")] + \
                   [(n, ctypes.c_void_p) for n in ("fi", "fis", "fl", "fls", "pi", "pis", "pl", "pls", "packed", "pks", "ws")] + \
                   [("ws_bytes", ctypes.c_size_t)]

    lib = _native.load()
    causal = (ctypes.c_int32 * 8)(2, 0, 0, 1, 0, 0, 0, 0)
    p = lambda a: ctypes.cast(a, ctypes.c_void_p)  # noqa: E731
    good = dict(terms=p(causal), n_terms=1, B=1, H=1, Sq=128, Sk=128, BQ=128, BK=64, fi=FAKE, fis=p(I4), fl=FAKE, fls=p(S3), pi=FAKE,
                pis=p(I4), pl=FAKE, pls=p(S3), ws=FAKE, ws_bytes=1 << 20)
    for bad, rc in ((dict(n_terms=9), _native.SA_ERR_INVALID_ARGUMENT), (dict(fi=None), _native.SA_ERR_INVALID_ARGUMENT),
                    (dict(BK=24), _native.SA_ERR_INVALID_ARGUMENT), (dict(ws_bytes=0), _native.SA_ERR_WORKSPACE)):
        for calls in ((dict(good, **bad), good), (good, dict(good, **bad))):
            a, b = (Call(**c) for c in calls)
            assert lib.sa_mask_classify_terms_pair(ctypes.byref(a), ctypes.byref(b), None) == rc, bad
    assert lib.sa_mask_classify_terms_pair(None, ctypes.byref(Call(**good)), None) == _native.SA_ERR_INVALID_ARGUMENT
