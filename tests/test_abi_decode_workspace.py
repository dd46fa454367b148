"""Sizes of the decode's workspace: room for the counters only where the launch that makes the parts merges them (no GPU needed)."""
import pytest

from sparseattention_amd import _native


@pytest.mark.parametrize("D,Sq,n,merges", [(128, 1, 2, True), (128, 16, 8, True), (64, 4, 8, True), (64, 16, 2, True),
                                           (128, 1, 1, False), (128, 1, 9, False), (128, 1, 16, False), (128, 17, 2, False), (64, 5, 7, False),
                                           (64, 16, 3, False), (128, 32, 4, False), (128, 1, 128, False), (128, 32, 1 << 27, False)])
def test_room_for_counters(D, Sq, n, merges):
    lib, B, H = _native.load(), 3, 5
    least = lib.sa_decode_workspace_bytes(B, H, Sq, D, n)
    assert least == (B * H * n * Sq * (D + 2) * 4 if n > 1 else 0)
    assert lib.sa_decode_workspace_bytes_ex(B, H, Sq, D, n) == least + (8 * B * H if merges else 0)
