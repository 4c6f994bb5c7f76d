"""Which steps of the delta rule run in chunks: where both forms were measured, the faster one (16 and 64 heads of 128, 64 heads
of 64), and always where token by token the step would be cut into pieces."""
import pytest

from mxserve.ops import seqmix


@pytest.mark.parametrize("heads,dk,dv,chunks,singles,faster", [
    (16, 128, 128, [70], 0, False), (16, 128, 128, [96], 0, True), (16, 128, 128, [4096], 0, True), (16, 128, 128, [32] * 4, 0, False),
    (16, 128, 128, [160] * 16, 0, True), (16, 128, 128, [128], 32, False), (16, 128, 128, [257], 32, True), (16, 128, 128, [512], 64, True),
    (64, 128, 128, [70], 0, False), (64, 128, 128, [128], 8, False), (64, 128, 128, [300], 32, False), (64, 128, 128, [400], 32, False),
    (64, 128, 128, [600], 32, True), (64, 128, 128, [160] * 16, 0, True), (64, 128, 128, [512], 64, False), (64, 64, 64, [300], 64, False),
    (64, 64, 64, [512], 64, True), (64, 64, 64, [160] * 16, 0, False), (16, 128, 64, [160] * 16, 0, False), (4, 64, 64, [300], 64, True),
    (32, 64, 64, [257], 32, True)])
def test_the_faster_form(heads, dk, dv, chunks, singles, faster):
    S, T = len(chunks) + singles, sum(chunks) + singles
    assert seqmix.delta_in_chunks(S, T, max(chunks), heads, dk, dv) == faster


def test_pieces_mean_chunks():
    for T in range(128, 5000, 129):
        if seqmix._scan_pieces(1, T, T, 2 * 256 * 128, 2, 1024)[1] >= seqmix.DELTA_MIN_PIECES:
            assert seqmix.delta_in_chunks(1, T, T, 2, 128, 128)
