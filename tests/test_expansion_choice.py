"""Which chunks of a latent attention expand their keys and values: the faster form where both were measured."""
import pytest

from mxserve.models import mixers


@pytest.mark.parametrize("heads,chunks,window,expands", [
    (16, [(0, 1024)], 0, True), (16, [(0, 256)], 0, False), (16, [(2048, 512)], 0, True), (16, [(2048, 64)], 0, False),
    (64, [(2048, 128)], 0, True), (64, [(2048, 64)], 0, False), (16, [(0, 4096)], 256, True), (16, [(0, 64)] * 8, 0, False),
    (4, [(8192, 256)], 0, False), (8, [(8192, 256)], 0, True), (16, [(8192, 256)], 0, True), (4, [(8192, 512)], 0, True),
    (4, [(16384, 256)], 0, False), (8, [(16384, 256)], 0, True), (4, [(16384, 1024)], 0, True), (16, [(16384, 512)], 1024, True)])
def test_the_faster_form(heads, chunks, window, expands):
    rows = mixers.expanded_rows(chunks, window, heads)
    assert (rows > 0) == expands
    if expands:  # from the page of the first query's oldest key
        assert rows == sum(p + n - (max(p - window + 1, 0) // 16 * 16 if window else 0) for p, n in chunks)
