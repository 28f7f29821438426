"""Compression of narrow sparse blocks on the GPU (marked gpu): rows long
enough to be split whose blocks are below, at and above the width from which
they are, against the host's arrays, bit for bit."""
import pytest

import test_gpu_compress_split as split

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hs", [[1, 70], [257]])
@pytest.mark.parametrize("ws", [[1] * 130, [3] * 50, [4] * 50, [3, 5] * 30, [5] * 3 + [1] * 40, [2] * 10])
def test_narrow_blocks_match_host(hs, ws):
    for keep in (1, 3):
        split.test_shares_match_host(hs, ws, keep)
