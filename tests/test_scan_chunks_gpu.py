"""The chunked linear-attention recurrence (two kinds of waves per block, conv
output by head) at the edges of its 64-token chunks and of its 16-token and
16-column tiles, with value heads whose rows and records are aligned to 4 bytes
only, against consecutive decode steps (custom_model.cpp:1074-1096)."""
import pytest

from test_prefill_gpu import test_linear_scan_matches_consecutive_steps as check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,T", [((16, 32, 128, 128, 4), 1), ((2, 2, 128, 128, 4), 63), ((2, 6, 128, 128, 4), 65),
                                     ((1, 1, 128, 128, 4), 128), ((1, 3, 128, 17, 3), 67), ((2, 4, 128, 1, 3), 16),
                                     ((1, 2, 128, 130, 4), 33)])
def test_chunk_edges(shape, T):
    check(shape, T, T & 3, True)
