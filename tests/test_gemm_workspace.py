"""The prefill GEMM's workspace query (no GPU needed): a session allocates one
workspace for its 512-token chunk and its largest need over the layers'
matrices, and every shorter prompt runs in it."""
import pytest

import xqbind as xb


def matrices(hidden, inter, nq, nkv, lk, lv):
    """(rows, cols) of a hybrid model's projections (head size 128, gated q_proj)."""
    return [(2 * nq * 128 + 2 * nkv * 128, hidden), (hidden, nq * 128), (2 * lk * 128 + 2 * lv * 128 + 2 * lv, hidden),
            (hidden, lv * 128), (2 * inter, hidden), (hidden, inter)]


@pytest.mark.parametrize("shape", [(4096, 12288, 32, 8, 16, 32), (2048, 6144, 16, 4, 8, 16), (4096, 1024, 16, 4, 16, 32)])
def test_a_chunk_workspace_serves_every_shorter_prompt(shape):
    """354 tokens of the 9B shape once needed more than 512 did (two K splits of
    the input projection), and xq_prefill refused the prompt."""
    need = xb.hip().xqhip_gemm_workspace_bytes
    mats = matrices(*shape)
    have = max(need(512, c, r) for r, c in mats)
    short = [(n, r, c) for n in range(1, 513) for r, c in mats if need(n, c, r) > have]
    assert not short, short[:5]


def test_workspace_of_the_largest_rows_serves_fewer_rows():
    need = xb.hip().xqhip_gemm_workspace_bytes
    assert all(need(512, 4096, r) <= need(512, 4096, 24576) for r in range(64, 24576, 64))
