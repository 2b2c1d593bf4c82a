"""Workspace sizes and the plans behind them, asked of the built library on the host (no GPU
needed)."""

import pytest

from nanospec_amd import _lib

ROW_PART = 32   # bytes of a row's partial statistics


@pytest.fixture(scope="module")
def lib():
    return _lib.load()


@pytest.mark.parametrize("v", [8, 264, 8192, 65536, 65792, 131336, 248320, 1 << 21, 1 << 24])
def test_few_rows_have_at_most_256_vocab_splits(lib, v):
    """A row merge over half vocab tiles forms each split's state in one of 256 threads.  The teacher's
    workspace is N x S partials, then two per vocab tile and row."""
    up = lambda x: (x + 255) // 256 * 256
    for n in (1, 7, 8, 64):
        tiles = up((v + 255) // 256 * 2 * n * ROW_PART)
        parts = lib.ns_workspace_bytes(_lib.NS_WS_TEACHER_LOGITS, n, v, 0) - tiles
        assert 0 < parts <= up(n * 256 * ROW_PART)
