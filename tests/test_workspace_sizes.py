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


@pytest.mark.parametrize("v,d", [(4096, 256), (4096, 2048), (32000, 1024), (65536, 256), (248320, 2048),
                                 (248320, 5120)])
@pytest.mark.parametrize("n", [1, 64, 224, 300, 500, 700, 1001, 1500, 4096])
def test_dh_splits_fill_the_xcds_evenly(lib, n, v, d):
    """dh's grid is laid out by XCD only when its workgroups are a multiple of the 8 XCDs: no plan
    leaves it short of that (the workspace is its splits' fp32 partials), and no small vocabulary is cut
    into shares that cost more to sum than they save (few rows' sum costs next to nothing)."""
    tiles = -(-n // 256) * -(-d // 256)
    splits = lib.ns_workspace_bytes(_lib.NS_WS_LMHEAD_BWD, n, v, d) // (4 * n * d)
    assert 1 <= splits <= -(-v // 64)
    assert splits * tiles % 8 == 0 or splits < 8
    if v <= 4096 and n >= 224:
        assert splits <= 24


@pytest.mark.parametrize("v", [4096, 16384, 65536])
@pytest.mark.parametrize("n", [1, 4, 8])
def test_dh_of_few_rows_takes_most_of_a_round(lib, n, v):
    """Few rows' partials are small, so that more workgroups pay: one for each K stage (64 entries), or
    for more than half of the CUs."""
    splits = lib.ns_workspace_bytes(_lib.NS_WS_LMHEAD_BWD, n, v, 256) // (4 * n * 256)
    assert splits == v // 64 or splits > 128


def test_windows_of_kept_values_are_the_largest_that_fit(lib):
    """At V = 248,320 2 GiB hold eight token tiles' values: 3000 rows are windows of 2048 and 952 (whole
    XCD blocks of four token tiles), not two of 1536."""
    bytes_of = lambda n: lib.ns_workspace_bytes(_lib.NS_WS_LMHEAD, n, 248320, 5120)
    values = 2048 * 248320 * 4
    assert bytes_of(3000) >= values and bytes_of(2304) >= values
    assert bytes_of(100000) < values + (1 << 28)


@pytest.mark.parametrize("kind,v,d", [
    (_lib.NS_WS_LOGITS, 248320, 0), (_lib.NS_WS_LOGITS, 50001, 0), (_lib.NS_WS_LOGITS, 8192, 0),
    (_lib.NS_WS_LOGITS, 1, 0), (_lib.NS_WS_RMS_NORM_BWD, 0, 5120), (_lib.NS_WS_RMS_NORM_BWD, 0, 8),
])
def test_a_workspace_for_the_largest_n_takes_every_smaller_one(lib, kind, v, d):
    sizes = [lib.ns_workspace_bytes(kind, n, v, d) for n in [*range(2300), 4096, 8191, 8192, 8193, 20000]]
    assert all(a <= b for a, b in zip(sizes, sizes[1:]))
