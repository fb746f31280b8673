"""The tile-row rule of an all-Q4_0 layer at its lines (lmoe_grouped_pick_tile_rows, a host function): 32 rows below 6
rows an expert (of at most 48 experts below 16, where split-K fills the chip), 64 below 48, else 128. The GEMMs give the
same bits at every tile height (test_gpu_grouped.py). On stream copies (lmoe_grouped_pick_tile_rows_sl) the lines are 40 and
64."""
import pytest

from larder_amd import _lib


@pytest.mark.parametrize("E", (1, 8, 48, 49, 60, 128, 512))
@pytest.mark.parametrize("rows,off,want", (("low", -1, 32), ("low", 0, 64), (48, -1, 64), (48, 0, 128)))
def test_q4_0_tile_rows_at_the_lines(built_lib, monkeypatch, E, rows, off, want):
    monkeypatch.delenv("LMOE_TILE_ROWS", raising=False)
    monkeypatch.delenv("LMOE_KSPLIT", raising=False)
    q = _lib.qcode("Q4_0")
    if rows == "low":
        rows = 16 if E <= 48 else 6
    assert built_lib.lmoe_grouped_pick_tile_rows(rows * E + off, E, q, q, q) == want
    # split-K up to the line, none past the 32-row tiles
    assert (built_lib.lmoe_grouped_pick_ksplit(rows * E + off, E, want, 2048) == 1) == (want != 32)


@pytest.mark.parametrize("R,E,want", ((0, 128, 32), (1, 1, 32), (2 ** 31 - 1, 1, 128), (2 ** 31 - 1, 2 ** 30, 32)))
def test_q4_0_tile_rows_at_the_ends(built_lib, monkeypatch, R, E, want):
    monkeypatch.delenv("LMOE_TILE_ROWS", raising=False)
    q = _lib.qcode("Q4_0")
    assert built_lib.lmoe_grouped_pick_tile_rows(R, E, q, q, q) == want


@pytest.mark.parametrize("E", (1, 48, 60, 512))
@pytest.mark.parametrize("rows,off,want", ((40, -1, 32), (40, 0, 64), (64, -1, 64), (64, 0, 128)))
def test_q4_0_tile_rows_on_stream_copies(built_lib, monkeypatch, E, rows, off, want):
    monkeypatch.delenv("LMOE_TILE_ROWS", raising=False)
    q, k = _lib.qcode("Q4_0"), _lib.qcode("Q4_K")
    assert built_lib.lmoe_grouped_pick_tile_rows_sl(rows * E + off, E, q, q, q) == want
    for ts in ((k, k, k), (q, q, k), (k, k, q)):  # the other types' heights do not depend on the layout
        assert built_lib.lmoe_grouped_pick_tile_rows_sl(rows * E + off, E, *ts) == \
            built_lib.lmoe_grouped_pick_tile_rows(rows * E + off, E, *ts)
    monkeypatch.setenv("LMOE_TILE_ROWS", "128")
    assert built_lib.lmoe_grouped_pick_tile_rows_sl(rows * E + off, E, q, q, q) == 128
