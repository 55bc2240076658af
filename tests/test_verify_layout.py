"""The verify's LDS staging of the 16x16x1 form (csrc/verify_kernel.cuh, `stage_slot`,
`stage_block` and `wide_block`), restated on the CPU for the chunk counts it is
instantiated with: rows of CPR = 16 chunks of 16 bytes (256 bytes) loaded over N = 16
blocks, and of CPR = 8 (64 16-bit elements) over N = 8. A block is 16 rows; load g
gives lane l the chunk kb of row ROWS*g + lr and writes it to slot r*CPR +
(c ^ swz(r)); operand register j of lane l reads chunk 4j + l / 16 of row l % 16 back.
Checked: every operand register receives exactly the chunk the matrix-core layout
assigns it, the loads cover the block once, and the 16 lanes of each quarter of a
write, and the 16 rows a read takes of one chunk, hit 16 distinct 16-byte bank
groups. The GPU tests compare the form's results with the 4x4x1 form's bit for bit."""

import pytest


def _geometry(cpr):
    n = cpr  # blocks (of four lanes) that share a row
    rows = 64 // n
    swz = (lambda r: ((r & 3) << 2) | (r >> 2)) if cpr == 16 else (lambda r: ((r & 2) << 1) | (r >> 2))
    return n, rows, lambda r, c: r * cpr + (c ^ swz(r))


def _written(cpr, g):
    """(row, chunk) of each lane of load g."""
    n, rows, _ = _geometry(cpr)
    return [(rows * g + (lane & 3 if n == 16 else 4 * (lane >> 5) + (lane & 3)), (lane >> 2) & (n - 1))
            for lane in range(64)]


@pytest.mark.parametrize("cpr", [16, 8])
def test_staging_maps_row_runs_to_the_operand_layout(cpr):
    _, rows, slot = _geometry(cpr)
    stage = {}
    for g in range(16 // rows):
        at = [slot(r, c) for r, c in _written(cpr, g)]
        for lane, rc in enumerate(_written(cpr, g)):
            assert at[lane] not in stage
            stage[at[lane]] = rc
        for quarter in range(0, 64, 16):
            assert len({x % 16 for x in at[quarter:quarter + 16]}) == 16, "bank conflict in a write"
    assert sorted(stage) == list(range(16 * cpr)), "the stage must be filled exactly once"
    for j in range(cpr // 4):
        for quarter in range(4):
            at = [slot(row, 4 * j + quarter) for row in range(16)]
            assert [stage[x] for x in at] == [(row, 4 * j + quarter) for row in range(16)]
            assert len({x % 16 for x in at}) == 16, "bank conflict among the lanes of one read"


@pytest.mark.parametrize("cpr", [16, 8])
def test_row_run_loads_cover_the_block_once(cpr):
    _, rows, _ = _geometry(cpr)
    seen = [rc for g in range(16 // rows) for rc in _written(cpr, g)]
    assert sorted(seen) == [(r, c) for r in range(16) for c in range(cpr)]
