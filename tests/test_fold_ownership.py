"""Which thread of which workgroup loads and stores each 16-byte chunk of a
(page, head) state tile, restated on the CPU from the index arithmetic of the
kernels that write state pages in place:

* the fold (csrc/fold.hip, ``fold_body``): one 256-thread workgroup per
  (layer, row, value head); thread ``tid`` owns chunk ``tid % KCH`` of rows
  ``tid // KCH + pass * RP``; passes go in batches of ``64 / E`` loads, each
  batch's stores after its loads;
* the deferred verify (csrc/verify_kernel.cuh, ``DEFER``): one wave per
  (row, value head, tile of 16, 32 or 64 rows); block ``rb``'s stores (final
  page and boundary snapshot) come after its loads, and the loads of block
  ``rb + 2`` after those stores.

A row's source, final and boundary pages may be one page (the plan makes
``boundary == source`` whenever the window crosses a block boundary from the
block the row started in; the alias case of the reference's
tests/test_math_oracle.py:206-235). Folding in place is then correct only if
every chunk of the tile is loaded and stored by exactly one thread, and that
thread stores it only after loading it: a chunk loaded by one thread after
another thread stored it would be folded twice. The checks below establish
both properties for every tile shape the kernels accept, and show that a
decomposition splitting a tile's passes between two workgroups whose batches
still span the whole tile breaks them (the failure such a split would have
in the alias case).
"""

import itertools

import pytest

FOLD_THREADS = 256


def _fold_events(K, V, E, vs, split=None):
    """(workgroup, thread, batch, kind, chunk) for every in-tile access of one
    fold tile, in each thread's program order. ``split`` models two
    workgroups per tile, workgroup h taking passes from h * passes / 2 and
    loading whole batches of ITERS passes from there (the mutant)."""
    kch, kch_log = 1, 0
    while kch * E < K:
        kch, kch_log = kch * 2, kch_log + 1
    RP = FOLD_THREADS // kch
    ITERS = 64 // E
    passes = -(-V // RP)
    events = []
    groups = [(0, 0, passes)] if split is None else [(h, h * passes // 2, (h + 1) * passes // 2) for h in range(2)]
    for wg, lo, hi in groups:
        for tid in range(FOLD_THREADS):
            kc, r0 = tid & (kch - 1), tid >> kch_log
            if kc * E >= K:
                continue
            last = hi if split is None else lo + ITERS * (-(-(hi - lo) // ITERS))
            for batch, first in enumerate(range(lo, last, ITERS)):
                rows = [r0 + (first + i) * RP for i in range(ITERS)]
                # The tile's buffer resource spans V rows of vs elements.
                chunks = [(r, kc) for r in rows if r * vs + kc * E < V * vs]
                for ch in chunks:
                    events.append((wg, tid, batch, "load", ch))
                for ch in chunks:
                    events.append((wg, tid, batch, "store", ch))
    return events


def _check_single_owner(events, K, V, E):
    """Every chunk of the tile loaded once and stored once, by the same
    (workgroup, thread), its store after its load in that thread's order."""
    want = {(r, c) for r in range(V) for c in range(-(-K // E))}
    owner_load, owner_store = {}, {}
    order = {}
    for i, (wg, tid, batch, kind, ch) in enumerate(events):
        table = owner_load if kind == "load" else owner_store
        if ch in table:
            return f"chunk {ch} {kind}ed twice"
        table[ch] = (wg, tid)
        order[(kind, ch)] = i
    if set(owner_load) != want or set(owner_store) != want:
        return "the accesses do not cover the tile"
    for ch in want:
        if owner_load[ch] != owner_store[ch]:
            return f"chunk {ch} stored by another thread than the one that loaded it"
        if order[("store", ch)] < order[("load", ch)]:
            return f"chunk {ch} stored before its load"
    return None


SHAPES = [
    # (K, V, E, row stride): FP32 (E=4) and 16-bit (E=8) state, the benchmark's
    # 128 x 128, head dims off the tile, several batches of passes, padded rows.
    (128, 128, 4, 128), (128, 128, 8, 128), (256, 1024, 4, 256), (96, 128, 4, 96), (192, 64, 8, 192),
    (16, 32, 4, 16), (256, 256, 8, 256), (128, 200, 4, 132), (64, 1024, 8, 64), (32, 8, 4, 32),
]


@pytest.mark.parametrize("K,V,E,vs", SHAPES)
def test_fold_tile_has_one_owner_per_chunk(K, V, E, vs):
    assert _check_single_owner(_fold_events(K, V, E, vs), K, V, E) is None


@pytest.mark.parametrize("K,V,E,vs", [(128, 128, 4, 128), (128, 128, 8, 128)])
def test_split_with_whole_batches_breaks_the_single_owner_rule(K, V, E, vs):
    """Two workgroups per tile whose batches run past their half of the
    passes load and store the same chunks: with source == boundary, the
    second can read a chunk after the first stored its snapshot there."""
    problem = _check_single_owner(_fold_events(K, V, E, vs, split=True), K, V, E)
    assert problem is not None and "twice" in problem


def _alias_fold(h0, decay, c, k, n, blen, two_pass):
    """The scalar alias case: source == boundary page. A correct fold reads
    the source once; a second reader after the snapshot store folds the
    snapshot again."""
    h = h0
    pages = {"src": h0}
    snap = None
    for t in range(n):
        h = c * k + h * decay
        if t + 1 == blen:
            snap = h
            pages["src"] = snap  # boundary page is the source page
    final = h
    if two_pass:
        h2 = pages["src"]  # a second workgroup loading after the snapshot store
        for t in range(n):
            h2 = c * k + h2 * decay
        final = h2
    return final, snap


def test_alias_case_known_answer_and_the_double_fold():
    """tests/test_math_oracle.py:206-235 of the reference: h0 = 10, decay 0.5,
    c = k = 1, n = 3, boundary after 2 tokens: final 3, boundary 4; reading
    the source again after the snapshot store gives 2.25."""
    final, snap = _alias_fold(10.0, 0.5, 1.0, 1.0, 3, 2, two_pass=False)
    assert (final, snap) == (3.0, 4.0)
    bad, _ = _alias_fold(10.0, 0.5, 1.0, 1.0, 3, 2, two_pass=True)
    assert bad == 2.25


def _defer_events(K, V, E, vs, tile, block=16):
    """The deferred verify for one (row, value head): wave vt covers rows
    [tile * vt, tile * vt + tile) in blocks; register g*J + j of a block is
    loaded, and stored back after its fold, at row ROWS*g + lr, chunk N*j + kb
    (RowLanes: a row over N = 16 blocks of four lanes, over 8 for up to 64
    16-bit elements). Blocks rb and rb + 1 are in flight together, rb + 2 is
    loaded after rb's stores. Chunks past K get an out-of-range offset, rows
    past V lie outside the tile's resource of tile_rows * vs elements."""
    kp = 64 if K <= 64 else 128 if K <= 128 else 256
    N = 8 if E == 8 and kp == 64 else 16
    J, rows_per_load = kp // (N * E), 64 // N
    events = []
    for vt in range(-(-V // tile)):
        row0 = vt * tile
        tile_rows = min(tile, V - row0)

        def accesses(rb):
            out = []
            for g in range(block // rows_per_load):
                for j in range(J):
                    for lane in range(64):
                        kb, ij = (lane >> 2) & (N - 1), lane & 3
                        lr = ij if N == 16 else 4 * (lane >> 5) + ij
                        r, c = rb * block + rows_per_load * g + lr, N * j + kb
                        if c * E < K and r * vs + c * E < tile_rows * vs:
                            out.append((lane, (row0 + r, c)))
            return out

        blocks = tile // block
        order = [("load", rb) for rb in range(min(2, blocks))]
        for rb in range(blocks):
            order.append(("store", rb))
            if rb + 2 < blocks:
                order.append(("load", rb + 2))
        for kind, rb in order:
            for lane, ch in accesses(rb):
                events.append((vt, lane, 0, kind, ch))
    return events


@pytest.mark.parametrize("K,E", [(128, 4), (128, 8), (256, 4), (256, 8), (64, 4), (64, 8), (8, 8), (16, 4), (96, 4),
                                 (136, 8)])
@pytest.mark.parametrize("V", [128, 96, 40, 17, 8])
@pytest.mark.parametrize("tile", [16, 32, 64])
def test_deferred_verify_tile_has_one_owner_per_chunk(K, V, E, tile):
    for block in (16, 8) if E == 4 and K > 128 else (16,):  # 8-row blocks: FP32 pages of K > 128 at Q > 4
        assert _check_single_owner(_defer_events(K, V, E, K, tile, block), K, V, E) is None


def test_overlapping_deferred_tiles_break_the_single_owner_rule():
    """Tiles that advance by less than their rows share chunks."""
    events = _defer_events(128, 64, 4, 128, 32)
    moved = [(wg, lane, b, kind, (r - 16 * wg, c)) for wg, lane, b, kind, (r, c) in events]
    problem = _check_single_owner(moved, 128, 48, 4)
    assert problem is not None and "twice" in problem


def test_plan_outputs_never_feed_the_fused_launch():
    """In the fused plan + fold launch the writer workgroups store the plan
    arrays while the folding workgroups plan from the step's metadata; the
    two sets must not share memory (the host refuses overlapping ranges).
    The folding workgroups' reads, per csrc/plan_row.cuh and csrc/fold.hip."""
    fold_reads = {"state_indices", "query_start_loc", "request_indices", "sampled", "num_computed", "block_table",
                  "layer_tables", "layer_groups", "records", "decay"}
    writer_writes = {"source_plan", "lens_plan", "final_plan", "boundary_plan", "boundary_lens_plan", "valid_plan",
                     "col_plan", "persistent_cols", "persistent_accepted"}
    assert not fold_reads & writer_writes
    for a, b in itertools.combinations(sorted(writer_writes), 2):
        assert a != b
