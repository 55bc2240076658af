"""The ordinary and gated verify's tiles of 16, 64 and 128 rows of V at their edges,
against the CPU oracle (float64): value dims around multiples of the tile, batches
on both sides of each line of `verify_tile` (csrc/verify.hip), the sweeps' draws
enlarged until their tiles are long, and q / k / v views whose rows start at odd
16-bit elements (`load_run`'s two alignments). The deferred verify's tiles:
test_gpu_verify_batch_bits.py.

Tolerances: test_gpu_verify's (FP32 corrections within 1e-5 norm-wise: sums of
K <= 256 products, 2^-23 each)."""

import pytest
import torch

import gdn_oracle as O
import sweep_cases as SC
from gdn_recoverssm_ascend.kernels import ReplayRecordBuffers, gdn_recoverssm_verify
from gpu_helpers import CORR_TOL, OUT_TOL, assert_norm_close
from test_gpu_verify import _gated_check, _problem, _run_and_check
from verify_tiles import verify_tile, window_capacity

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev(gpu_device):
    return gpu_device


@pytest.mark.parametrize("V", [1, 15, 16, 17, 63, 65, 127, 129, 144, 200])
@pytest.mark.parametrize("state", [torch.float32, torch.bfloat16])
def test_value_dims_around_the_tiles(dev, V, state):
    # 16-row tiles (few waves).
    _run_and_check(_problem(3, 1, 2, 64, V, 4, qlens=[4, 1, 3], seed=V, state_dtype=state), dev)


def _tile(B, HV, K, V, Q, state=torch.float32):
    return verify_tile(B, HV, K, V, state == torch.float32, window_capacity(Q), False)


LINES = [  # (value heads, K, V, Q, largest batch on one side, its tile, the next batch's)
    (32, 128, 128, 4, 5, 16, 64), (32, 128, 120, 4, 40, 64, 128), (32, 128, 120, 8, 5, 16, 64), (32, 128, 120, 8, 16, 64, 128),
    (32, 128, 128, 1, 48, 16, 128), (32, 256, 120, 1, 16, 16, 64), (32, 128, 120, 1, 48, 16, 128),
    (32, 64, 120, 1, 6, 16, 64), (32, 128, 120, 2, 15, 64, 16), (32, 128, 120, 2, 32, 16, 64),
]


@pytest.mark.parametrize("HV,K,V,Q,B,tile,after", LINES)
def test_batches_around_each_line(dev, HV, K, V, Q, B, tile, after):
    assert (_tile(B, HV, K, V, Q), _tile(B + 1, HV, K, V, Q)) == (tile, after)
    for rows in (B, B + 1):
        _run_and_check(_problem(rows, 4, HV, K, V, Q, seed=rows + V, null_rows=(1,)), dev)


@pytest.mark.parametrize("V,tile", [(32, 16), (33, 64), (64, 64), (65, 128), (128, 128), (129, 64), (192, 64), (193, 128)])
def test_value_dims_around_each_line(dev, V, tile):
    B = 72  # past every line in waves
    assert _tile(B, 64, 16, V, 4) == tile
    _run_and_check(_problem(B, 4, 64, 16, V, 4, seed=V, null_rows=(2,), oob_rows=(5,)), dev)


def _enlarged(p, tile):
    """A sweep draw's problem with more value heads and rows (its windows
    repeated), so that its verify takes tiles of `tile` rows."""
    H, K, Q, state = p["H"], p["K"], p["Q"], p["state_dtype"]
    HV = H * 4 * (16 // H)
    V = p["V"] if p["V"] > 32 else 100
    if tile == 128 and (V - 1) % 128 < 64:
        V += 64
    for B in range(len(p["qlens"]), 400):
        if _tile(B, HV, K, V, Q, state) == tile:
            qlens = (p["qlens"] * B)[:B]
            return dict(p, B=B, HV=HV, V=V, qlens=qlens)
    raise AssertionError((p, tile))


@pytest.mark.parametrize("case", range(10))
@pytest.mark.parametrize("tile", [64, 128])
def test_random_configurations_on_long_tiles(dev, case, tile):
    c = SC.verify_case(case)
    p = _enlarged(c["problem"], tile)
    run = dict(c["run"], record_rows=p["B"] - case % 2)
    print(f"long tiles {tile} case {case}: {p} {run}", flush=True)
    _run_and_check(_problem(**p), dev, **run)


@pytest.mark.parametrize("case", range(6))
@pytest.mark.parametrize("tile", [64, 128])
def test_random_gated_on_long_tiles(dev, case, tile):
    c = SC.gated_case(case)
    p = _enlarged(dict(B=c["B"], H=c["H"], HV=c["HV"], K=c["K"], V=c["V"], Q=c["Q"], qlens=c["qlens"],
                       null_rows=c["null_rows"], oob_rows=c["oob_rows"], normalise=False, act=c["act"],
                       state_dtype=c["state"], seed=c["seed"]), tile)
    print(f"gated long tiles {tile} case {case}: {p}", flush=True)
    _gated_check(dev, _problem(**p), c["ab"], c["param"], seed=c["seed"] + 1)


@pytest.mark.parametrize("B,K,Q,state", [(65, 256, 1, torch.float32), (41, 136, 2, torch.float32),
                                         (41, 256, 4, torch.float32), (17, 256, 8, torch.float32),
                                         (17, 160, 6, torch.bfloat16)])
def test_long_tiles_of_wide_rows(dev, B, K, Q, state):
    # 128-row tiles with K > 128: two waves per SIMD, and 8-row blocks at Q = 8 (verify_block_rows).
    _run_and_check(_problem(B, 4, 32, K, 120, Q, seed=B + K, state_dtype=state), dev)


@pytest.mark.parametrize("K", [8, 48, 64])
@pytest.mark.parametrize("Q", [1, 2, 4, 8])
@pytest.mark.parametrize("state,act", [(torch.bfloat16, torch.bfloat16), (torch.float16, torch.float16),
                                       (torch.bfloat16, torch.float32)])
@pytest.mark.parametrize("B,V", [(3, 33), (14, 120), (66, 120)])
def test_narrow_16bit_rows(dev, K, Q, state, act, B, V):
    # Pages of K <= 64 16-bit elements: a row over 8 blocks, tiles of 16, 64 and 128.
    _run_and_check(_problem(B, 2, 32, K, V, Q, seed=B + K + Q, state_dtype=state, act=act), dev)


@pytest.mark.parametrize("act", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("Q,state", [(1, torch.float32), (2, torch.bfloat16), (4, torch.float32), (4, torch.bfloat16),
                                     (8, torch.float32)])
def test_rows_starting_at_odd_elements(dev, act, Q, state):
    """q, k and v as views at an odd element offset and an odd token stride,
    ending with their storage (the last run's loads stay inside it)."""
    P = _problem(3, 2, 4, 64, 48, Q, seed=Q, act=act, state_dtype=state)
    inp, T = P["inp"], P["T"]

    def odd(x):
        heads, dim = x.shape[2:]
        width = heads * dim
        store = torch.full((1 + (T - 1) * (width + 1) + width,), float("nan"), dtype=x.dtype, device=dev)
        view = store.as_strided((1, T, heads, dim), (store.numel(), width + 1, dim, 1), 1)
        view.copy_(x)
        return view

    rec = ReplayRecordBuffers.allocate(3, 4, 2, Q, 48, 64, device=dev, key_dtype=act)
    out = gdn_recoverssm_verify(inp.g.to(dev), inp.beta.to(dev), odd(inp.q), odd(inp.k), odd(inp.v),
                                checkpoint_state=P["ckpt"].to(dev), replay_cache=rec,
                                query_start_loc=P["qsl"].to(dev), state_indices=P["idx"].to(dev), spec_query_len=Q)
    res = O.oracle_verify(inp.q, inp.k, inp.v, inp.g, inp.beta, P["ckpt"], P["qsl"], P["idx"], Q)
    assert_norm_close(out.cpu()[0].double(), res.out, OUT_TOL, "out")
    assert_norm_close(rec.correction.cpu().double(), res.correction, CORR_TOL, "correction")
    assert torch.equal(rec.key.cpu().float(), res.key.float())
