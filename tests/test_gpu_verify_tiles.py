"""The verify's tiles of 16, 32, 64 and 128 rows of V at their edges, against the
CPU oracle (float64): value dims around multiples of the tile, batches on both
sides of each line of `verify_tile` (csrc/verify.hip), and q / k / v views whose
rows start at odd 16-bit elements (`load_run`'s two alignments).

Tolerances: test_gpu_verify's (FP32 corrections within 1e-5 norm-wise: sums of
K <= 256 products, 2^-23 each)."""

import pytest
import torch

import gdn_oracle as O
from gdn_recoverssm_ascend.kernels import ReplayRecordBuffers, gdn_recoverssm_verify
from gpu_helpers import CORR_TOL, OUT_TOL, assert_norm_close
from test_gpu_verify import _problem, _run_and_check

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev(gpu_device):
    return gpu_device


@pytest.mark.parametrize("V", [1, 15, 16, 17, 63, 65, 127, 129, 144, 200])
@pytest.mark.parametrize("state", [torch.float32, torch.bfloat16])
def test_value_dims_around_the_tiles(dev, V, state):
    # 16-row tiles (few waves).
    _run_and_check(_problem(3, 1, 2, 64, V, 4, qlens=[4, 1, 3], seed=V, state_dtype=state), dev)


@pytest.mark.parametrize("B,HV,V,Q", [(5, 32, 128, 4), (6, 32, 120, 4), (20, 32, 72, 3), (26, 32, 130, 4), (28, 32, 130, 4),
                                      (26, 32, 136, 8), (65, 32, 128, 1), (66, 32, 136, 1), (30, 32, 128, 2)])
def test_batches_around_each_line(dev, B, HV, V, Q):
    # 16 -> 64 rows past 1280 waves of 16, 64 -> 128 past 2560 waves of 64 (Q = 8:
    # 1024); Q = 1 keeps 16 rows to 16384 waves.
    _run_and_check(_problem(B, 4, HV, 128, V, Q, seed=B + V, null_rows=(1,)), dev)


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
