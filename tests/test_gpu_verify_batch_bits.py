"""A row's verify gives the same bits in any launch: alone with few rows (16-row
tiles) and in batches whose tiles are longer (`verify_tile`, csrc/verify.hip), where
products may take another matrix instruction; ordinary, gated and deferred."""

import pytest
import torch

from gdn_recoverssm_ascend import workloads as W
from gdn_recoverssm_ascend.kernels import ReplayRecordBuffers, gdn_recoverssm_verify, gdn_recoverssm_verify_gated
from test_gpu_deferred import _assert_flows_equal, _flow
from verify_tiles import verify_tile, window_capacity

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev(gpu_device):
    return gpu_device


def _batch(B, H, HV, K, V, Q, state, act, dev, gated):
    gen = torch.Generator(device=dev).manual_seed(K + Q)

    def randn(*shape):
        return torch.randn(*shape, generator=gen, device=dev)

    q, k = randn(1, B * Q, H, K), randn(1, B * Q, H, K)
    if not gated:
        q, k = (x / x.norm(dim=-1, keepdim=True) for x in (q, k))
    return dict(g=-torch.nn.functional.softplus(randn(B * Q, HV)), beta=torch.sigmoid(randn(B * Q, HV)), q=q.to(act),
                k=k.to(act), v=randn(1, B * Q, HV, V).to(act), pages=(0.1 * randn(B + 1, HV, V, K)).to(state))


def _verify(x, rows, Q, dev, gated):
    """The first `rows` rows of the batch (full windows)."""
    T, (HV, V), (H, K) = rows * Q, x["v"].shape[2:], x["k"].shape[2:]
    rec = ReplayRecordBuffers.allocate(rows, HV, H, Q, V, K, device=dev, key_dtype=torch.float32)
    kw = dict(checkpoint_state=x["pages"], replay_cache=rec, spec_query_len=Q,
              query_start_loc=torch.arange(0, T + 1, Q, dtype=torch.int32, device=dev),
              state_indices=torch.arange(1, rows + 1, dtype=torch.int32, device=dev))
    args = (x["g"][:T], x["beta"][:T], x["q"][:, :T], x["k"][:, :T], x["v"][:, :T])
    if gated:
        out = gdn_recoverssm_verify_gated(*args, A_log=torch.zeros(HV, device=dev), dt_bias=torch.zeros(HV, device=dev),
                                          **kw)
    else:
        out = gdn_recoverssm_verify(*args, **kw)
    return out[0].view(rows, Q, HV, V), rec.correction, rec.key, rec.decay


@pytest.mark.parametrize("gated", [False, True])
@pytest.mark.parametrize("K,V,state,act", [
    (128, 120, torch.float32, torch.bfloat16), (64, 120, torch.float32, torch.bfloat16),
    (256, 72, torch.float32, torch.float16), (128, 120, torch.bfloat16, torch.bfloat16),
    (112, 100, torch.float16, torch.float32), (64, 120, torch.float16, torch.float16),
    (48, 88, torch.bfloat16, torch.float32), (256, 120, torch.bfloat16, torch.bfloat16)])
@pytest.mark.parametrize("Q", [1, 2, 4, 5, 8])
def test_rows_give_the_same_bits_in_any_launch(dev, Q, K, V, state, act, gated):
    HV, sizes = 32, (3, 14, 70)
    tiles = [verify_tile(rows, HV, K, V, state == torch.float32, window_capacity(Q), False) for rows in sizes]
    assert tiles[0] == 16 and tiles[2] == 128, tiles
    print(f"batch bits Q={Q} K={K} V={V} {state} {act} gated={gated}: tiles {tiles}", flush=True)
    x = _batch(sizes[-1], 4, HV, K, V, Q, state, act, dev, gated)
    want = _verify(x, sizes[-1], Q, dev, gated)
    for rows in sizes[:-1]:
        for name, got, ref in zip(("out", "correction", "key", "decay"), _verify(x, rows, Q, dev, gated), want):
            assert torch.equal(got, ref[:rows]), f"{name} of {rows} rows"


@pytest.mark.parametrize("K,V,state,act", [
    (128, 96, torch.float32, torch.bfloat16), (64, 120, torch.float32, torch.float16),
    (256, 64, torch.float32, torch.bfloat16), (128, 120, torch.bfloat16, torch.bfloat16),
    (64, 64, torch.float16, torch.float16), (48, 40, torch.bfloat16, torch.float32),
    (256, 56, torch.float16, torch.float16)])
@pytest.mark.parametrize("Q", [1, 3, 6])
def test_deferred_tiles_equal_the_ordinary_flow(dev, Q, K, V, state, act):
    """The deferred flow of a batch whose verify takes 32- and 64-row tiles equals
    the ordinary flow (verify then commit) bit for bit, boundary snapshots and a
    last tile cut by V included."""
    H, HV, steps = 4, 32, 3
    seen = set()
    for rows in (22, 58):
        tile = verify_tile(rows, HV, K, V, state == torch.float32, window_capacity(Q), True)
        seen.add(tile)
        print(f"deferred bits Q={Q} K={K} V={V} {state} {act}: {rows} rows, tile {tile}", flush=True)
        w = W.make_workload("decode_loop_l48", layers=1, rows=rows, key_heads=H, value_heads=HV, key_dim=K, value_dim=V,
                            window=Q, act_dtype=act, state_dtype=state, steps=steps, max_position=256, block_size=8,
                            padded_rows=1, seed=K + V + Q + rows, gen_device=dev.type)
        gen = torch.Generator().manual_seed(K * V + Q)
        acc_steps = [W.sample_accepted(w.spec, rows, gen) for _ in range(steps)]
        qsl_steps = [w.meta.query_start_loc.clone() for _ in range(steps)]
        lens = torch.full((rows,), Q, dtype=torch.int32)
        lens[rows // 2] = 0  # a row with nothing to verify, its commit pending
        qsl_steps[-1][1:] = torch.cumsum(lens, 0)
        ref = _flow(w, dev, acc_steps, qsl_steps, deferred=False)
        _assert_flows_equal(ref, _flow(w, dev, acc_steps, qsl_steps, deferred=True))
    assert seen - {16}
