"""The key record holds the input key's own bits: signed zeros, subnormals and
infinities included, for every window capacity, activation type and page type,
also where a row's window starts at an odd 16-bit element."""

import pytest
import torch

from gdn_recoverssm_ascend.kernels import ReplayRecordBuffers, gdn_recoverssm_verify
from test_gpu_verify import _problem

pytestmark = pytest.mark.gpu

_BITS = {2: torch.int16, 4: torch.int32}


@pytest.fixture(scope="module")
def dev(gpu_device):
    return gpu_device


@pytest.mark.parametrize("Q", [1, 2, 3, 5])
@pytest.mark.parametrize("K", [64, 128, 256])
@pytest.mark.parametrize("act,state", [(torch.bfloat16, torch.float32), (torch.float32, torch.float32),
                                       (torch.float16, torch.float16), (torch.bfloat16, torch.bfloat16)])
@pytest.mark.parametrize("odd", [False, True])
def test_key_record_keeps_the_bits(dev, Q, K, act, state, odd):
    P = _problem(3, 2, 4, K, 32, Q, seed=Q + K, act=act, state_dtype=state)
    inp, T = P["inp"], P["T"]
    width = 2 * K
    tiny = torch.finfo(act).smallest_normal / 4  # subnormal
    marks = torch.tensor([0.0, -0.0, tiny, -tiny, float("inf"), -float("inf")], dtype=act)
    flat = inp.k.view(T, width)
    place = torch.arange(T * width).view(T, width)
    flat[place % 3 == 0] = marks[(place[place % 3 == 0] // 3) % len(marks)]
    store = torch.zeros(1 + T * (width + 1), dtype=act, device=dev)
    k = store.as_strided((1, T, 2, K), (store.numel(), width + odd, K, 1), int(odd))
    k.copy_(inp.k)
    rec = ReplayRecordBuffers.allocate(3, 4, 2, Q, 32, K, device=dev, key_dtype=act)
    gdn_recoverssm_verify(inp.g.to(dev), inp.beta.to(dev), inp.q.to(dev), k, inp.v.to(dev),
                          checkpoint_state=P["ckpt"].to(dev), replay_cache=rec, query_start_loc=P["qsl"].to(dev),
                          state_indices=P["idx"].to(dev), spec_query_len=Q)
    want = inp.k.view(3, Q, 2, K).transpose(1, 2)  # full windows: [row, head, token, K]
    bits = _BITS[act.itemsize]
    assert torch.equal(rec.key.cpu().view(bits), want.contiguous().view(bits))
