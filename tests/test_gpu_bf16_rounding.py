"""BF16 pages are stored with round-to-nearest-even, NaN kept and infinities and
subnormals included: a fold whose result is the FP32 correction itself (zero
state, unit decay and keys) against torch's conversion, bit for bit."""

import pytest
import torch

from gdn_recoverssm_ascend.kernels import GDNRecoverSSMCommitContext, ReplayRecordBuffers

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [8, 64])
def test_bf16_store_rounding(gpu_device, K):
    dev, B, HV, V = gpu_device, 4, 8, 256
    gen = torch.Generator().manual_seed(K)
    n = B * HV * V
    bits = torch.randint(-(1 << 31), 1 << 31, (n,), generator=gen, dtype=torch.int64)
    bits[::4] = (bits[::4] & ~0xFFFF) | 0x8000  # ties
    bits[1::16] &= 0x807FFFFF  # subnormals
    edges = [0, 0x80000000, 0x7F800000, 0xFF800000, 0x7F7FFFFF, 0x7F7F8000, 0x7F7F7FFF, 0x7FC00000, 0x7F800001, 0x007F8000,
             0x00008000, 0x00007FFF, 0x3F808000, 0x3F818000, 0x3F80FFFF]
    bits[:len(edges)] = torch.tensor(edges)
    bits &= 0xFFFFFFFF
    bits = torch.where(bits >= 1 << 31, bits - (1 << 32), bits).to(torch.int32)
    corr = bits.view(torch.float32).view(B, HV, 1, V).to(dev)
    rec = ReplayRecordBuffers(corr, torch.ones(B, HV, 1, K, dtype=torch.bfloat16, device=dev),
                              torch.ones(B, HV, 1, device=dev))
    state = torch.zeros(B + 1, HV, V, K, dtype=torch.bfloat16, device=dev)
    conv = torch.zeros(B + 1, 4, 3, dtype=torch.bfloat16, device=dev)
    ctx = GDNRecoverSSMCommitContext.from_tensors([conv], [state], [rec], spec_query_len=1, max_num_reqs=B)
    ctx.commit(torch.ones(B, dtype=torch.int32, device=dev), torch.arange(1, B + 1, dtype=torch.int32, device=dev),
               torch.arange(B + 1, dtype=torch.int32, device=dev))
    want = corr[:, :, 0, :, None].expand(B, HV, V, K).cpu().to(torch.bfloat16)
    got = state[1:].cpu()
    nan = want.isnan()
    assert torch.equal(got.isnan(), nan)
    # The sum of a negative zero or underflow and +0 may lose its sign: compared by value.
    assert torch.equal(got[~nan], want[~nan])
