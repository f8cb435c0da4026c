"""What a call of the attention takes for a workspace: the shares of that call, and nothing where the keys are shared by wavefronts alone (a
workspace for other forms of the call costs an allocation, about 1 us of the host's time, at every step)."""
import math

import pytest
import torch

from gpu_util import note
from var_q_amd import _lib, ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('D', [64, 128])
@pytest.mark.parametrize('limits', [False, True])
@pytest.mark.parametrize('B,H,Lq,Lk', [(1, 8, 200, 400), (1, 8, 200, 200), (2, 16, 16, 21), (1, 8, 300, 2000), (2, 16, 144, 300)])
def test_allocates_what_the_call_uses(dev, D, limits, B, H, Lq, Lk):
    note('attention workspace', D, limits, B, H, Lq, Lk)
    lib = _lib.load()
    want = lib.varq_fused_attn_workspace_bytes_call(B, H, Lq, Lk, D, 1, 0, int(limits))
    assert want <= lib.varq_fused_attn_workspace_bytes(B, H, Lq, Lk, D, 1, 0)
    if (D, Lk, limits) == (64, 400, False):
        assert want == 0 and lib.varq_fused_attn_key_waves(B, H, Lq, Lk, D, int(limits)) > 1
    k, v = (ops.quant_pack_rows(torch.randn(B, H, Lk, D, device=dev), 64, 4, True) for _ in range(2))
    q, out = (torch.randn(B, H, Lq, D, device=dev).bfloat16() for _ in range(2))
    lim = torch.full((Lq,), Lk, dtype=torch.int32, device=dev) if limits else None
    run = lambda: ops.fused_attn(q, *k, *v, 4, 4, Lk, 1 / math.sqrt(D), kv_limit=lim, out=out)
    run()
    torch.cuda.synchronize()
    before = torch.cuda.memory_stats()['allocation.all.allocated']
    run()
    assert torch.cuda.memory_stats()['allocation.all.allocated'] - before == (1 if want else 0)
