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
        assert want == 0 and lib.varq_fused_attn_key_waves(B, H, Lq, Lk, D, 1, int(limits)) > 1
    k, v = (ops.quant_pack_rows(torch.randn(B, H, Lk, D, device=dev), 64, 4, True) for _ in range(2))
    q, out = (torch.randn(B, H, Lq, D, device=dev).bfloat16() for _ in range(2))
    lim = torch.full((Lq,), Lk, dtype=torch.int32, device=dev) if limits else None
    run = lambda: ops.fused_attn(q, *k, *v, 4, 4, Lk, 1 / math.sqrt(D), kv_limit=lim, out=out)
    run()
    torch.cuda.synchronize()
    before = torch.cuda.memory_stats()['allocation.all.allocated']
    run()
    assert torch.cuda.memory_stats()['allocation.all.allocated'] - before == (1 if want else 0)


def test_a_workspace_that_cannot_be_used(dev):
    """Off a 16-byte boundary, where only the shares under key limits would use it: let alone, and the call is served without."""
    from ctypes import c_float, c_size_t, c_void_p
    B, H, D, Lq, Lk = 1, 200, 64, 132, 2131
    note('attention: unaligned workspace')
    lib = _lib.load()
    k, v = (ops.quant_pack_rows(torch.randn(B, H, Lk, D, device=dev), 64, 4, True) for _ in range(2))
    q = torch.randn(B, H, Lq, D, device=dev).bfloat16()
    lim = torch.full((Lq,), Lk, dtype=torch.int32, device=dev)
    need = lib.varq_fused_attn_workspace_bytes_call(B, H, Lq, Lk, D, 1, 0, 1)
    assert need > 0
    ws = torch.empty(need + 16, dtype=torch.uint8, device=dev)
    out = torch.empty_like(q)

    def run(off):
        p = lambda t: c_void_p(t.data_ptr())
        return lib.varq_fused_attn(p(q), p(out), *map(p, k), 4, 64, *map(p, v), 4, 64, B, H, H, None, Lq, Lk, Lk, D, p(lim),
                                   c_float(1 / math.sqrt(D)), 0, 1, 0, c_void_p(ws.data_ptr() + off), c_size_t(need), 0, c_void_p(torch.cuda.current_stream().cuda_stream))
    assert run(8) == 0
    got = out.clone()
    assert run(0) == 0
    torch.testing.assert_close(got.float(), out.float(), rtol=2 ** -6, atol=2 ** -7 * float(out.abs().max()))   # (another order of the sums)
