"""Row-local quantize+pack in windows of 256 octets: every group a lane can share, at the ends of a wavefront's and a workgroup's window,
into rows that lie side by side and into a cache whose tokens lie apart.  Codes, scales and zero-points bit for bit the oracle's."""
import pytest
import torch

import varq_oracle as O
from gpu_util import note
from var_q_amd import PackedKVCache, ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize('bits', [2, 4, 8])
@pytest.mark.parametrize('c,group', [(32, 32), (96, 32), (128, 64), (192, 64), (384, 128), (256, 256), (512, 512)])
def test_ends_of_windows(dev, dtype, bits, c, group):
    for octets in (256, 1024):
        for n in sorted({1, octets // (c // 8), octets // (c // 8) + 1}):
            note('windows', dtype, bits, c, group, n)
            x = (torch.randn(2, 3, n, c, generator=torch.Generator().manual_seed(n)) * 3).to(dtype)
            x[..., 7] *= 15
            q, s, z = O.quant_groupwise(x, group, bits, True)
            w, gs, gz = ops.quant_pack_rows(x.to(dev), group, bits, True)
            assert torch.equal(w.cpu(), O.pack_last_dim(q, bits)[0]) and torch.equal(gs.cpu(), s) and torch.equal(gz.cpu(), z)


@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16])
@pytest.mark.parametrize('bits', [2, 4, 8])
@pytest.mark.parametrize('group', [32, 64, 128])
@pytest.mark.parametrize('n', [1, 17, 65])
def test_token_major_rows(dev, dtype, bits, group, n):
    note('token-major windows', dtype, bits, group, n)
    k, v = ((torch.randn(2, n, 3, 128, generator=torch.Generator().manual_seed(i)) * 3).to(dtype).to(dev) for i in (1, 2))
    caches = [PackedKVCache(2, 3, n + 2, 128, bits, group, dev) for _ in range(2)]
    caches[0].append(k, v, layout='BLHc')
    caches[1].append(k.transpose(1, 2).contiguous(), v.transpose(1, 2).contiguous(), layout='BHLc')
    for name, t in caches[0].tensors().items():
        assert torch.equal(t[:, :, :n], caches[1].tensors()[name][:, :, :n]), name
