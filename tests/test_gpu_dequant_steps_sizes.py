"""A cache with one table per step dequantized with an octet per lane (up to 2^18 octets) and with four: the edges of workgroups of 256 and
1024 octets, step ends inside a workgroup and a wavefront, rows that are no power of two, both sides of the line."""
from ctypes import c_int32

import pytest
import torch

from gpu_util import note
from var_q_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('first', [0, 1])
@pytest.mark.parametrize('bits,asym', [(8, False), (4, True), (2, True)])
@pytest.mark.parametrize('B,H,c,ends', [
    (1, 1, 16, [1]), (3, 1, 16, [1, 5, 32]), (1, 2, 16, [127, 128, 129]), (2, 3, 48, [1, 2, 3, 43]), (1, 1, 128, list(range(1, 17))), (2, 4, 64, [32]),
    (32, 16, 64, [1, 63, 64]),             # 2^18 octets, and more
    (32, 16, 64, [1, 63, 65]), (40, 5, 48, [7, 300, 301, 450]), (9, 30, 64, [3, 17, 18, 19, 120, 129]), (2, 1, 16, [40000, 65537, 131074]), (1, 3, 48, list(range(1000, 17000, 1000))),
])
def test_both_sides_of_the_line(dev, first, bits, asym, B, H, c, ends):
    note('dequant_steps, sizes', first, bits, asym, B, H, c, ends)
    n, cap = ends[-1], ends[-1] + 3
    g = torch.Generator(device=dev).manual_seed(bits + n)
    half = 1 << (bits - 1)
    codes = torch.randint(-half, half, (B, cap, H, c) if first else (B, H, cap, c), device=dev, generator=g, dtype=torch.int32)
    fields = codes.reshape(*codes.shape[:3], -1, 32 // bits) & ((1 << bits) - 1)
    words = (fields << (torch.arange(32 // bits, device=dev, dtype=torch.int32) * bits)).sum(-1).to(torch.int32)
    scale = torch.rand(len(ends), H, c, device=dev, generator=g) + 0.1
    zp = torch.randn(len(ends), H, c, device=dev, generator=g).round() if asym else None
    step = torch.bucketize(torch.arange(n, device=dev), torch.tensor(ends, device=dev), right=True)
    table = (lambda t: t[step]) if first else (lambda t: t[step].transpose(0, 1))
    q = (codes[:, :n] if first else codes[:, :, :n]).float()
    want = (q - table(zp)) * table(scale) if asym else q * table(scale)
    lib, st = _lib.load(), torch.cuda.current_stream().cuda_stream
    for code, dt in ((0, torch.float32), (1, torch.bfloat16), (2, torch.float16)):
        buf = torch.full((want.numel() + 64,), 99.0, dtype=dt, device=dev)
        out = buf[32:][:want.numel()]
        _lib.check(lib.varq_dequant_steps(words.data_ptr(), scale.data_ptr(), None if zp is None else zp.data_ptr(), len(ends), (c_int32 * len(ends))(*ends),
                                          B, H, cap, c, bits, first, out.data_ptr(), code, st), 'varq_dequant_steps')
        assert torch.equal(out.view(want.shape), want.to(dt))
        assert bool((buf[:32] == 99.0).all()) and bool((buf[32 + want.numel():] == 99.0).all()), 'wrote around its output'
