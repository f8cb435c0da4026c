"""Tokens first with so many heads that a row of codes (all heads of a token) is 16 MiB or longer: the kernel
addresses its tiles with 64 bits per lane there.  The result of a head is that of the same head in a short call."""
import math

import pytest
import torch

from gpu_util import note
from var_q_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('H', [262143, 262144])          # rows just below and of 2^24 bytes
@pytest.mark.parametrize('Lk', [3, 70])                  # part of a tile; a whole one and part of the next
def test_long_rows(dev, H, Lk):
    D, bits, group, Lq = 64, 8, 32, 17
    gen = torch.Generator(device=dev).manual_seed(Lk)
    kw, vw = (torch.randint(-2 ** 31, 2 ** 31 - 1, (1, Lk, H, D * bits // 32), device=dev, generator=gen, dtype=torch.int32) for _ in range(2))
    ks, vs = (torch.rand(1, Lk, H, D // group, device=dev, generator=gen) * 0.02 + 0.01 for _ in range(2))
    kz, vz = (torch.randint(-9, 9, (1, Lk, H, D // group), device=dev, generator=gen).float() for _ in range(2))
    q = torch.randn(1, Lq, H, D, device=dev, generator=gen).bfloat16()
    part = lambda t, at: None if t is None else t[:, :, at:at + 8].contiguous()
    for zk, zv in ((kz, vz), (None, None)):
        note('long rows', H, Lk, zk is not None)
        out = ops.fused_attn(q, kw, ks, zk, vw, vs, zv, bits, bits, Lk, 1 / math.sqrt(D), layout='BLHc', splits=1)
        for at in (0, H // 2, H - 8):
            few = [part(t, at) for t in (q, kw, ks, zk, vw, vs, zv)]
            want = ops.fused_attn(*few, bits, bits, Lk, 1 / math.sqrt(D), layout='BLHc', splits=1)
            assert torch.equal(out[:, :, at:at + 8], want), at
