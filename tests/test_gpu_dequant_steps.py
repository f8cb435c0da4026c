"""The cache of a stepwise quantizer dequantized from one scale table per step, against the oracle's
dequantization of every step: step ends inside a lane's pieces and workgroups, rows that are no power
of two, spare room in the buffer, the largest number of steps."""
import pytest
import torch

import varq_oracle as O
from gpu_util import note
from var_q_amd import VAR_Q

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('fmt', ['BLHc', 'BHLc'])
@pytest.mark.parametrize('bits,H,c', [(8, 5, 24), (4, 3, 40), (2, 7, 80), (8, 30, 64), (4, 2, 128)])
@pytest.mark.parametrize('steps', [(1,), (1, 3, 2, 5), tuple(range(1, 17)), (300, 1, 700)])
def test_stepwise_cache(dev, fmt, bits, H, c, steps):
    note('dequant_steps', fmt, bits, H, c, steps)
    g = torch.Generator().manual_seed(bits + H + c)
    dim = 1 if fmt == 'BLHc' else 2
    for sym in (True, False):
        q = VAR_Q(bits, fmt, symmetric=sym)
        want = []
        for i, n in enumerate(steps):
            x = torch.randn(*((2, n, H, c) if dim == 1 else (2, H, n, c)), generator=g) * (i + 1) + 0.3
            codes, s, z = O.quant_reduce(x, (0, dim), bits, not sym)
            want.append(O.dequant_sym(codes, s) if sym else O.dequant_asym(codes, s, z))
            got = q.use_var_q(x.to(dev))
        want = torch.cat(want, dim)
        assert torch.equal(got.cpu(), want)
        for dt in (torch.bfloat16, torch.float16):
            assert torch.equal(q.dequant_all(dt).cpu(), want.to(dt))
