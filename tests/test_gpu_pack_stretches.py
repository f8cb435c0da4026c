"""Rows of codes that do not fill their last word, in several launches (as tensors of 2^31 codes and more are), and both ways to unpack them:
16 codes per thread and a word per thread.  Words and codes against the oracle's, nothing written around them."""
import pytest
import torch

import varq_oracle as O
from gpu_util import note

pytestmark = pytest.mark.gpu

GUARD = 48


@pytest.mark.parametrize('bits', [2, 4, 8])
@pytest.mark.parametrize('c', [1, 3, 14, 15, 17, 31, 33, 100, 255])
@pytest.mark.parametrize('rows,in_one', [(7, 7), (7, 3), (300, 100), (300, 299), (300, 1), (1501, 1501)])
@pytest.mark.parametrize('code_offset', [0, 5])
def test_stretches(dev, bits, c, rows, in_one, code_offset):
    from var_q_amd import _lib
    note('packing in stretches', bits, c, rows, in_one, code_offset)
    lib, st = _lib.load(), torch.cuda.current_stream().cuda_stream
    lo, hi = O.qrange(bits)
    q = torch.randint(lo, hi + 1, (rows, c), generator=torch.Generator().manual_seed(bits + rows + c), dtype=torch.int8)
    want, _ = O.pack_last_dim(q, bits)
    stretch = in_one * want.shape[1] * (32 // bits)
    buf = torch.full((rows * c + 2 * GUARD,), 99, dtype=torch.int8, device=dev)
    codes = buf[GUARD + code_offset:][:rows * c]
    codes.copy_(q.flatten())
    out = torch.full((want.numel() + 2 * GUARD,), 0x5a5a5a5a, dtype=torch.int32, device=dev)
    words = out[GUARD:][:want.numel()]
    _lib.check(lib.varq_pack_stretches(codes.data_ptr(), rows, c, bits, words.data_ptr(), stretch, st), 'varq_pack_stretches')
    torch.cuda.synchronize()
    assert torch.equal(words.cpu().view(want.shape), want)
    for by_pieces in (1, 0, -1):
        codes.fill_(99)
        _lib.check(lib.varq_unpack_stretches(words.data_ptr(), rows, c, bits, codes.data_ptr(), stretch, by_pieces, st), 'varq_unpack_stretches')
        torch.cuda.synchronize()
        assert torch.equal(codes.cpu().view(rows, c), q), by_pieces
    codes.fill_(99)
    words.fill_(0x5a5a5a5a)
    assert bool((buf == 99).all()) and bool((out == 0x5a5a5a5a).all()), 'wrote around its codes or words'
