"""Rows of codes that do not fill their last word, and code buffers off a 16-byte boundary, through the C ABI: the kernels load and
store up to 16 codes wherever they begin, across the ends of rows.  Words and codes against the oracle's, nothing written around them."""
import pytest
import torch

import varq_oracle as O
from gpu_util import note

pytestmark = pytest.mark.gpu

GUARD = 48


@pytest.mark.parametrize('bits', [2, 4, 8])
@pytest.mark.parametrize('rows', [1, 2, 41, 3001])
@pytest.mark.parametrize('c', [1, 2, 3, 7, 15, 16, 17, 31, 33, 100, 145, 255])
@pytest.mark.parametrize('code_offset,word_offset', [(0, 0), (5, 1)])
def test_ragged_rows(dev, bits, rows, c, code_offset, word_offset):
    from var_q_amd import _lib
    note('ragged rows', bits, rows, c, code_offset, word_offset)
    lib, st = _lib.load(), torch.cuda.current_stream().cuda_stream
    lo, hi = O.qrange(bits)
    q = torch.randint(lo, hi + 1, (rows, c), generator=torch.Generator().manual_seed(bits + rows + c), dtype=torch.int8)
    want, _ = O.pack_last_dim(q, bits)
    buf = torch.full((rows * c + 2 * GUARD,), 99, dtype=torch.int8)
    buf[GUARD + code_offset:][:rows * c] = q.flatten()
    buf = buf.to(dev)
    out = torch.full((want.numel() + 2 * GUARD,), 0x5a5a5a5a, dtype=torch.int32, device=dev)
    words = out[GUARD + word_offset:][:want.numel()]
    _lib.check(lib.varq_pack(buf[GUARD + code_offset:].data_ptr(), rows, c, bits, words.data_ptr(), st), 'varq_pack')
    torch.cuda.synchronize()
    assert torch.equal(words.cpu().view(want.shape), want)
    words.fill_(0x5a5a5a5a)
    assert bool((out == 0x5a5a5a5a).all()), 'wrote around its words'
    words.copy_(want.flatten())
    codes = buf[GUARD + code_offset:][:rows * c]
    codes.fill_(99)
    _lib.check(lib.varq_unpack(words.data_ptr(), rows, c, bits, codes.data_ptr(), st), 'varq_unpack')
    torch.cuda.synchronize()
    assert torch.equal(codes.cpu().view(rows, c), q)
    codes.fill_(99)
    assert bool((buf == 99).all()), 'wrote around its codes'
