"""Dequantizing packed words through the kernel for whole octets, and through the general one where it does not apply: groups, tables per channel
that the tokens share and that they do not, rows of any number of octets, the ends of tiles, windows of a buffer.  Bit for bit (q - zp) * scale in fp32."""
import pytest
import torch

import varq_oracle as O
from gpu_util import note

pytestmark = pytest.mark.gpu

DTYPES = (torch.float32, torch.bfloat16, torch.float16)


def _codes(shape, bits, seed):
    lo, hi = O.qrange(bits)
    return torch.randint(lo, hi + 1, shape, generator=torch.Generator().manual_seed(seed), dtype=torch.int8)


def _values(q, scale, zp, dt):
    g = q.shape[-1] // scale.shape[-1]
    s, z = scale.repeat_interleave(g, -1), None if zp is None else zp.repeat_interleave(g, -1)
    return ((q.float() if z is None else q.float() - z) * s).to(dt)


@pytest.mark.parametrize('bits', [2, 4, 8])
@pytest.mark.parametrize('n,c', [(1, 8), (127, 8), (129, 16), (513, 40), (85, 72), (33, 96), (65, 128), (3, 264), (1, 2048)])
@pytest.mark.parametrize('kind', ['row', 'groups', 'shared_table', 'token_table', 'head_table'])
@pytest.mark.parametrize('affine', [True, False])
def test_words(dev, bits, n, c, kind, affine):
    from var_q_amd import ops
    note('words', bits, n, c, kind, affine)
    q = _codes((2, 3, n, c), bits, n + c)
    words, _ = O.pack_last_dim(q, bits)
    shape = {'row': (2, 3, n, 1), 'groups': (2, 3, n, c // 8), 'shared_table': (1, 3, 1, c), 'token_table': (1, 1, n, c), 'head_table': (2, 1, n, c)}[kind]
    g = torch.Generator().manual_seed(c)
    scale = torch.rand(shape, generator=g) + 0.1
    zp = torch.randint(-200, 200, shape, generator=g).float() if affine else None
    for dt in DTYPES:
        got = ops.dequant(words.to(dev), scale.to(dev), None if zp is None else zp.to(dev), c, bits, dt)
        assert torch.equal(got.cpu(), _values(q, scale, zp, dt))


@pytest.mark.parametrize('bits', [2, 4, 8])
@pytest.mark.parametrize('tokens_first', [True, False])
@pytest.mark.parametrize('word_offset,scale_offset', [(0, 0), (1, 0), (0, 1)])      # (off the alignment that the loads want: the general kernel)
def test_window(dev, bits, tokens_first, word_offset, scale_offset):
    """Tokens 5 to 42 of a buffer of 50, one scale per (head, channel)."""
    from var_q_amd import ops
    note('window', bits, tokens_first, word_offset, scale_offset)
    B, H, cap, n, c = 2, 5, 50, 37, 48
    q = _codes((B, cap, H, c) if tokens_first else (B, H, cap, c), bits, 7)
    words, _ = O.pack_last_dim(q, bits)
    buf = torch.zeros(words.numel() + 1, dtype=torch.int32)
    buf[word_offset:][:words.numel()] = words.flatten()
    buf, scale = buf.to(dev), torch.rand(H * c + 1) + 0.1
    table = scale[scale_offset:][:H * c]
    if tokens_first:
        shape, strides, rowmap, window, s = [B, n, H, c], [0, 0, c, 1], [B, n, H, cap * H, H, 1, 5 * H, -1], q[:, 5:5 + n], table.view(1, 1, H, c)
    else:
        shape, strides, rowmap, window, s = [B, H, n, c], [0, c, 0, 1], [B, H, n, H * cap, cap, 1, 5, -1], q[:, :, 5:5 + n], table.view(1, H, 1, c)
    on_gpu = scale.to(dev)[scale_offset:]
    for dt in DTYPES:
        got = ops.dequant_window(buf[word_offset:], on_gpu, None, shape, strides, 1, bits, rowmap, dt)
        assert torch.equal(got.cpu(), _values(window, s.expand(1, *s.shape[1:]), None, dt))


@pytest.mark.parametrize('dt', DTYPES)
def test_past_the_caches(dev, dt):
    """An output that does not fit the Infinity Cache, and one of a piece less."""
    from var_q_amd import ops
    note('past the caches', dt)
    c, rows = 128, (240 << 20) // (128 * (4 if dt == torch.float32 else 2))
    words = torch.randint(-2 ** 31, 2 ** 31, (1, 2, rows // 2, c // 8), device=dev, dtype=torch.int64).to(torch.int32)
    scale = torch.rand((1, 2, rows // 2, 1), device=dev) + 0.1
    nibble = torch.arange(0, 32, 4, device=dev, dtype=torch.int32)
    for n in (rows // 2, rows // 2 - 1):
        w, s = words[:, :, :n].contiguous(), scale[:, :, :n].contiguous()
        q = ((w.unsqueeze(-1) >> nibble & 15) ^ 8) - 8
        assert torch.equal(ops.dequant(w, s, None, c, 4, dt), (q.view(1, 2, n, c).float() * s).to(dt))


@pytest.mark.parametrize('bits', [2, 4, 8])
@pytest.mark.parametrize('n,c', [(1, 8), (63, 8), (64, 8), (127, 8), (128, 8), (255, 8), (256, 8), (257, 8), (30, 64), (16, 128)])
@pytest.mark.parametrize('kind', ['row', 'shared_table', 'token_table'])
def test_pairs_of_one_workgroup(dev, bits, n, c, kind):
    """Pairs of up to 256 pieces of 16 bytes (an octet in 16 bits, half of one in 32), one per lane, and just more."""
    from var_q_amd import ops
    note('pairs of one workgroup', bits, n, c, kind)
    q = _codes((5, 7, n, c), bits, n + c)
    words, _ = O.pack_last_dim(q, bits)
    shape = {'row': (5, 7, n, 1), 'shared_table': (1, 7, 1, c), 'token_table': (1, 1, n, c)}[kind]
    g = torch.Generator().manual_seed(c)
    scale, zp = torch.rand(shape, generator=g) + 0.1, torch.randint(-200, 200, shape, generator=g).float()
    for dt in DTYPES:
        got = ops.dequant(words.to(dev), scale.to(dev), zp.to(dev), c, bits, dt)
        assert torch.equal(got.cpu(), _values(q, scale, zp, dt))


@pytest.mark.parametrize('octets', [2047, 2048, 2049, 3070, 3072, 4096, 4100])
@pytest.mark.parametrize('c', [96, 100])
def test_general_kernel_octets_of_a_lane(dev, octets, c):
    """One, two and four octets of a lane one after the other: int8 codes, and packed rows that are no whole octets."""
    from var_q_amd import ops
    note('general dequantizing', octets, c)
    n = -(-octets // (-(-c // 8)))
    q = _codes((2, 3, n, c), 4, octets)
    g = torch.Generator().manual_seed(octets)
    scale, zp = torch.rand((2, 3, n, 1), generator=g) + 0.1, torch.randint(-20, 20, (2, 3, n, 1), generator=g).float()
    for codes in ([q] if c == 96 else [q, O.pack_last_dim(q, 4)[0]]):
        for dt in DTYPES:
            assert torch.equal(ops.dequant(codes.to(dev), scale.to(dev), zp.to(dev), c, 4, dt).cpu(), _values(q, scale, zp, dt))
