"""The quantizer's one-launch kernel at the edges of its plans: one row per group, row counts around a
workgroup's row lanes and its 16 (fp32: 8) register steps, the row count from which the three launches
take over, column slices with a remainder (an octet count that is no power of two), kept inner indices
that do not fill the last tile.  Bit-exact against the CPU oracle."""
import pytest
import torch

import varq_oracle as O
from gpu_util import note
from var_q_amd import VAR_Q, ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('shape,dims,dtype', [
    ((3, 1, 5, 64), (1,), torch.bfloat16),            # every row its own group, channel by channel
    ((2, 16, 1, 128), (0, 2), torch.float16),         # two rows per group
    ((2, 1, 33, 16), (2,), torch.bfloat16),           # one octet pair, 33 rows
    ((1, 3, 511, 8), (2,), torch.float32),            # one octet
    ((1, 3, 513, 72), (2,), torch.bfloat16),          # nine octets: a slice with one live lane
    ((2, 4, 1025, 128), (0, 2), torch.bfloat16),
    ((64, 3, 16, 64), (0, 1), torch.float16),         # strided rows, inner index kept
    ((64, 33, 3, 48), (0, 1), torch.float32),
    ((1, 4096, 2, 64), (0, 1), torch.bfloat16),
    ((1, 8192, 2, 32), (0, 1), torch.float16),        # the most rows of a group
    ((1, 8193, 2, 32), (0, 1), torch.float16),        # one row more
    ((1, 4, 2047, 512), (2,), torch.float32),
    ((7, 5, 3, 64), (0, 3), torch.bfloat16),          # channel dim reduced: one scale per kept index
    ((2, 40, 65, 80), (0, 1, 3), torch.float32),
    ((2, 3, 129, 520), (0, 2), torch.bfloat16),       # 65 octets: past the column lanes
])
def test_one_launch_edges(dev, shape, dims, dtype):
    g = torch.Generator().manual_seed(sum(shape))
    x = (torch.randn(*shape, generator=g) * 2).to(dtype)
    x[..., 3] *= 15
    x[0, 0, 0] = 0
    for bits, asym, pack in ((8, False, True), (4, True, True), (2, True, True), (5, False, False)):
        if pack and (shape[-1] * bits) % 32:
            continue
        note('quant one', shape, dims, dtype, bits, asym, pack)
        q, s, z = O.quant_reduce(x, dims, bits, asym)
        gq, gs, gz = ops.quant_pack(x.to(dev), dims, bits, asym=asym, pack=pack)
        torch.cuda.synchronize()
        assert torch.equal(gs.cpu(), s)
        assert not asym or torch.equal(gz.cpu(), z)
        assert torch.equal(gq.cpu(), O.pack_last_dim(q, bits)[0] if pack else q)


@pytest.mark.parametrize('shape,dims,dtype', [
    ((3, 700, 5, 64), (0, 1), torch.float16),         # 2100 rows per group, few heads: slices of one octet
    ((3, 700, 5, 72), (0, 1), torch.bfloat16),        # nine octets
    ((1, 3, 4097, 24), (0, 2), torch.float32),
    ((2, 2, 2500, 8), (0, 2), torch.bfloat16),        # nothing to slice
    ((64, 30, 4, 128), (0, 1), torch.float16),
])
def test_narrow_slices(dev, shape, dims, dtype):
    """Few workgroups' worth of columns: 8- and 4-bit codes in slices of one octet, 2-bit codes (two octets to a word)
    in slices of two, and K and V of a step together, which are enough for wider slices."""
    test_one_launch_edges(dev, shape, dims, dtype)
    g = torch.Generator().manual_seed(1)
    xs = [torch.randn(*shape, generator=g).to(dtype) for _ in range(2)]
    for bits in (8, 4, 2):
        if shape[3] * bits % 32:
            continue
        pair = [VAR_Q(bits, 'BLHc' if dims == (0, 1) else 'BHLc') for _ in xs]
        note('quant one, two tensors', shape, dims, dtype, bits)
        assert VAR_Q._step_fast_pair(*pair, *[x.to(dev) for x in xs])
        for x, z in zip(xs, pair):
            q, s, _ = O.quant_reduce(x, dims, bits, False)
            assert torch.equal(z.cached_item.cpu(), O.pack_last_dim(q, bits)[0]) and torch.equal(z.scale.cpu(), s)


@pytest.mark.parametrize('shape,dims,dtype', [
    ((8, 30, 1024, 64), (0, 2), torch.bfloat16),      # two tensors: 60 MiB, all 16 register steps
    ((8, 400, 16, 128), (0, 1), torch.float16),       # two tensors: 25 MiB, one: 16-byte pieces
    ((3, 24, 701, 128), (0, 2), torch.bfloat16),
    ((5, 20, 333, 72), (0, 2), torch.float32),        # nine octets of sixteen lanes
    ((6, 30, 1024, 128), (0, 2), torch.float32),      # 90 MiB, behind itself 180: fewer workgroups per compute unit in the second pass
    ((24, 6, 171, 64), (0, 2), torch.float16),        # few heads: one tensor is left to the three launches
    ((32, 30, 201, 64), (0, 3), torch.bfloat16),      # groups of whole rows: 24 MiB of one tensor, 47 of two
])
def test_sizes_where_one_launch_takes_over(dev, shape, dims, dtype):
    """The same groups with the batch behind itself until they are too long for one launch, or the tensor too large: max and min,
    scales, zero-points and codes are those of the three launches bit for bit, whichever way the call itself goes."""
    gen = torch.Generator(device=dev).manual_seed(shape[2])
    xs = [(torch.randn(*shape, generator=gen, device=dev) * 2).to(dtype) for _ in range(2)]
    xs[0][..., 3] *= 15
    xs[1][:, :, 0] = 0
    rows = xs[0].numel() // shape[3] // (1 if 3 in dims else shape[1] if dims == (0, 2) else shape[2])
    times = 8192 // rows + 1 if 3 not in dims else (128 << 20) // (xs[0].numel() * xs[0].element_size()) + 1
    for bits, asym in ((8, False), (4, True), (2, False)):
        note('quant one, sizes', shape, dims, dtype, bits, asym)
        pair = ops.quant_pack_pair(*xs, dims, bits, asym)
        for x, two in zip(xs, pair):
            q, s, z = ops.quant_pack(x.repeat(times, 1, 1, 1), dims, bits, asym=asym)
            for got in (two, ops.quant_pack(x, dims, bits, asym=asym)):
                assert torch.equal(got[0], q[:shape[0]]) and torch.equal(got[1], s) and (not asym or torch.equal(got[2], z))
