"""Bit-widths and row lengths that do not fit each other are errors of the host layer: the kernels take rows to be as long as
the channel count says."""
import pytest
import torch

from gpu_util import note
from var_q_amd import ops
from var_q_amd._lib import VarqError

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('bits', [0, -4, 1, 3, 16, 33, 64])
def test_bits_of_pack_and_unpack(dev, bits):
    note('bits', bits)
    for call in (lambda: ops.pack(torch.zeros(3, 32, dtype=torch.int8, device=dev), bits),
                 lambda: ops.unpack(torch.zeros(3, 4, dtype=torch.int32, device=dev), 32, bits),
                 lambda: ops.dequant(torch.zeros(1, 1, 3, 4, dtype=torch.int32, device=dev), torch.ones(1, 1, 1, 1, device=dev), None, 32, bits)):
        with pytest.raises((AssertionError, VarqError)):
            call()


@pytest.mark.parametrize('c', [1, 24, 25, 33, 40, 4096])
def test_channels_that_the_rows_do_not_hold(dev, c):
    note('row length', c)
    words, codes = torch.zeros(2, 3, 5, 4, dtype=torch.int32, device=dev), torch.zeros(2, 3, 5, 32, dtype=torch.int8, device=dev)
    one = torch.ones(1, 1, 1, 1, device=dev)
    calls = [lambda: ops.dequant(codes, one, None, c, 8)]
    if (c + 7) // 8 != 4:
        calls += [lambda: ops.unpack(words, c, 4), lambda: ops.dequant(words, one, None, c, 4), lambda: ops.dequant(words[:, :, 1:3], one, None, c, 4)]
    for call in calls:
        with pytest.raises((AssertionError, VarqError)):
            call()
    assert ops.unpack(words, 29, 4).shape == (2, 3, 5, 29) and ops.dequant(words, one, None, 29, 4).shape == (2, 3, 5, 29)
