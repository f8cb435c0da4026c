"""A quantizer whose cache grows on another stream than the one its buffers were made on: the copy into the new buffer may still wait
on that stream when the old one is let go of, so its memory must not be handed out to the first stream before."""
import pytest
import torch

from gpu_util import note
from var_q_amd import VAR_Q

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('method', ['G_SCALE_HEAD_DIM', 'G_TOKEN', 'G_HEAD_DIM'])
def test_the_old_buffer_waits_for_the_copy(dev, method):
    note('growing on another stream', method)
    gen = torch.Generator(device=dev).manual_seed(1)
    steps = [torch.randn(2, 4, n, 64, device=dev, generator=gen) for n in (50, 70)]
    want, z, side = VAR_Q(8, 'BHLc', method), VAR_Q(8, 'BHLc', method), torch.cuda.Stream()
    for x in steps:
        want.quant(x)
        want.cache()
    z.quant(steps[0])
    z.cache()
    torch.cuda.synchronize()
    old, like = z._c_item.buf.data_ptr(), z._c_item.buf.shape
    busy = torch.cuda.Event()
    with torch.cuda.stream(side):
        torch.cuda._sleep(100_000_000)      # (some 50 ms, in front of the copy)
        z.quant(steps[1])
        z.cache()
        busy.record()
    fresh = [torch.zeros(like, dtype=torch.int32, device=dev) for _ in range(32)]
    assert not busy.query(), 'the side stream was done before anything could be seen'
    assert all(t.data_ptr() != old for t in fresh)
    torch.cuda.synchronize()
    assert torch.equal(z.cached_item, want.cached_item) and torch.equal(z.dequant_all(), want.dequant_all())
