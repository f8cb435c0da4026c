"""A step through use_var_q whose result cannot be made (no room for it, or more tokens than the launch behind it counts) is not in the cache
afterwards, so that a caller who tries again does not append it twice."""
import pytest
import torch

from gpu_util import note
from var_q_amd import VAR_Q
from var_q_amd._lib import VarqError

pytestmark = pytest.mark.gpu


def _state(z):
    return z._c_item.len, z._tok_scale.len, list(z._seg_ends), z.cached_item.shape, z.cached_scale.shape


@pytest.mark.parametrize('method', ['G_TOKEN', 'G_TOKEN_HEAD'])
def test_more_tokens_than_the_grid(dev, method):
    note('use_var_q beyond the grid', method)
    z = VAR_Q(8, 'BLHc', method)
    z.reserve_tokens(65600)
    z.use_var_q(torch.randn(1, 65530, 1, 8, device=dev))
    before = _state(z)
    with pytest.raises(VarqError):
        z.use_var_q(torch.randn(1, 6, 1, 8, device=dev))
    assert _state(z) == before
    assert z.use_var_q(torch.randn(1, 5, 1, 8, device=dev)).shape == (1, 65535, 1, 8)


@pytest.mark.parametrize('method', ['G_SCALE_HEAD_DIM', 'G_SCALE', 'G_HEAD', 'G_TOKEN', 'G_TOKEN_HEAD'])
@pytest.mark.parametrize('layout', ['BLHc', 'BHLc'])
def test_no_room_for_the_result(dev, method, layout):
    note('use_var_q without room', method, layout)
    shape = lambda n: (4, n, 16, 128) if layout == 'BLHc' else (4, 16, n, 128)
    z = VAR_Q(2, layout, method)
    z.reserve_tokens(8193)
    z.use_var_q(torch.randn(shape(1), device=dev).half())
    x = torch.randn(shape(8192), device=dev).half()     # 268 MB of result, 17 MB of codes that are there
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    before, total = _state(z), torch.cuda.get_device_properties(dev).total_memory
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + 100e6) / total, dev)
    held = []
    try:
        with pytest.raises(torch.OutOfMemoryError):     # (what other tests have left of their allocations is taken)
            while True:
                held.append(torch.empty(64 << 20, dtype=torch.uint8, device=dev))
        with pytest.raises(torch.OutOfMemoryError):
            z.use_var_q(x)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0, dev)
    del held
    assert _state(z) == before
    assert z.use_var_q(x).shape == shape(8193)
