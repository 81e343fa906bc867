"""Host test: the row width and stride that a KV store is launched with, read off the shape, equal those of the view they replace, and what
the view refuses is still refused."""
import pytest
import torch

from sglang_amd.kernels import _row_width


@pytest.mark.parametrize("size,stride", [((5, 4, 64), (256, 64, 1)), ((5, 4, 64), (1024, 64, 1)), ((1, 4, 64), (1024, 64, 1)), ((5, 1, 64), (96, 80, 1)),
                                         ((5, 4, 1), (8, 1, 3)), ((5, 256), (512, 1)), ((5, 4, 64), (0, 64, 1)), ((2, 3, 4, 8), (96, 32, 8, 1))])
def test_row_width_is_that_of_the_view(size, stride):
    x = torch.empty(5000).as_strided(size, stride)
    v = x.view(size[0], -1)
    assert _row_width(x, size[0]) == (v.shape[1], v.stride(0))


@pytest.mark.parametrize("size,stride,n", [((5, 4, 64), (512, 128, 1), 5), ((5, 4, 64), (64, 320, 1), 5), ((0, 4, 64), (256, 64, 1), 0), ((5, 4, 64), (256, 64, 1), 6)])
def test_what_the_view_refuses_is_refused(size, stride, n):
    x = torch.empty(5000).as_strided(size, stride)
    with pytest.raises(RuntimeError):
        x.view(n, -1)
    with pytest.raises(RuntimeError):
        _row_width(x, n)
