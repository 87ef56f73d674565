"""Which images are uploaded with their stride: those whose rows lie within the
device's room; a stride for which (height - 1) * stride wraps does not."""
import ctypes

import pytest

from tests import oracle_lib


@pytest.mark.parametrize("capacity,w,h,stride,fits", [
    (64 * 48, 64, 48, 64, 1), (64 * 48, 64, 48, 65, 0), (64 * 48 + 47, 64, 48, 65, 1),
    (64 * 48 + 46, 64, 48, 65, 0), (64, 64, 1, 1 << 40, 1),
    (1920 * 1088, 64, 3, 1 << 63, 0), (1920 * 1088, 64, 5, 1 << 62, 0),
    (1920 * 1088, 64, 48, 2**64 - 64, 0), (1920 * 1088, 64, 16, (2**64 - 1) // 15, 0)])
def test_rows_fit(capacity, w, h, stride, fits):
    f = oracle_lib.load().oracle_rows_fit
    f.argtypes = [ctypes.c_size_t] * 4
    assert f(capacity, w, h, stride) == fits
    if stride < 1 << 40:
        assert fits == ((h - 1) * stride + w <= capacity)
