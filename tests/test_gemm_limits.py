"""The packed GEMMs refuse, before any launch, a K whose weight offsets would not fit 32 bits."""
import ctypes

import pytest

from estudiocanciones_amd import _ffi

ENOTSUP = -95


def fake():
    buf = ctypes.create_string_buffer(64)
    return buf, (ctypes.addressof(buf) + 15) & ~15


@pytest.mark.parametrize("K", [2 ** 26, 2 ** 28])
def test_weight_offsets_are_checked(K):
    buf, p = fake()
    lib = _ffi.lib()
    assert lib.ecd_gemm_f16p_tuned(p, K, p, None, 1.0, None, 0, p, 64, 1, 64, K, 0, 0, None) == ENOTSUP
    assert lib.ecd_gemm_i8p(p, K, p, p, None, 0, p, 64, 1, 64, K, None) == ENOTSUP
    assert lib.ecd_gemm_f16p_partial(p, K, p, p, 1, 64, K, 2, None) == ENOTSUP
    assert lib.ecd_gemm_i8p_partial(p, K, p, p, p, 1, 64, K, 2, None) == ENOTSUP
    del buf


def test_wide_tiles_are_refused_before_narrow_ones():
    buf, p = fake()
    K = 2 ** 24  # 256 features of it pass 4 GiB
    assert _ffi.lib().ecd_gemm_f16p_tuned(p, K, p, None, 1.0, None, 0, p, 64, 1, 64, K, 0, 1, None) == ENOTSUP
    del buf
