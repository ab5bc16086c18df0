"""K so large that the weights of one tile pass 4 GiB: the GEMMs take it, the split products leave it to them."""
import ctypes

import pytest

from estudiocanciones_amd import _ffi

ENOTSUP = -95


def fake():
    buf = ctypes.create_string_buffer(64)
    return buf, (ctypes.addressof(buf) + 15) & ~15


@pytest.mark.parametrize("K", [2 ** 25, 2 ** 26, 2 ** 28])
def test_split_products_refuse_before_any_launch(K):
    buf, p = fake()
    lib = _ffi.lib()
    assert lib.ecd_gemm_f16p_splits(1, 64, K) == 1 and lib.ecd_gemm_i8p_splits(1, 64, K) == 1
    assert lib.ecd_gemm_f16p_partial(p, K, p, p, 1, 64, K, 2, None) == ENOTSUP
    assert lib.ecd_gemm_i8p_partial(p, K, p, p, p, 1, 64, K, 2, None) == ENOTSUP
    del buf


# rows 48 .. 63 of the weights lie past 4 GiB from the first (fp16 6.4 GB of weights in all, int8 6.4 GB).  x is zero
# but for a few values at both ends of K, so the product is a few exact terms.
@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["f16", "f16_wide_tile", "f16_below", "i8", "i8_rowmajor"])
def test_weights_past_4_gib(kind):
    import torch
    from estudiocanciones_amd.kernels import gemm_f16_packed, gemm_packed, pack_f16, pack_i8, stream_ptr
    dev = torch.device("cuda:0")
    f16 = kind.startswith("f16")
    # the row-major product reads 16 rows from one base below 2 GiB (beyond, its own path): 64 of them pass 4 GiB too
    # f16_below: the largest offsets lie between 2 and 4 GiB, the ordinary 64-feature tiles
    K = 29 * 2 ** 20 if kind == "f16_below" else 3 * 2 ** 24 if f16 else 2 ** 27 - 64 if kind == "i8_rowmajor" else 3 * 2 ** 25
    M, N = (17 if kind == "i8_rowmajor" else 2), 66
    M = min(M, (2 ** 31 - 1) // (2 * K))
    at = [0, 5, 63, 64, K // 2, K - 65, K - 1]
    g = torch.Generator().manual_seed(3)
    x = torch.zeros(M, K, device=dev, dtype=torch.float16)
    x[:, at] = torch.randint(-3, 4, (M, len(at)), generator=g).half().to(dev)
    w = torch.zeros(N, K, device=dev, dtype=torch.float16 if f16 else torch.int8)
    cols = torch.randint(-9, 10, (N, len(at)), generator=g)
    w[:, at] = cols.to(device=dev, dtype=w.dtype)
    want = x[:, at].double().cpu() @ cols.double().t()
    s = torch.ones(N, device=dev, dtype=torch.float16)
    if f16:
        wp = pack_f16(w)
        del w
        if kind != "f16_wide_tile":
            y = gemm_f16_packed(x, wp, N, K)
        else:
            y = torch.empty(M, N, device=dev, dtype=torch.float16)
            _ffi.call("ecd_gemm_f16p_tuned", x.data_ptr(), K, wp.data_ptr(), None, 1.0, None, 0, y.data_ptr(), N, M, N, K,
                      0, 1, stream_ptr(dev))
    elif kind == "i8":
        wp = pack_i8(w)
        del w
        y = gemm_packed(x, wp, s, N, K)
    else:
        y = torch.empty(M, N, device=dev, dtype=torch.float16)
        _ffi.call("ecd_gemm_i8p_tuned", x.data_ptr(), K, w.data_ptr(), s.data_ptr(), None, 0, y.data_ptr(), N, M, N, K, 1, 0,
                  stream_ptr(dev))
    assert torch.equal(y.double().cpu(), want)
