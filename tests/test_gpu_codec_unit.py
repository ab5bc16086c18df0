"""The waveform decoder's one-pass stages against the separate convolutions they replace."""
import ctypes

import numpy as np
import pytest

from helpers import randn16, rng
from oracle.numerics import f16

pytestmark = pytest.mark.gpu
P = 60


@pytest.fixture(scope="module")
def dev():
    import torch
    return torch.device("cuda:0")


def _conv(dev, N, k, seed, C=64):
    import torch
    from estudiocanciones_amd.kernels import pack_f16
    g = rng(seed)
    w = f16(g.standard_normal((N, k * C)) * (k * C) ** -0.5)
    b = (g.standard_normal(N) * 0.1).astype(np.float32)
    return pack_f16(torch.from_numpy(w).to(dev)), torch.from_numpy(b).to(dev), w, b


def _padded(dev, S, T, seed):
    import torch
    x = np.zeros((S * (P + T) + 8, 64), np.float16)
    for b in range(S):
        x[b * (P + T) + P:(b + 1) * (P + T)] = randn16(seed + b, T, 64)
    return torch.from_numpy(x).to(dev)


# one row; one short of, at and past one and two tiles of 128 rows; then more than two tiles for each of the 512 workgroups
# (two on each of 256 CUs), so that a window buffer is loaded again behind the counted wait for stores: 626 tiles (a second tile
# for some), 1094 with partial last tiles and 2200 with full ones (a third and a fifth for some, the last tile 32 rows or 128)
@pytest.mark.parametrize("S,T,dil", [(1, 1, 9), (2, 127, 1), (2, 128, 3), (3, 129, 5), (2, 255, 2), (1, 256, 4), (2, 257, 6),
                                     (2, 700, 10), (2, 40000, 7), (2, 70000, 1), (2, 140800, 10)])
def test_unit64_equals_two_convs(dev, S, T, dil):
    import torch
    from estudiocanciones_amd import _ffi
    from estudiocanciones_amd.kernels import stream_ptr
    st = stream_ptr(dev)
    (w1, b1, *_), (w2, b2, *_) = _conv(dev, 64, 7, 1), _conv(dev, 64, 1, 2)
    x = _padded(dev, S, T, 10)
    off, zero = (ctypes.c_int * 7)(*[(j - 6) * dil for j in range(7)]), (ctypes.c_int * 1)(0)
    h, want, got = torch.empty(S * T, 64, device=dev, dtype=torch.float16), x.clone(), torch.zeros_like(x)
    _ffi.call("ecd_gemm_f16p_conv", x.data_ptr(), 64, w1.data_ptr(), b1.data_ptr(), 0.25, None, 0, h.data_ptr(), 64,
              S * T, 64, 448, T, P, -1, off, 7, 1, 2, st)
    _ffi.call("ecd_gemm_f16p_conv", h.data_ptr(), 64, w2.data_ptr(), b2.data_ptr(), 0.125, want.data_ptr(), 64,
              want.data_ptr(), 64, S * T, 64, 64, T, 0, P, zero, 0, 1, 2, st)
    _ffi.call("ecd_codec_unit64", x.data_ptr(), got.data_ptr(), w1.data_ptr(), b1.data_ptr(), 0.25, w2.data_ptr(),
              b2.data_ptr(), 0.125, S, T, P, dil, st)
    assert torch.equal(got, want)  # every row, the zero pad rows among them


# one source row; one short of, at and past one and two tiles of 61 source rows; 656 tiles (a second for some of the
# 512 workgroups), then third tiles (1082, the last partial) and fifth ones (2200, all full)
@pytest.mark.parametrize("S,T", [(1, 1), (2, 3), (2, 60), (2, 61), (1, 62), (3, 121), (2, 122), (3, 123), (2, 1000),
                                 (2, 20000), (2, 33000), (2, 67100)])
def test_post_final_equals_two_convs(dev, S, T):
    """The wide conv's samples are the same bits; the final conv sums its 7 taps' fp32 products in another order,
    so it is held to float64 over those fp16 samples: 448 products and the bias summed in fp32, each addition within
    2^-24 of a partial sum no larger than sum |u w| + |b|, and one fp16 rounding (2^-11 relative, 2^-25 below the normal
    numbers)."""
    import torch
    from estudiocanciones_amd import _ffi
    from estudiocanciones_amd.kernels import stream_ptr
    st = stream_ptr(dev)
    w1, b1, *_ = _conv(dev, 64, 7, 3)
    wf, bf, wn, bn = _conv(dev, 1, 7, 4)
    x = _padded(dev, S, T, 20)
    off = (ctypes.c_int * 7)(*range(-6, 1))
    u = torch.empty(S * 2 * T, 64, device=dev, dtype=torch.float16)
    _ffi.call("ecd_gemm_f16p_conv", x.data_ptr(), 64, w1.data_ptr(), b1.data_ptr(), 0.25, None, 0, u.data_ptr(), 64,
              S * 2 * T, 64, 448, 2 * T, P, -1, off, 7, 2, 2, st)
    y = torch.empty(S, 2 * T, device=dev, dtype=torch.float16)
    _ffi.call("ecd_codec_post_final", x.data_ptr(), w1.data_ptr(), b1.data_ptr(), 0.25, wf.data_ptr(), bf.data_ptr(),
              y.data_ptr(), S, T, P, st)
    up = torch.nn.functional.pad(u.double().view(S, 2 * T, 64), (0, 0, 6, 0)).cpu()
    w64 = torch.from_numpy(wn).double().view(7, 64)
    want = sum(up[:, j:j + 2 * T] @ w64[j] for j in range(7)) + float(bn[0])
    mag = sum(up[:, j:j + 2 * T].abs() @ w64[j].abs() for j in range(7)) + abs(float(bn[0]))
    err = (y.double().cpu() - want).abs()
    assert bool((err <= 1.001 * (want.abs() * 2.0 ** -11 + 2.0 ** -25 + 449 * 2.0 ** -24 * mag)).all()), float(err.max())


def test_unit64_refuses_what_it_does_not_take(dev):
    import torch
    from estudiocanciones_amd import _ffi
    t = torch.zeros(4096, device=dev, dtype=torch.float16)
    f = torch.zeros(64, device=dev)
    a = lambda x, y, pad, dil: _ffi.lib().ecd_codec_unit64(
        x.data_ptr(), y.data_ptr(), t.data_ptr(), f.data_ptr(), 0.1, t.data_ptr(), f.data_ptr(), 0.1, 1, 4, pad, dil, None)
    assert a(t, t, 60, 1) == _ffi.ECD_EINVAL          # in place
    assert a(t, t[64:], 60, 11) == _ffi.ECD_EINVAL    # reach past the padding
    assert a(t, t[64:], 5, 1) == _ffi.ECD_EINVAL
