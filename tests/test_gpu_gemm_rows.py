"""GEMM outputs and residuals in rows of any alignment: the same bits as in 16-byte aligned rows, and nothing
written between the rows."""
import pytest
import torch

from estudiocanciones_amd import _ffi
from estudiocanciones_amd.kernels import pack_f16, pack_i8, stream_ptr

pytestmark = pytest.mark.gpu
FILL = 7.0


def rows(M, N, ld, lead, data=None):
    """[M, N] view of a buffer with row stride ld that starts ``lead`` elements past a 16-byte boundary."""
    buf = torch.full((lead + M * ld + 16,), FILL, device="cuda", dtype=torch.float16)
    view = buf[lead:lead + M * ld].view(M, ld)[:, :N]
    if data is not None:
        view.copy_(data)
    return buf, view


def gaps_kept(buf, view, lead, ld):
    M, N = view.shape
    return bool((buf[lead:lead + M * ld].view(M, ld)[:, N:] == FILL).all() and (buf[:lead] == FILL).all()
                and (buf[lead + M * ld:] == FILL).all())


# N: whole pieces of 8 features; tails of 4 + 2 + 1, 4, 1; one feature.  Row strides and starts: 8-byte, 4-byte
# and 2-byte aligned.  Rows at and around a tile, and enough of them for the 256-wide tiles.
@pytest.mark.parametrize("N", [64, 1, 71, 100, 129, 1021])
@pytest.mark.parametrize("M", [1, 65, 130, 2100])
@pytest.mark.parametrize("kind", ["f16", "f16_prelu", "i8", "i8_rowmajor"])
def test_rows_of_any_alignment(kind, M, N):
    K, st = 192, stream_ptr(torch.device("cuda"))
    g = torch.Generator().manual_seed(N + M)
    x = torch.randn(M, K, generator=g).half().cuda()
    q = torch.randint(-127, 128, (N, K), generator=g, dtype=torch.int8).cuda()
    s = (torch.rand(N, generator=g) * 1e-3 + 1e-4).half().cuda()
    w = (torch.randn(N, K, generator=g) * K ** -0.5).half().cuda()
    b = torch.randn(N, generator=g).cuda()
    res = torch.randn(M, N, generator=g).half().cuda()
    wp = pack_f16(w) if kind.startswith("f16") else pack_i8(q)

    def run(r, ldr, y, ldy):
        rp = None if r is None else r.data_ptr()
        if kind == "f16":
            _ffi.call("ecd_gemm_f16p", x.data_ptr(), K, wp.data_ptr(), b.data_ptr(), 0.5, rp, ldr, y.data_ptr(), ldy, M,
                      N, K, st)
        elif kind == "f16_prelu":
            _ffi.call("ecd_gemm_f16p_prelu", x.data_ptr(), K, wp.data_ptr(), b.data_ptr(), 0.25, rp, ldr, y.data_ptr(),
                      ldy, M, N, K, st)
        elif kind == "i8":
            _ffi.call("ecd_gemm_i8p", x.data_ptr(), K, wp.data_ptr(), s.data_ptr(), rp, ldr, y.data_ptr(), ldy, M, N, K,
                      st)
        else:
            _ffi.call("ecd_gemv_i8", x.data_ptr(), K, q.data_ptr(), s.data_ptr(), rp, ldr, y.data_ptr(), ldy, M, N, K,
                      1, st)

    n8 = (N + 7) // 8 * 8
    for with_res in (False, True):
        _, want = rows(M, N, n8, 0)
        _, r = rows(M, N, n8, 0, res)
        run(r if with_res else None, n8, want, n8)
        for ldy, lead, ldr, rlead in [(n8 + 4, 4, n8, 0), (n8, 4, n8 + 4, 4), (n8 + 2, 2, n8 + 6, 0), (n8 + 1, 1, n8 + 3, 3),
                                      (N, 0, N, 1)]:
            buf, y = rows(M, N, ldy, lead)
            _, r = rows(M, N, ldr, rlead, res)
            run(r if with_res else None, ldr, y, ldy)
            assert torch.equal(y, want), (with_res, ldy, lead, ldr, rlead)
            assert gaps_kept(buf, y, lead, ldy)
        if with_res and kind != "i8" and kind != "i8_rowmajor":  # in place
            buf, y = rows(M, N, n8 + 1, 3, res)
            run(y, n8 + 1, y, n8 + 1)
            assert torch.equal(y, want) and gaps_kept(buf, y, 3, n8 + 1)


@pytest.mark.parametrize("F", [32, 33, 70, 515])
@pytest.mark.parametrize("kind", ["f16", "i8"])
def test_silu_rows_of_any_alignment(kind, F):
    M, K, st = 70, 128, stream_ptr(torch.device("cuda"))
    g = torch.Generator().manual_seed(F)
    F += F % 2 if kind == "i8" else 0  # the int8 entry takes even widths
    x = torch.randn(M, K, generator=g).half().cuda()
    q = torch.randint(-127, 128, (2 * F, K), generator=g, dtype=torch.int8).cuda()
    s = (torch.rand(2 * F, generator=g) * 1e-3 + 1e-4).half().cuda()
    wp = pack_f16(q.half() * 1e-3, interleave=True) if kind == "f16" else pack_i8(q, interleave=True)

    def run(y, ldy):
        if kind == "f16":
            _ffi.call("ecd_gemm_f16p_silu", x.data_ptr(), K, wp.data_ptr(), y.data_ptr(), ldy, M, F, K, st)
        else:
            _ffi.call("ecd_gemm_i8p_silu", x.data_ptr(), K, wp.data_ptr(), s.data_ptr(), y.data_ptr(), ldy, M, F, K, st)

    f8 = (F + 7) // 8 * 8
    _, want = rows(M, F, f8, 0)
    run(want, f8)
    for ldy, lead in [(f8 + 2, 0), (f8 + 4, 2), (f8 + 6, 4)]:
        buf, y = rows(M, F, ldy, lead)
        run(y, ldy)
        assert torch.equal(y, want) and gaps_kept(buf, y, lead, ldy)


# the rule for short K: up to and past one round of 64 x 128 tiles, its second round where 128 x 128 tiles need one too,
# the last K it takes and the first it does not, ragged rows and features
@pytest.mark.parametrize("M,N,K", [(16384, 64, 64), (16385, 40, 64), (8193, 128, 512), (8193, 128, 576), (16256, 127, 128),
                                   (16383, 128, 128), (8065, 193, 256), (4033, 513, 192),
                                   (16500, 191, 64), (1, 64, 64)])
def test_short_k_choice_equals_every_tile(M, N, K):
    st = stream_ptr(torch.device("cuda"))
    g = torch.Generator().manual_seed(M + K)
    x = torch.randn(M, K, generator=g).half().cuda()
    w = (torch.randn(N, K, generator=g) * K ** -0.5).half().cuda()
    b = torch.randn(N, generator=g).cuda()
    wp, res = pack_f16(w), torch.randn(M, N, generator=g).half().cuda()

    def run(cfg):
        y = torch.empty(M, N, device="cuda", dtype=torch.float16)
        _ffi.call("ecd_gemm_f16p_tuned", x.data_ptr(), K, wp.data_ptr(), b.data_ptr(), 0.25, res.data_ptr(), N, y.data_ptr(),
                  N, M, N, K, 2, cfg, st)
        return y

    y = run(0)
    assert all(torch.equal(y, run(cfg)) for cfg in (1, 5, 8, 9, 10))
    v = x.double() @ w.double().t() + b.double()
    want = torch.where(v < 0, 0.25 * v, v) + res.double()
    # three fp16 roundings of values no larger than |v| + |res|, and K fp32 additions
    tol = 3 * 2.0 ** -11 * (v.abs() + res.double().abs()) + K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t()) + 1e-6
    assert bool(((y.double() - want).abs() <= tol).all())
