"""Products split over K whose fp32 partial sums the next norm adds (the codec's and the prompt pass's
residual branches), against the exact product and the unsplit kernels' rounding points."""
import pytest
import torch

from estudiocanciones_amd import _ffi
from estudiocanciones_amd.kernels import gemm_rms_packed, pack_f16, pack_i8, stream_ptr

pytestmark = pytest.mark.gpu


def rms_of(h, w, eps=1e-5):
    f = h.double()
    return ((f / (f.pow(2).mean(1, keepdim=True) + eps).sqrt()).half() * w)


# rows at and around a tile, ways that do not divide the chunks, the most ways, K of two chunks per way
@pytest.mark.parametrize("M,N,K,ks", [(1, 64, 128, 2), (63, 192, 320, 2), (65, 1536, 1536, 5), (187, 1536, 4096, 3),
                                      (130, 320, 1024, 8), (64, 64, 64, 1)])
@pytest.mark.parametrize("kind", ["f16", "i8"])
def test_partials_sum_to_the_product(kind, M, N, K, ks):
    g = torch.Generator().manual_seed(M + N + K)
    st = stream_ptr(torch.device("cuda"))
    big = torch.randn(M, K + 8, generator=g).half().cuda()
    x = big[:, :K]  # a row stride of its own
    ws = torch.full((ks * M * N + 64,), 7.0, device="cuda")
    if kind == "f16":
        w = (torch.randn(N, K, generator=g) * K ** -0.5).half().cuda()
        wp = pack_f16(w)
        _ffi.call("ecd_gemm_f16p_partial", x.data_ptr(), K + 8, wp.data_ptr(), ws.data_ptr(), M, N, K, ks, st)
    else:
        q = torch.randint(-127, 128, (N, K), generator=g, dtype=torch.int8).cuda()
        s = (torch.rand(N, generator=g) * 1e-3 + 1e-4).half().cuda()
        w = q.half() * s[:, None]
        wp = pack_i8(q)
        _ffi.call("ecd_gemm_i8p_partial", x.data_ptr(), K + 8, wp.data_ptr(), s.data_ptr(), ws.data_ptr(), M, N, K,
                  ks, st)
    ref = x.double().cpu() @ w.double().cpu().t()
    mag = x.double().abs().cpu() @ w.double().abs().cpu().t()
    got = ws[:ks * M * N].view(ks, M, N).double().sum(0).cpu()
    # each fp32 addition of at most K + ks rounds at 2^-24 of a partial sum no larger than sum |x w|
    assert bool(((got - ref).abs() <= (K + ks) * 2.0 ** -24 * mag).all())
    assert bool((ws[ks * M * N:] == 7.0).all())


@pytest.mark.parametrize("M,N,K", [(17, 512, 1024), (77, 3072, 512), (40, 192, 2048), (600, 3072, 256)])
def test_residual_and_norm_after_a_split_product(M, N, K):
    g = torch.Generator().manual_seed(N)
    x = torch.randn(M, K, generator=g).half().cuda()
    q = torch.randint(-127, 128, (N, K), generator=g, dtype=torch.int8).cuda()
    s = (torch.rand(N, generator=g) * 1e-3 + 1e-4).half().cuda()
    res = torch.randn(M, N, generator=g).half().cuda()
    nw = torch.randn(N, generator=g).half().cuda()
    keep = res.clone()
    h, y = gemm_rms_packed(x, pack_i8(q), s, N, K, res, nw)
    assert torch.equal(res, keep)
    ref = (x.double().cpu() @ (q.half() * s[:, None]).double().cpu().t()).half() + res.cpu()
    # one fp16 ulp of either rounding of h (the fp32 sum against the exact one at a tie)
    tol = 2.0 ** -10 * (ref.double().abs() + (ref.double() - res.cpu().double()).abs()) + 1e-6
    assert bool(((h.double().cpu() - ref.double()).abs() <= tol).all())
    want = rms_of(h, nw).double()
    # two fp16 roundings, each one ulp off at most where the fp32 norm lies at a tie
    assert bool(((y.double() - want).abs() <= 2 * 2.0 ** -10 * want.abs() + 1e-6).all())


@pytest.mark.parametrize("norm", [0, 1])
def test_modulated_norm_adds_the_partials(norm):
    M, D, T, ks = 37, 200, 20, 3
    g = torch.Generator().manual_seed(norm)
    st = stream_ptr(torch.device("cuda"))
    r = lambda *s: torch.randn(*s, generator=g).half().cuda()
    parts = torch.randn(ks, M, D, generator=g).cuda()
    acc = parts[0].clone()
    for k in range(1, ks):
        acc = acc + parts[k]
    h, x1, w, tab, tm = acc.half(), r(M, D), r(D), r(3, D), r(2, 3 * D)
    x2, y1, y2 = x1.clone(), torch.empty_like(x1), torch.empty_like(x1)
    o = lambda t, i: t.data_ptr() + 2 * D * i
    tail = (o(tab, 0), o(tm, 0), 3 * D, w.data_ptr(), o(tab, 1), o(tm, 1), o(tab, 2), o(tm, 2), 3 * D)
    _ffi.call("ecd_codec_norm_mod", x1.data_ptr(), h.data_ptr(), *tail, y1.data_ptr(), M, T, D, norm, 1e-6, st)
    _ffi.call("ecd_codec_norm_mod_sum", x2.data_ptr(), parts.data_ptr(), ks, *tail, y2.data_ptr(), M, T, D, norm,
              1e-6, st)
    assert torch.equal(x1, x2) and torch.equal(y1, y2)


def test_split_rule():
    lib = _ffi.lib()
    for f in (lib.ecd_gemm_f16p_splits, lib.ecd_gemm_i8p_splits):
        assert f(77, 3072, 8192) > 1 and f(4096, 3072, 8192) == 1
        assert f(77, 3000, 8192) == 1 and f(77, 3072, 64) == 1 and f(0, 3072, 64) == 1
