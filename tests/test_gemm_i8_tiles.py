"""The int8 GEMM's choice of tile, and every tile on ragged shapes in both weight layouts."""
import pytest
import torch

from estudiocanciones_amd import _ffi

TILE = {1: (256, 128), 2: (128, 128), 3: (64, 128), 4: (64, 64), 5: (128, 128)}


@pytest.mark.parametrize("M,N,K,tile", [
    # more than two 128 x 128 workgroups per CU, 256 x 128 tiles in 1.03 to 1.5 and 2.25 to 2.5 rounds: us of the tile
    # before, of three workgroups per CU: 93.8, 77.8 | 84.3, 74.9 | 219, 208 | 137, 130 | 130, 119 | 130, 113
    (4096, 3072, 3072, 5), (3840, 3072, 3072, 5), (4096, 3072, 8192, 5), (4096, 5120, 3072, 5), (3600, 5120, 3072, 5),
    (1152, 16384, 3072, 5),
    # 256 x 128 tiles in whole rounds: 49.1 against 49.4 | 95.2, 107 | 100, 110 | 296, 310 | 405, 455
    (2560, 3072, 3072, 1), (3072, 5120, 3072, 1), (1024, 16384, 3072, 1), (3072, 16384, 3072, 1), (4096, 16384, 3072, 1),
    # one or two of 128 x 128 per CU, few rows
    (1024, 3072, 3072, 2), (154, 16384, 3072, 2), (154, 5120, 3072, 4), (154, 3072, 3072, 4)])
def test_tile_choice(M, N, K, tile):
    assert _ffi.lib().ecd_gemm_i8p_tile(M, N, K) == tile


def test_tile_choice_refuses_no_size():
    lib = _ffi.lib()
    assert lib.ecd_gemm_i8p_tile(0, 64, 64) == 0 and lib.ecd_gemm_i8p_tile(4, 64, 65) == 0
    assert lib.ecd_gemm_i8p_tile(2 ** 20, 2 ** 20, 2 ** 30) in TILE


# rows and features one short of, at and one past each tile's edge (rows of one workgroup and of two), few features;
# K of one chunk, fewer chunks than any tile's stages, more than every tile's
@pytest.mark.gpu
@pytest.mark.parametrize("K", [64, 192, 1088])
@pytest.mark.parametrize("rowmajor", [0, 1])
@pytest.mark.parametrize("tile", [1, 2, 3, 4, 5])
def test_every_tile_on_ragged_shapes(tile, rowmajor, K):
    from estudiocanciones_amd.kernels import pack_i8, stream_ptr
    st = stream_ptr(torch.device("cuda"))
    bn, bm = TILE[tile]
    g = torch.Generator().manual_seed(tile + K)
    for N in (5, bn - 1, bn, bn + 1, 8 * bn + 21):
        q = torch.randint(-127, 128, (N, K), generator=g, dtype=torch.int8).cuda()
        s = (torch.rand(N, generator=g) * 1e-3 + 1e-4).half().cuda()
        w = q if rowmajor else pack_i8(q)
        w64 = (q.half() * s[:, None]).double()
        for M in (1, bm - 1, bm, bm + 1, 2 * bm + 37):
            x = torch.randn(M, K + 8, generator=g).half().cuda()[:, :K]  # a row stride of its own
            res = torch.randn(M, N, generator=g).half().cuda()
            out = torch.full((M + 1, N), 7.0, device="cuda", dtype=torch.float16)
            _ffi.call("ecd_gemm_i8p_tuned", x.data_ptr(), K + 8, w.data_ptr(), s.data_ptr(), res.data_ptr(), N,
                      out.data_ptr(), N, M, N, K, rowmajor, tile, st)
            p = x.double() @ w64.t()
            mag = x.double().abs() @ w64.abs().t()
            # K fp32 additions of at most mag, the fp16 rounding of the product and that of the residual's sum
            tol = K * 2.0 ** -24 * mag + 2.0 ** -11 * p.abs() + 2.0 ** -11 * (p + res.double()).abs() + 2.0 ** -24
            assert bool(((out[:M].double() - (p + res.double())).abs() <= 1.01 * tol).all()), (N, M)
            assert bool((out[M] == 7.0).all())


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["packed", "rowmajor", "silu", "rope"])
def test_entry_points_on_three_workgroups_per_cu(kind):
    """A ragged shape of the rule's own through each entry point: as tile 2 there, but for the order of the sums."""
    from estudiocanciones_amd.kernels import gemm_packed, gemm_rope_packed, gemm_silu_packed, int8_mm, pack_i8
    M, N, K = 1155, 8448, 128
    assert _ffi.lib().ecd_gemm_i8p_tile(M, N, K) == 5
    g = torch.Generator().manual_seed(5)
    x = torch.randn(M, K, generator=g).half().cuda()
    q = torch.randint(-127, 128, (N, K), generator=g, dtype=torch.int8).cuda()
    s = (torch.rand(N, generator=g) * 1e-3 + 1e-4).half().cuda()
    y64 = x.double() @ (q.half() * s[:, None]).double().t()
    rel = lambda a, b: float((a.double() - b).norm() / b.norm())
    if kind == "packed":
        assert rel(gemm_packed(x, pack_i8(q), s, N, K), y64) < 3e-4
    elif kind == "rowmajor":
        assert rel(int8_mm(x, q, s), y64) < 3e-4
    elif kind == "silu":
        # interleaved: packed row 2 j is source row j, 2 j + 1 is source row N / 2 + j; scales in packed order
        sp = torch.stack([s[:N // 2], s[N // 2:]], 1).reshape(-1).contiguous()
        mm = gemm_silu_packed(x, pack_i8(q, interleave=True), sp, N // 2, K)
        a, b = y64[:, :N // 2], y64[:, N // 2:]
        assert rel(mm, torch.nn.functional.silu(a) * b) < 6e-4
    else:
        Hq, Hk, HD, S = 44, 11, 128, M
        rope = torch.zeros(S, HD, device="cuda")
        ang = torch.rand(S, HD // 2, generator=g).cuda()
        rope[:, 0::2], rope[:, 1::2] = ang.cos(), ang.sin()
        pos = torch.arange(S, device="cuda")
        qo = torch.empty(M, Hq * HD, device="cuda", dtype=torch.float16)
        kc, vc = (torch.zeros(1, Hk, S, HD, device="cuda", dtype=torch.float16) for _ in range(2))
        gemm_rope_packed(x, pack_i8(q), s, rope, pos, qo, kc, vc, S, Hq, Hk, S, HD, K)
        h = y64.view(M, Hq + 2 * Hk, HD)
        c, t = ang.double().cos()[:, None], ang.double().sin()[:, None]
        r = torch.empty_like(h)
        r[..., 0::2] = h[..., 0::2] * c - h[..., 1::2] * t
        r[..., 1::2] = h[..., 1::2] * c + h[..., 0::2] * t
        assert rel(qo.view(M, Hq, HD), r[:, :Hq]) < 6e-4
        assert rel(kc[0].transpose(0, 1), r[:, Hq:Hq + Hk]) < 6e-4
        assert rel(vc[0].transpose(0, 1), h[:, Hq + Hk:]) < 6e-4
