"""The GEMM epilogues' SiLU on every finite fp16 gate value: the nearest fp16 to x * sigmoid(x)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["f16", "i8"])
def test_silu_is_the_nearest_fp16_for_every_input(kind):
    import torch
    from estudiocanciones_amd.kernels import gemm_f16_silu_packed, gemm_silu_packed, pack_f16, pack_i8
    a = np.arange(65536, dtype=np.uint32).astype(np.uint16).view(np.float16)
    a = a[np.isfinite(a)]
    x = torch.zeros(a.size, 64, dtype=torch.float16)
    x[:, 0], x[:, 1] = torch.from_numpy(a), 1.0
    # feature j: gate row e_0 (the value itself), up row e_1 (one)
    F = 2
    w = torch.zeros(2 * F, 64, dtype=torch.float16)
    w[:F, 0], w[F:, 1] = 1.0, 1.0
    if kind == "f16":
        mm = gemm_f16_silu_packed(x.cuda(), pack_f16(w.cuda(), interleave=True), F, 64)
    else:
        s = torch.ones(2 * F, device="cuda", dtype=torch.float16)
        mm = gemm_silu_packed(x.cuda(), pack_i8(w.to(torch.int8).cuda(), interleave=True), s, F, 64)
    with np.errstate(over="ignore"):
        want = (a.astype(np.longdouble) / (1 + np.exp(-a.astype(np.longdouble)))).astype(np.float16)
    assert np.array_equal(mm[:, 0].cpu().numpy(), want) and torch.equal(mm[:, 0], mm[:, 1])
