"""e4m3 products on the large tiles (csrc/kernels/gemm_f8.hip): rings of one slab to several, cut slabs, ragged rows and columns.
Operands are whole numbers up to 4 and scales powers of two, so every sum is exact in fp32 and the result is its one rounding."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

DEPTHS = [16, 128, 144, 256, 272, 384, 528, 1040]


def operands(M, N, K_, n):
    gen = torch.Generator(device="cuda").manual_seed(M + N + K_)
    codes = [torch.randint(-4, 5, (r, K_), generator=gen, device="cuda").float().to(torch.float8_e4m3fn) for r in [M] + [N] * n]
    scales = [2.0 ** torch.randint(-6, -3, (r,), generator=gen, device="cuda").float() for r in [M] + [N] * n]
    values = [q.float().double() * s.double()[:, None] for q, s in zip(codes, scales)]
    return [q.view(torch.uint8) for q in codes], scales, values, gen


@pytest.mark.parametrize("K_", DEPTHS)
@pytest.mark.parametrize("M,N", [(2048, 8192), (1800, 8008), (2000, 6152), (1793, 5960), (2000, 6144), (2000, 10240), (1990, 10216), (1030, 4104), (300, 520)])
# 256 x 256 tiles of the first three, 256 x 192 of the others (whole and ragged columns; 32 to 54 tiles of columns), at last 128 rows on eight wavefronts
def test_products(M, N, K_):
    from nanoflow_amd import kernels as K
    (a, b), (sa, sb), (av, bv), gen = operands(M, N, K_, 1)
    want = av @ bv.t()
    assert torch.equal(K.gemm_f8(a, sa, b, sb), want.half())
    c = torch.randint(-9, 10, (M, N), generator=gen, device="cuda").half()
    assert torch.equal(K.gemm_f8(a, sa, b, sb, c, alpha=0.5, beta=-1.0), (0.5 * want - c.double()).half())


@pytest.mark.parametrize("K_", DEPTHS)
@pytest.mark.parametrize("M,N", [(2048, 3072), (1937, 3080), (1937, 4232), (2048, 6144), (300, 520)])
# 256 x 128 tiles; the third and fourth with a last round of half the height; 128 x 128 on eight wavefronts
def test_pairs(M, N, K_):
    from nanoflow_amd import kernels as K
    (a, b, u), (sa, sb, su), (av, bv, uv), _ = operands(M, N, K_, 2)
    g, up = (av @ bv.t()).half().double(), (av @ uv.t()).half().double()
    pair = torch.nn.functional.silu(g) * up
    got = K.dual_swiglu_f8q(a, sa, b, sb, u, su)
    assert bool(((got.double() - pair).abs() <= 2.0 ** -10 * pair.abs() + 2.0 ** -24).all())  # fp32 exponential, then one rounding
