"""Products of 129 to 256 rows against many columns, whose tiles are as high as the rows need, and the tiles on eight wavefronts at their edges:
whole numbers, so every result is exact."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("M", [129, 160, 161, 192, 193, 224, 225])
@pytest.mark.parametrize("N,Kd", [(65536, 64), (65400, 136), (65288, 712), (82000, 72)])   # the last: a part of a second round, in two heights
def test_heights(dtype, M, N, Kd):
    from nanoflow_amd import kernels as K
    gen = torch.Generator(device="cuda").manual_seed(M + Kd)
    whole = lambda *shape, top: torch.randint(-top, top + 1, shape, generator=gen, device="cuda")
    a, b, c = whole(M, Kd, top=1), whole(N, Kd, top=1), whole(M, N, top=8)      # results stay below 256 but for a chance of 1e-20
    want = a.double() @ b.double().t()
    cast = lambda t: t.to(getattr(torch, dtype))
    assert want.abs().max() < 240
    guard = torch.full((M + 1, N), 77.0, dtype=getattr(torch, dtype), device="cuda")
    K.gemm(cast(a), cast(b), b_col_major=True, out=guard[:M])
    assert torch.equal(guard[:M].double(), want) and (guard[M] == 77.0).all()
    K.gemm(cast(a), cast(b), Cmat=cast(c), beta=1.0, b_col_major=True, out=guard[:M])
    assert torch.equal(guard[:M].double(), want + c) and (guard[M] == 77.0).all()


@pytest.mark.parametrize("nk", [True, False])
@pytest.mark.parametrize("M,N,Kd", [(129, 264, 64), (300, 4104, 200), (513, 6152, 136), (700, 2040, 712), (1000, 4096, 72), (2040, 8184, 136), (1793, 8200, 328)])
def test_eight_wavefronts(nk, M, N, Kd):
    from nanoflow_amd import kernels as K
    gen = torch.Generator(device="cuda").manual_seed(M + Kd)
    whole = lambda *shape, top: torch.randint(-top, top + 1, shape, generator=gen, device="cuda")
    a, b, c = whole(M, Kd, top=1), whole(N, Kd, top=1), whole(M, N, top=8)
    want = a.double() @ b.double().t()
    guard = torch.full((M + 1, N), 77.0, dtype=torch.float16, device="cuda")
    w = b.half() if nk else b.half().t().contiguous()
    K.gemm(a.half(), w, Cmat=c.half(), beta=1.0, b_col_major=nk, out=guard[:M])
    assert torch.equal(guard[:M].double(), want + c) and (guard[M] == 77.0).all()
    if nk:
        sums = K.gemm_nk_sums(a.bfloat16(), b.bfloat16(), 16)
        assert torch.equal(sums.double().sum(0), want)


# by the tiles they are computed in on 256 CUs
ROUND = {"128 x 128": [(65, 16392, 2048), (128, 16392, 4096)], "128 x 256": [(66, 33608, 2048), (128, 65400, 2048)], "160 x 256": [(129, 49864, 2048), (160, 65400, 2048)],
         "192 x 256": [(161, 49864, 2048), (192, 65400, 2048)], "224 x 256": [(193, 49160, 2048), (224, 65400, 2048)], "256 x 256": [(225, 49864, 2048), (256, 65400, 2048)],
         "256 x 192": [(129, 32776, 2048), (192, 32776, 4096), (256, 49152, 2048)]}


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("M,N,Kd", [s for shapes in ROUND.values() for s in shapes])
def test_contractions_that_go_round(M, N, Kd, dtype):
    """Column tiles that start K at slabs of their own: every first slab there is, and a last column tile that is cut."""
    from nanoflow_amd import kernels as K
    assert N * Kd * 2 >= 64 << 20 and (N + 255) // 256 >= Kd // 64
    gen = torch.Generator(device="cuda").manual_seed(M)
    whole = lambda *shape, top=1: torch.randint(-top, top + 1, shape, generator=gen, device="cuda", dtype=torch.int8)
    cast = lambda t: t.to(getattr(torch, dtype))
    a, b, c = whole(M, Kd), whole(N, Kd), whole(M, N, top=8)
    want = a.float() @ b.float().t()
    assert want.abs().max() <= 1024
    guard = torch.full((M + 1, N), 77.0, dtype=getattr(torch, dtype), device="cuda")
    K.gemm(cast(a), cast(b), b_col_major=True, out=guard[:M])
    assert torch.equal(guard[:M], cast(want)) and (guard[M] == 77.0).all()
    K.gemm(cast(a), cast(b), Cmat=cast(c), beta=1.0, b_col_major=True, out=guard[:M])
    assert torch.equal(guard[:M], cast(want + c)) and (guard[M] == 77.0).all()


# 128 x 128, and 256 x 128, of both matrices
@pytest.mark.parametrize("M,N,Kd", [(65, 16392, 2048), (128, 16392, 4096), (129, 49864, 2048), (180, 49864, 2048), (256, 49864, 2048)])
def test_pairs_that_go_round(M, N, Kd):
    from nanoflow_amd import kernels as K
    gen = torch.Generator(device="cuda").manual_seed(M)
    a, g, u = (torch.randint(-1, 2, shape, generator=gen, device="cuda", dtype=torch.int8).half() for shape in ((M, Kd), (N, Kd), (N, Kd)))
    assert torch.equal(K.dual_swiglu(a, g, u, b_col_major=True), K.dual_swiglu(a, g.t().contiguous(), u.t().contiguous()))
