"""Products of more than 320 rows that are split over K (mid_split_plan in csrc/kernels/gemm_impl.h) against float64, with the bound
of test_gpu_few_rows.py: one rounding to 16 bits, and K 2^-24 sum |a||b| of fp32 sums."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
from test_gpu_few_rows import check, operands

SHAPES = [(321, 2048, 4096), (383, 520, 2048), (385, 264, 8200), (512, 2048, 4104), (513, 4096, 14336), (640, 2056, 8192), (767, 1032, 6152),
          (769, 520, 4096), (1000, 4096, 8192), (1025, 2048, 8200), (1281, 1024, 4096), (1500, 4096, 14336)]


@pytest.mark.parametrize("M,N,K_", SHAPES)
def test_split_products(M, N, K_):
    from nanoflow_amd import kernels as K
    ws = torch.empty(64 << 20, dtype=torch.uint8, device="cuda")
    a, b = operands(M, N, K_, torch.float16)
    want = a.double() @ b.double().t()
    kn = b.t().contiguous()
    c, bias = torch.randn(M, N, device="cuda").half(), torch.randn(N, device="cuda").half()
    for w, col in ((b, True), (kn, False)):
        got, _ = K.gemm_ws(a, w, b_col_major=col, workspace=ws)
        check(got, want, a, b, K_, 11)
        d = c.clone()
        K.gemm_ws(a, w, d, alpha=0.5, beta=1.0, b_col_major=col, out=d, workspace=ws)
        check(d, 0.5 * want + c.double(), a, b, K_, 11)
        check(K.gemm_ws(a, w, bias=bias, beta=1.0, b_col_major=col, workspace=ws)[0], want + bias.double(), a, b, K_, 11)
        small, _ = K.gemm_ws(a, w, b_col_major=col, workspace=ws[:16])              # no room: unsplit
        assert torch.equal(small, K.gemm(a, w, b_col_major=col))
    need = K.lib().nf_gemm_nk_workspace_bytes_upto(M, N, K_)
    assert K.lib().nf_gemm_workspace_bytes_upto(M, N, K_) <= max(64 << 20, 2 * M * N * 4)
    a, b = operands(M, N, K_, torch.bfloat16)
    want = a.double() @ b.double().t()
    ws = torch.empty(max(need, 16), dtype=torch.uint8, device="cuda")
    check(K.gemm_nk(a, b, workspace=ws), want, a, b, K_, 8)
    relu2 = K.gemm_nk(a, b, workspace=ws, act=K.ACT_SQUARED_RELU)
    lost = 2 * want.abs() * K_ * 2.0 ** -24 * (a.double().abs() @ b.double().abs().t())
    r = want.clamp(min=0) ** 2
    assert bool(((relu2.double() - r).abs() <= 2.0 ** -8 * r + 1.1 * lost + 1e-7).all())


@pytest.mark.parametrize("col", [True, False])
@pytest.mark.parametrize("M,N,K_", [(321, 2048, 4096), (400, 4096, 8192), (400, 4096, 14336), (512, 2048, 4104), (600, 1024, 4096), (640, 2056, 8192),
                                    (640, 4096, 14336), (769, 520, 4096), (1024, 4096, 14336), (1500, 4096, 14336)])
def test_workspace_beyond_what_a_shape_asks_for_changes_nothing(M, N, K_, col):
    """nf_gemm_workspace_bytes is the whole contract: 0 = the workspace is not touched, and bytes past the ones asked for neither."""
    from nanoflow_amd import kernels as K
    a, b = operands(M, N, K_, torch.float16)
    w = b if col else b.t().contiguous()
    need = K.lib().nf_gemm_workspace_bytes(M, N, K_)
    ws = torch.full(((96 << 20) + 16,), 0x5a, dtype=torch.uint8, device="cuda")
    big, _ = K.gemm_ws(a, w, b_col_major=col, workspace=ws)
    untouched = bool((ws[need:] == 0x5a).all())
    assert untouched
    exact = K.gemm_ws(a, w, b_col_major=col, workspace=torch.empty(need, dtype=torch.uint8, device="cuda"))[0] if need else K.gemm(a, w, b_col_major=col)
    assert torch.equal(big, exact)
    ab, bb = a.bfloat16(), b.bfloat16()                          # the bf16 entry: two sizes that both suffice
    upto = K.lib().nf_gemm_nk_workspace_bytes_upto(M, N, K_)
    assert torch.equal(K.gemm_nk(ab, bb, workspace=ws), K.gemm_nk(ab, bb, workspace=torch.empty(max(upto, 16), dtype=torch.uint8, device="cuda")))


@pytest.mark.parametrize("M,N", [(321, 2048), (448, 2048), (512, 1024)])
def test_contractions_of_2048_are_not_split(M, N):
    from nanoflow_amd import kernels as K
    a, b = operands(M, N, 2048, torch.bfloat16)
    assert torch.equal(K.gemm_nk(a, b, workspace=torch.empty(64 << 20, dtype=torch.uint8, device="cuda")), K.gemm_nk(a, b))


@pytest.mark.parametrize("M,N,K_", [(1, 4096, 4096), (16, 2048, 2048), (33, 4096, 14336), (64, 4096, 4096), (200, 2048, 4096), (300, 4096, 4096), (400, 1024, 14336),
                                    (400, 2048, 4096), (640, 4096, 14336), (1024, 4096, 14336), (1500, 4096, 14336)])
def test_a_workspace_that_is_not_aligned(M, N, K_):
    """Refused where it would hold sums (up to 512 rows whatever the launch runs on, and of dense launches); else not looked at."""
    from nanoflow_amd import kernels as K
    a, b = operands(M, N, K_, torch.float16)
    ws = torch.empty((96 << 20) + 8, dtype=torch.uint8, device="cuda")[8:]
    asked = K.lib().nf_gemm_workspace_bytes(M, N, K_) > 0
    for w, col in ((b, True), (b.t().contiguous(), False)):
        if asked and not 512 < M <= 768:
            with pytest.raises(K.NanoflowKernelError, match="aligned"):
                K.gemm_ws(a, w, b_col_major=col, workspace=ws)
        else:
            assert torch.equal(K.gemm_ws(a, w, b_col_major=col, workspace=ws)[0], K.gemm(a, w, b_col_major=col))
        if K.lib().nf_dual_swiglu_workspace_bytes(M, N, K_):
            with pytest.raises(K.NanoflowKernelError, match="aligned"):
                K.dual_swiglu_ws(a, w, w, b_col_major=col, workspace=ws)
    ab, bb = a.bfloat16(), b.bfloat16()
    if asked and M <= 320:
        with pytest.raises(K.NanoflowKernelError, match="aligned"):
            K.gemm_nk(ab, bb, workspace=ws)
    else:
        assert torch.equal(K.gemm_nk(ab, bb, workspace=ws), K.gemm_nk(ab, bb))


@pytest.mark.parametrize("col", [True, False])
@pytest.mark.parametrize("M,N,K_", [(321, 2048, 4096), (330, 256, 12288), (383, 520, 16384), (400, 2048, 8192), (400, 1024, 14336), (512, 2048, 4104), (512, 512, 14336)])
def test_products_without_a_workspace_of_the_callers(M, N, K_, col):
    """nf_gemm_f16_noalloc has the bits of nf_gemm_f16_ws up to 512 rows."""
    from nanoflow_amd import kernels as K
    l = K.lib()
    assert l.nf_gemm_workspace_bytes(M, N, K_) <= l.nf_gemm_noalloc_scratch_bytes()
    a, b = operands(M, N, K_, torch.float16)
    w = b if col else b.t().contiguous()
    out = torch.empty((M, N), dtype=torch.float16, device="cuda")
    assert l.nf_gemm_f16_noalloc(a.data_ptr(), w.data_ptr(), None, out.data_ptr(), M, N, K_, 1.0, 0.0, int(col), torch.cuda.current_stream().cuda_stream) == 0
    assert torch.equal(out, K.gemm_ws(a, w, b_col_major=col)[0])


@pytest.mark.parametrize("M,N,K_", [(65, 520, 512), (128, 4104, 968), (127, 33000, 136), (129, 66008, 72), (200, 65544, 328), (256, 49160, 64), (64, 264, 1000)])
def test_one_row_of_tiles(M, N, K_):
    """Unsplit launches whose tiles share no weights: those are read with a hint of their own."""
    from nanoflow_amd import kernels as K
    a, b = operands(M, N, K_, torch.float16)
    check(K.gemm(a, b, b_col_major=True), a.double() @ b.double().t(), a, b, K_, 11)
    half = N // 16 * 8
    g, u = b[:half].contiguous(), b[half:2 * half].contiguous()
    p, q = a.double() @ g.double().t(), a.double() @ u.double().t()
    pair = torch.nn.functional.silu(p.half().double()) * q.half().double()
    lost = lambda r, w: 2.0 ** -11 * r.abs() + K_ * 2.0 ** -24 * (a.double().abs() @ w.double().abs().t())
    got = K.dual_swiglu(a, g, u, b_col_major=True)
    assert bool(((got.double() - pair).abs() <= 1.1 * q.abs() * lost(p, g) + p.abs() * lost(q, u) + 2.0 ** -10 * pair.abs() + 1e-6).all())
