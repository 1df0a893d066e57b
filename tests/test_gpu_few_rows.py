"""Products of at most 64 rows on whole-K workgroups (csrc/kernels/gemm_rows.h), and on the tiles that take [K][N] weights in the same
order: every tile of the dispatches (for 256 CUs) on ragged columns and at the edges of its rows, against
float64.  An element may be off by its one rounding to 16 bits and by what fp32 sums of K terms can lose:
2^-p |r| + K 2^-24 sum |a||b| (p = 11 significant bits for fp16, 8 for bf16)."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

BITS = {torch.float16: 11, torch.bfloat16: 8}


def operands(M, N, K, dtype, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed + M + N + K)
    return (torch.empty(s, device="cuda").normal_(0, d, generator=g).to(dtype) for s, d in (((M, K), 1.0), ((N, K), K ** -0.5)))


def check(got, want, a, b, K, bits, scale=1.0):
    sums = a.double().abs() @ b.double().abs().t()
    bound = 2.0 ** -bits * want.abs() + scale * K * 2.0 ** -24 * sums + 1e-7
    assert bool(((got.double() - want).abs() <= bound).all()), float(((got.double() - want).abs() / bound).max())


# rows at the edges of the row tiles, columns at those of the panels (and a lone one), K of whole and of cut units
SHAPES = [(m, n, k) for m in (1, 8, 9, 16, 17, 32, 33, 64) for n, k in ((8, 1536), (72, 1544), (4104, 2048), (264, 4096))] + \
    [(3, 8200, 1600), (13, 16392, 1536), (30, 16392, 1536), (64, 8200, 1544), (61, 16384, 1536), (40, 24, 6000), (17, 520, 8192), (5, 24, 8200)]


@pytest.mark.parametrize("M,N,K_", SHAPES)
def test_products_of_few_rows(M, N, K_):
    from nanoflow_amd import kernels as K
    a, b = operands(M, N, K_, torch.float16)
    want = a.double() @ b.double().t()
    got, _ = K.gemm_ws(a, b, b_col_major=True)
    check(got, want, a, b, K_, 11)
    c = torch.randn(M, N, device="cuda").half()
    d = c.clone()
    K.gemm_ws(a, b, d, alpha=0.5, beta=1.0, b_col_major=True, out=d)                 # in place, as the residual stream is
    check(d, 0.5 * want + c.double(), a, b, K_, 11)
    bias = torch.randn(N, device="cuda").half()
    check(K.gemm_ws(a, b, bias=bias, beta=1.0, b_col_major=True)[0], want + bias.double(), a, b, K_, 11)
    if M <= 16 or K_ <= 4096:   # a row is the same whatever comes with it
        assert torch.equal(got[M - 1:], K.gemm_ws(a[M - 1:].clone(), b, b_col_major=True)[0])


# every count of shares that the [K][N] tiles take (1, 2, 4, 8 of the classes), units that do not fill the classes evenly, cut slabs; and
# launches that are split over K into runs
LAYOUTS = SHAPES + [(17, 8200, 1600), (32, 14344, 1544), (16, 8264, 1544), (16, 5128, 4160), (33, 4104, 4104), (16, 33000, 1536), (24, 33008, 1544), (1, 4096, 4096), (16, 1000, 5000), (33, 8192, 4104), (64, 2056, 4160), (9, 10240, 8192), (48, 12296, 4096), (64, 28680, 2048),
                    (5, 33000, 1536), (3, 1024, 8200), (16, 2048, 14336), (9, 1032, 9000), (17, 4096, 14336), (64, 40, 8200), (50, 5120, 5128)]


@pytest.mark.parametrize("M,N,K_", LAYOUTS)
def test_both_layouts_of_the_weights_have_the_same_bits(M, N, K_):
    from nanoflow_amd import kernels as K
    a, b = operands(M, N, K_, torch.float16)
    kn = b.t().contiguous()
    c, bias = torch.randn(M, N, device="cuda").half(), torch.randn(N, device="cuda").half()
    need = K.lib().nf_gemm_workspace_bytes(M, N, K_)
    for size in {max(need, 16), 64 << 20}:
        ws = torch.empty(size, dtype=torch.uint8, device="cuda")
        both = lambda **kw: [K.gemm_ws(a, w, b_col_major=col, workspace=ws, **kw)[0] for w, col in ((b, True), (kn, False))]
        assert torch.equal(*both())
        assert torch.equal(*both(Cmat=c, alpha=0.7, beta=-1.3))
        assert torch.equal(*both(bias=bias, alpha=0.7, beta=1.9))
    assert torch.equal(K.gemm(a, b, c, 0.7, -1.3, b_col_major=True), K.gemm(a, kn, c, 0.7, -1.3))
    ab, bb = a.bfloat16(), b.bfloat16()
    assert torch.equal(K.gemm(ab, bb, b_col_major=True), K.gemm(ab, bb.t().contiguous()))
    check(K.gemm_ws(a, kn)[0], a.double() @ b.double().t(), a, b, K_, 11)
    half = max(N // 16 * 8, 8)                                   # the pair, with its workspace, with a short one and without
    g, u = b[:half].contiguous(), b[-half:].contiguous()
    kg, ku = g.t().contiguous(), u.t().contiguous()
    need = K.lib().nf_dual_swiglu_workspace_bytes(M, half, K_)
    for size in {max(need, 16), 16}:
        ws = torch.empty(size, dtype=torch.uint8, device="cuda")
        assert torch.equal(K.dual_swiglu_ws(a, g, u, b_col_major=True, workspace=ws)[0], K.dual_swiglu_ws(a, kg, ku, workspace=ws)[0])
    assert torch.equal(K.dual_swiglu(a, g, u, b_col_major=True), K.dual_swiglu(a, kg, ku))


@pytest.mark.parametrize("M,N,K_", [(1, 2048, 2048), (16, 40, 1544), (33, 72, 2048), (64, 2056, 4096), (40, 264, 8192), (64, 64, 2048), (17, 1024, 4104),
                                    (16, 1024, 14336), (9, 520, 9000), (2, 40, 4096), (1, 4104, 1536), (16, 4104, 1544), (32, 2056, 1536), (64, 4104, 1544),
                                    (32, 8200, 1544), (64, 8200, 1536)])
def test_bfloat16_products_and_sums(M, N, K_):
    from nanoflow_amd import kernels as K
    a, b = operands(M, N, K_, torch.bfloat16)
    ws = torch.empty(max(K.lib().nf_gemm_nk_workspace_bytes_upto(M, N, K_), 16), dtype=torch.uint8, device="cuda")
    want = a.double() @ b.double().t()
    check(K.gemm_nk(a, b, workspace=ws), want, a, b, K_, 8)
    check(K.gemm_nk(a, b, workspace=ws, squared_relu=True), want.clamp(min=0).square(), a, b, K_, 7, scale=2 * float(want.abs().max()) + 1)
    bias = torch.randn(N, device="cuda").bfloat16()
    check(K.gemm_nk(a, b, workspace=ws, bias=bias), want + bias.double(), a, b, K_, 8)
    check(K.gemm_nk_sums(a, b, 16).sum(0), want, a, b, K_, 20)


@pytest.mark.parametrize("M", [1, 8, 9, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("N,K_", [(72, 1544), (520, 2048), (1160, 4096)])
def test_gate_up_pair_of_few_rows(M, N, K_):
    from nanoflow_amd import kernels as K
    a, g = operands(M, N, K_, torch.float16)
    _, u = operands(M, N, K_, torch.float16, seed=1)
    gv, uv = (a.double() @ w.double().t() for w in (g, u))
    want = torch.nn.functional.silu(gv) * uv
    got, _ = K.dual_swiglu_ws(a, g, u, b_col_major=True)
    # both products are rounded to fp16 ahead of silu(g) * u, whose slopes are at most 1.1 |u| and |g|
    lost = lambda v, w: 2.0 ** -11 * v.abs() + K_ * 2.0 ** -24 * (a.double().abs() @ w.double().abs().t())
    bound = 1.1 * uv.abs() * lost(gv, g) + gv.abs() * lost(uv, u) + 2.0 ** -10 * want.abs() + 1e-6
    assert bool(((got.double() - want).abs() <= bound).all())
    if M <= 32:                 # [K][N] weights: the same bits
        assert torch.equal(got, K.dual_swiglu_ws(a, g.t().contiguous(), u.t().contiguous())[0])


# between 48 and 64 columns a CU: its edges, a cut tile, a last unit that is cut; a column's sums do not depend on the tile, so the bits are
# those of the same columns in launches of 32 a CU, whose tile the tests above hold to float64
@pytest.mark.parametrize("N,K_", [(12280, 1544), (12288, 1544), (14344, 3088), (16376, 1552), (16384, 4096)])
@pytest.mark.parametrize("M", [17, 32, 33, 64])
def test_gate_up_pair_on_wide_tiles(M, N, K_):
    from nanoflow_amd import kernels as K
    a, g = operands(M, N, K_, torch.float16)
    _, u = operands(M, N, K_, torch.float16, seed=1)
    halves = lambda pair: torch.cat([pair(slice(0, 8192))[:, :N - 8192], pair(slice(N - 8192, N))], 1)
    pair = lambda r: K.dual_swiglu_ws(a, g[r], u[r], b_col_major=True)[0]
    assert torch.equal(pair(slice(0, N)), halves(pair))
    if K_ < 3072:   # shorter e4m3 rows are not this stream's
        return
    qa, qg, qu = ((16 * w).to(torch.float8_e4m3fn).view(torch.uint8) for w in (a, g, u))
    sa, sg, su = (torch.rand(n, device="cuda") + 0.01 for n in (M, N, N))
    pair = lambda r: K.dual_swiglu_f8q(qa, sa, qg[r], sg[r], qu[r], su[r])
    assert torch.equal(pair(slice(0, N)), halves(pair))


@pytest.mark.parametrize("M", [1, 8, 9, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("N,K_", [(72, 3088), (4104, 4096), (264, 8192)])
def test_e4m3_products_of_few_rows(M, N, K_):
    from nanoflow_amd import kernels as K
    gen = torch.Generator(device="cuda").manual_seed(M + N + K_)
    codes = lambda r: (torch.randn((r, K_), generator=gen, device="cuda")).to(torch.float8_e4m3fn)
    a, b, u = codes(M), codes(N), codes(N)
    sa, sb, su = (torch.rand(n, generator=gen, device="cuda") * K_ ** -0.25 + 0.01 for n in (M, N, N))
    value = lambda q, s: q.float().double() * s.double()[:, None]
    av, bv, uv = value(a, sa), value(b, sb), value(u, su)
    c = torch.randn(M, N, generator=gen, device="cuda").half()
    raw = lambda q: q.view(torch.uint8)
    want = av @ bv.t()
    check(K.gemm_f8(raw(a), sa, raw(b), sb), want, av, bv, K_, 11)
    check(K.gemm_f8q(raw(a), sa, raw(b), sb, c, alpha=0.5, beta=1.0), 0.5 * want + c.double(), av, bv, K_, 11)
    g, up = want, av @ uv.t()
    lost = lambda v, w: 2.0 ** -11 * v.abs() + K_ * 2.0 ** -24 * (av.abs() @ w.abs().t())
    pair = torch.nn.functional.silu(g) * up
    got = K.dual_swiglu_f8q(raw(a), sa, raw(b), sb, raw(u), su)
    assert bool(((got.double() - pair).abs() <= 1.1 * up.abs() * lost(g, bv) + g.abs() * lost(up, uv) + 2.0 ** -10 * pair.abs() + 1e-6).all())


@pytest.mark.parametrize("M,N,K_", [(17, 14344, 3088), (32, 8200, 3104), (33, 8264, 3072), (64, 8200, 3088), (1, 16392, 3088), (8, 20488, 8176),
                                    (8, 20488, 8192), (17, 24584, 4096), (32, 24584, 3088), (32, 24584, 4112)])
def test_e4m3_products_of_few_rows_against_many_columns(M, N, K_):
    test_e4m3_products_of_few_rows(M, N, K_)


# 33 to 44 columns a CU against a long contraction: shares of K from 9 rows on, where the workspace holds their sums
@pytest.mark.parametrize("M,N,K_,shared", [(9, 8200, 9232, True), (32, 11264, 9232, True), (33, 12288, 8208, True), (64, 8200, 14336, True),
                                           (8, 8200, 9232, False), (32, 8200, 9216, False), (64, 8200, 8192, False), (16, 8200, 14352, False)])
def test_e4m3_products_in_shares(M, N, K_, shared):
    from nanoflow_amd import kernels as K
    gen = torch.Generator(device="cuda").manual_seed(M + N + K_)
    codes = lambda r: torch.randn((r, K_), generator=gen, device="cuda").to(torch.float8_e4m3fn)
    scales = lambda r: torch.rand(r, generator=gen, device="cuda") + 0.5
    a, b, sa, sb = codes(M), codes(N), scales(M), scales(N) * K_ ** -0.5
    av, bv = a.float().double() * sa.double()[:, None], b.float().double() * sb.double()[:, None]
    need = K.lib().nf_gemm_f8w_split_workspace_bytes(M, N, K_)
    ws = torch.full((need,), 255, dtype=torch.uint8, device="cuda")
    check(K.gemm_f8q(a.view(torch.uint8), sa, b.view(torch.uint8), sb, workspace=ws), av @ bv.t(), av, bv, K_, 11)
    assert bool((ws != 255).any()) == shared
    short = torch.full((need - 256,), 255, dtype=torch.uint8, device="cuda")
    check(K.gemm_f8q(a.view(torch.uint8), sa, b.view(torch.uint8), sb, workspace=short), av @ bv.t(), av, bv, K_, 11)
    assert bool((short == 255).all())


@pytest.mark.parametrize("K_", [4096, 8192, 14336, 32784])
def test_row_quantiser_of_nan_and_infinity(oracle, K_):
    """NaN takes no part in a row's maximum and becomes 448 like everything above it, of either sign; beside an infinity finite values become
    zeros of their sign.  Quiet and signalling NaN of both signs in every lane position of a chunk, on every row length's kernel."""
    import numpy as np
    from nanoflow_amd import kernels as K
    rng = np.random.default_rng(K_)
    x = (rng.standard_normal((24, K_)) * 10.0 ** rng.integers(-6, 4, (24, 1))).astype(np.float16).view(np.uint16)
    for row in range(24):
        at = rng.choice(K_, 64, replace=False)
        at[:8] = np.arange(8) + 8 * rng.integers(0, K_ // 8)                      # a whole chunk of them
        x[row, at] = np.resize(np.array([0x7e00, 0xfe00, 0x7c01, 0xfc01, 0x7d55, 0xffff], dtype=np.uint16), 64)
    x[16:20, rng.integers(0, K_, 3)] = 0x7c00
    x[18:22, rng.integers(0, K_, 3)] = 0xfc00
    x[22] = np.resize(np.array([0x7e00, 0xfc01], dtype=np.uint16), K_)           # nothing else: the scale of a row of zeros
    v = x.view(np.float16).astype(np.float32)
    q, s = K.quantize_rows_e4m3(torch.from_numpy(x.view(np.float16).copy()).cuda())
    q_ref, s_ref = oracle.quantize_rows_e4m3(x.view(np.float16))
    assert np.array_equal(s.cpu().numpy(), s_ref) and s_ref[22] == 1 and np.isinf(s_ref[16:22]).all()
    q, special = q.cpu().numpy(), np.isnan(v) | (np.isinf(v) & np.isinf(s_ref)[:, None])   # NaN, or infinity over infinity: no sign to speak of
    assert np.array_equal(q[~special], q_ref[~special])
    assert (q[special] & 0x7f == 0x7e).all() and (q_ref[special] & 0x7f == 0x7e).all()


@pytest.mark.parametrize("K_", [4096, 8192, 14336, 32784])
def test_row_quantiser_over_every_half(oracle, K_):
    """Rows that hold all halves up to a maximum (the largest, ordinary ones, the smallest, subnormal ones), on every row length's
    kernel: the oracle's bytes and scales; of rows with an infinity the scales."""
    import numpy as np
    from nanoflow_amd import kernels as K
    every = np.arange(65536, dtype=np.uint16)
    every = every[~((every & 0x7fff) > 0x7c00)]
    maxima = [0x7bff, 0x7c00, 0x5640, 0x3c00, 0x3555, 0x0401, 0x0400, 0x0003, 0x0001]
    rows = []
    for m in maxima:
        some = every[(every & 0x7fff) <= m]
        for at in range(0, len(some), K_):
            rows.append(np.concatenate(([np.uint16(m)], np.resize(some[at:at + K_], K_ - 1))))
    x = np.stack(rows).view(np.float16)
    q, s = K.quantize_rows_e4m3(torch.from_numpy(x.copy()).cuda())
    q_ref, s_ref = oracle.quantize_rows_e4m3(x)
    finite = np.isfinite(x.astype(np.float32)).all(1)
    assert np.array_equal(s.cpu().numpy(), s_ref)
    assert np.array_equal(q.cpu().numpy()[finite], q_ref[finite])


# rows of each expert, and whether every token also goes to one more
COUNTS = [([1], False), ([0, 1, 15, 16, 0, 3, 9, 0], False), ([17, 0, 32, 31, 1, 2, 0, 0, 0, 16], False), ([33, 48, 47, 0, 16, 1], False),
          ([49, 0, 0, 64, 5, 8], False), ([65, 128, 1, 0, 0, 7, 0, 0, 0, 0, 0, 0, 2], False), ([33, 48, 7, 0, 16, 2, 25, 0], True),
          ([100, 64, 65, 63], False), ([300, 129, 128, 1], False), ([1, 260, 2], True), ([192, 193, 64, 65], False)]


@pytest.mark.parametrize("N,K_", [(48, 1536), (272, 1544), (528, 2048), (784, 72), (1040, 2056)])
@pytest.mark.parametrize("counts,shared", COUNTS)
def test_experts_at_the_edges_of_their_tiles(counts, shared, N, K_):
    """Every kernel for the experts' products, each activation with its inputs gathered and weighed or as they lie."""
    from nanoflow_amd import kernels as K
    T, e, bf16 = sum(counts), len(counts), torch.bfloat16
    gen = torch.Generator(device="cuda").manual_seed(T + N + K_)
    randn = lambda *s: torch.randn(s, generator=gen, device="cuda")
    of = torch.repeat_interleave(torch.arange(e, device="cuda"), torch.tensor(counts, device="cuda"))[torch.randperm(T, generator=gen, device="cuda")]
    z = torch.full((1, T, (e + 7) // 8 * 8), -1.0, device="cuda")
    z[0, torch.arange(T), of] = 2.0
    n, groups = T * (1 + shared), e + shared
    r, t = K.route(z, e, e, 1, None, 1.5, K.lib().nf_grouped_tile_rows(K.BF16, n, groups), always=int(shared), scores=K.SCORES_SIGMOID, always_plain=True)
    offsets = t["offsets"].tolist()
    assert [b - a for a, b in zip(offsets, offsets[1:])] == counts + [T] * shared
    h, w = randn(T, K_).to(bf16), (randn(groups, N, K_) * K_ ** -0.5).to(bf16)
    tokens = t["row_of"].long()
    for act, gather, weigh in ((K.ACT_NONE, False, False), (K.ACT_GELU, True, False), (K.ACT_SQUARED_RELU, True, True), (K.ACT_GATED, True, True)):
        a = h if gather else h[tokens].contiguous()
        d = torch.full((n, N // 2 if act == K.ACT_GATED else N), 9.0, dtype=bf16, device="cuda")
        K.gemm_grouped_experts(a, w, d, r, n, gather, act, weigh=weigh, gated=(1.7, 1.0, None))
        for g in range(groups):
            rows = slice(offsets[g], offsets[g + 1])
            x = h[tokens[rows]].double()
            scale = t["row_weight"][rows].double()[:, None] if weigh else 1.0
            p = x @ w[g].double().t() * scale
            lost = K_ * 2.0 ** -24 * (x.abs() @ w[g].double().abs().t()) * scale + 2.0 ** -23 * p.abs()
            if act == K.ACT_GELU:
                want, lost = torch.nn.functional.gelu(p), 1.13 * lost
            elif act == K.ACT_SQUARED_RELU:
                want, lost = p.clamp(min=0) ** 2, 2 * p.abs() * lost + lost ** 2
            elif act == K.ACT_GATED:
                gate, up = p[:, ::2], p[:, 1::2] + 1.0
                want = gate * torch.sigmoid(1.7 * gate) * up
                lost = 1.2 * lost[:, ::2] * up.abs() + gate.abs() * lost[:, 1::2]  # 1.2: the gate's largest slope
            else:
                want = p
            bound = 2.0 ** -8 * want.abs() + lost + 2.0 ** -18
            assert bool(((d[rows].double() - want).abs() <= bound).all()), (g, act, float(((d[rows].double() - want).abs() / bound).max()))
