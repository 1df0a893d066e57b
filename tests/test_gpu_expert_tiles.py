"""Products of routed experts over small whole numbers: every sum is exact in fp32 whatever its order, so the results are those of
integer arithmetic, rounded once.  Experts with no row, one, a few more than a tile's and several tiles; contractions of one slab of
64 and a few, of whole slabs and not; columns that end inside a tile."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

FEW = (0, 1, 16, 33, 49, 64, 65)                       # tile lists of 64 rows
MANY = (0, 129, 1, 300, 128, 96, 257, 511, 32)         # of 128


def routing(K, counts, tile, rows, rng):
    """Rows of the tokens in the order of their experts, and the tile list."""
    e, slots = len(counts), int(sum(counts))
    i32 = lambda a: torch.from_numpy(np.ascontiguousarray(a, dtype=np.int32)).cuda()
    tiles = [(g, r) for g in range(e) for r in range(0, counts[g], tile)]
    room = K.lib().nf_routing_max_tiles(slots, e, tile)
    assert len(tiles) <= room
    pad = [(0, 0)] * (room - len(tiles))
    row_of = rng.integers(0, rows, slots)
    weight = rng.integers(1, 4, slots).astype(np.float32)
    t = dict(row_of=i32(row_of), offsets=i32(np.concatenate([[0], np.cumsum(counts)])), tile_group=i32([g for g, _ in tiles + pad]),
             tile_row=i32([r for _, r in tiles + pad]), n_tiles=i32([len(tiles)]), row_weight=torch.from_numpy(weight).cuda())
    return K.Routing(tile_rows=tile, **{k: v.data_ptr() for k, v in t.items()}), t, row_of, weight


@pytest.mark.parametrize("counts", [FEW, MANY], ids=["lists of 64", "lists of 128"])
@pytest.mark.parametrize("N,Kd", [(8, 64), (136, 72), (256, 128), (264, 200), (520, 1000), (1032, 2048), (2048, 2056), (1024, 2112), (1048, 2184), (512, 3000), (2192, 2048)])
def test_whole_numbers(counts, N, Kd):
    check(counts, N, Kd, torch.full((len(counts),), 7.0))


@pytest.mark.parametrize("N,Kd", [(8192, 2112), (12288, 2184), (16384, 2112), (8192, 2048), (12240, 2048)])
def test_workgroups_that_go_from_tile_to_tile(N, Kd):
    """Two to four tiles a workgroup, of other experts, heights and first slabs, the last one cut in its columns or its contraction."""
    tiles = sum((n + 127) // 128 for n in MANY) * ((N + 255) // 256)
    assert tiles >= 2 * torch.cuda.get_device_properties(0).multi_processor_count
    check(MANY, N, Kd, torch.linspace(0.5, 4.0, len(MANY)))


@pytest.mark.parametrize("counts", [(0, 1, 16, 20, 0, 10, 65), (3, 0, 65, 0, 0), (0, 0, 0, 5)], ids=str)
@pytest.mark.parametrize("N,Kd", [(520, 1600), (1032, 2048), (2048, 1544)])
def test_last_expert_first(counts, N, Kd):
    """Few rows an expert, for this depth, and at most 30: the weight stream goes through the experts from the last one on."""
    assert N >= 512 and sum(counts) <= min(30, 16 + (Kd - 1536) * 24 // 512) * len(counts)
    check(counts, N, Kd, torch.full((len(counts),), 7.0))


@pytest.mark.parametrize("counts", [(64, 65, 1, 0, 20), (64, 65, 2, 0, 20)], ids=["30 rows an expert", "more"])
def test_either_order_of_experts(counts):
    """The most rows of which the last expert comes first, and a row more, of which the first one does."""
    check(counts, 1032, 2048, torch.full((len(counts),), 7.0))


def check(counts, N, Kd, limits):
    from nanoflow_amd import kernels as K
    rng = np.random.default_rng(N + Kd)
    counts = np.array(counts)
    e, slots, rows = len(counts), int(counts.sum()), 300
    tile = K.lib().nf_grouped_tile_rows(K.BF16, slots, e)
    assert tile == (128 if max(counts) > 65 else 64)
    r, hold, row_of, weight = routing(K, counts, tile, rows, rng)
    a, b = rng.integers(-2, 3, (rows, Kd), dtype=np.int8), rng.integers(-2, 3, (e, N, Kd), dtype=np.int8)
    gather, given = torch.from_numpy(a).cuda(), torch.from_numpy(a[row_of]).cuda().bfloat16()
    w = torch.from_numpy(b).cuda()
    group = np.repeat(np.arange(e), counts)
    product = torch.cat([gather[row_of[group == g]].double() @ w[g].double().T for g in range(e)])      # whole numbers below 2^24
    bf16 = lambda x: x.float().bfloat16()
    gather, w = gather.bfloat16(), w.bfloat16()

    def run(act, source, out, **kw):
        d = torch.full((slots, out), 9.0, dtype=torch.bfloat16, device="cuda")
        K.gemm_grouped_experts(source, w, d, r, slots, source is gather, act, **kw)
        return d

    assert torch.equal(run(K.ACT_NONE, gather, N), bf16(product))
    assert torch.equal(run(K.ACT_NONE, given, N), bf16(product))
    assert torch.equal(run(K.ACT_SQUARED_RELU, gather, N), bf16(product.clamp(min=0).float().square()))
    assert torch.equal(run(K.ACT_NONE, given, N, weigh=True), bf16(product * torch.from_numpy(weight).cuda()[:, None].double()))
    # gate and up, weighed first: all exact but the sigmoid (some 2^-20) and one rounding to bf16 (2^-9)
    x = product * torch.from_numpy(weight).cuda()[:, None].double() / 64
    limits = limits.cuda()
    scaled = (w.float() / 64).bfloat16()
    d = torch.full((slots, N // 2), 9.0, dtype=torch.bfloat16, device="cuda")
    if N // 2 % 8 == 0:
        K.gemm_grouped_experts(gather, scaled, d, r, slots, True, K.ACT_GATED, weigh=True, gated=(1.702, 1.0, limits))
        most = limits[torch.from_numpy(group).cuda()][:, None].double()
        g, u = x[:, 0::2].minimum(most), x[:, 1::2].clamp(-most, most)
        ref = g * torch.sigmoid(1.702 * g) * (u + 1.0)
        assert ((d.double() - ref).abs() <= 2 ** -8 * ref.abs()).all()


@pytest.mark.parametrize("counts,N,Kd", [((65, 96, 70, 80), 1536, 2048), ((72, 65, 90, 66), 256, 4096), ((300, 129, 65, 140), 520, 6144),
                                             ((70, 120, 128, 100, 129, 110, 75, 90), 2816, 2048)],
                         ids=["lists of 64", "lists of 64, 4096 deep", "lists of 128", "part of a round"])
def test_few_weights_are_walked_straight(counts, N, Kd):
    """Experts of less than 128 MB of weights begin at their first k however long a row of weights is, and are not chained where a round holds them: the
    bits of the plain product of their rows."""
    from nanoflow_amd import kernels as K
    rng = np.random.default_rng(N)
    counts = np.array(counts)
    slots, e = int(counts.sum()), len(counts)
    tile = K.lib().nf_grouped_tile_rows(K.BF16, slots, e)
    r, hold, row_of, _ = routing(K, counts, tile, 300, rng)
    gen = torch.Generator(device="cuda").manual_seed(Kd)
    a, w = (torch.randn(shape, generator=gen, device="cuda").bfloat16() for shape in ((300, Kd), (e, N, Kd)))
    d = torch.zeros((slots, N), dtype=torch.bfloat16, device="cuda")
    K.gemm_grouped_experts(a, w, d, r, slots, True)
    group = np.repeat(np.arange(e), counts)
    assert torch.equal(d, torch.cat([K.gemm_nk(a[row_of[group == g]].contiguous(), w[g]) for g in range(e)]))
