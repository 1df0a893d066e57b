"""The order of the routed rows by expert, at the edges of what one workgroup places: whole numbers and copied weights, so exact."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,experts,identity,top,always", [(1, 3, 0, 1, 0), (255, 5, 2, 3, 1), (2047, 32, 8, 5, 0), (3276, 33, 0, 4, 1), (4096, 7, 0, 3, 1), (4096, 40, 3, 4, 0),
                                                           (4097, 40, 3, 4, 0), (273, 100, 20, 58, 2), (16384, 2, 0, 1, 0), (5462, 3, 1, 1, 2), (1024, 32, 0, 3, 1), (4097, 9, 0, 1, 0), (8200, 5, 0, 4, 1)])
def test_rows_by_expert(T, experts, identity, top, always):
    from nanoflow_amd import kernels as K
    outputs, per = experts + identity, top + always
    z = torch.from_numpy(np.random.default_rng(T).standard_normal((1, T, (outputs + 8) // 8 * 8)).astype(np.float32)).cuda()
    if identity and always:
        identity, outputs = 0, experts  # experts of every token come behind the outputs
    r, t = K.route(z, outputs, experts, top, None, 1.5, 64, always=always)
    get = lambda k: t[k].cpu().numpy()
    choice, place, weight = get("choice").reshape(T, per), get("place").reshape(T, per), get("weight").reshape(T, per)
    assert (choice[:, top:] == outputs + np.arange(always)).all()
    group = np.where(choice < experts, choice, np.where(np.arange(per) >= top, experts + np.arange(per) - top, -1))
    counts = np.bincount(group[group >= 0], minlength=experts + always)
    offsets = get("offsets")
    np.testing.assert_array_equal(np.diff(offsets), counts)
    assert ((place == -1) == (group < 0)).all()
    token, k = np.nonzero(group >= 0)
    at = place[token, k]
    assert (np.sort(at) == np.arange(counts.sum())).all()
    assert ((offsets[group[token, k]] <= at) & (at < offsets[group[token, k] + 1])).all()
    np.testing.assert_array_equal(get("row_of")[at], token)
    np.testing.assert_array_equal(get("row_weight")[at], weight[token, k])


PLACES = [{"place": "choice"}, {"place": "weight"}]
SORTED = [{"row_of": "choice", "row_weight": "weight"}, {"place": "weight", "row_of": "choice"}]    # up to 16384 entries


@pytest.mark.parametrize("T,experts,top,always,shared", [(*size, shared) for size in [(3, 4, 2, 0), (700, 9, 5, 0), (2047, 32, 5, 1), (3276, 33, 5, 0), (4100, 6, 3, 1)]
                                                         for shared in (PLACES + SORTED if size[0] * (size[2] + size[3]) <= 16384 else PLACES)])
def test_arrays_that_share_memory(T, experts, top, always, shared):
    """Places over the choices or weights of any number of entries, sorted rows over them up to 16384: the same plan as in arrays of their own."""
    import ctypes as C

    from nanoflow_amd import kernels as K
    n = T * (top + always)
    z = torch.from_numpy(np.random.default_rng(T).standard_normal((1, T, (experts + 8) // 8 * 8)).astype(np.float32)).cuda()
    _, own = K.route(z, experts, experts, top, None, 1.5, 64, always=always)
    t = {k: torch.full_like(v, -7) for k, v in own.items()}
    for out, source in shared.items():
        t[out] = t[source].view(t[out].dtype)
    r = K.Routing(tile_rows=64, **{k: v.data_ptr() for k, v in t.items()})
    a = K.RouteArgs(z=z.data_ptr(), shares=1, ld=z.shape[2], rows=T, outputs=experts, experts=experts, top=top, always=always, groups=1, keep_groups=1, scale=1.5)
    K._call("nf_route", C.byref(a), C.byref(r), K._stream())
    get = lambda d, k: d[k].cpu().numpy()
    for k in ("offsets", "n_tiles"):
        np.testing.assert_array_equal(get(t, k), get(own, k))
    tiles = int(own["n_tiles"].item())
    for k in ("tile_group", "tile_row"):
        np.testing.assert_array_equal(get(t, k)[:tiles], get(own, k)[:tiles])
    # inside an expert's run the order is free: as sets of (expert, token, weight), and every place leads to its token
    assert get(own, "offsets")[-1] == n
    expert = np.searchsorted(get(own, "offsets")[1:], np.arange(n), side="right")
    rows = lambda d: sorted(zip(expert.tolist(), get(d, "row_of").tolist(), get(d, "row_weight").tolist()))
    assert rows(t) == rows(own)
    place = get(t, "place")
    assert (np.sort(place) == np.arange(n)).all()
    np.testing.assert_array_equal(get(t, "row_of")[place], np.arange(n) // (top + always))
    np.testing.assert_array_equal(expert[place], expert[get(own, "place")])
