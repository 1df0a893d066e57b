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
