"""The greedy sampler over columns at the edges of a thread's loads: whole numbers and bytes, so exact."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def literal(x):
    """(column, value's bits) of a row: the largest above -10000, NaN aside; of equals the one whose bits of column mod 1024 are
    smallest from the last to the first, then the smallest column."""
    v = x.view(np.float16).astype(np.float32)
    if not (v > -10000).any():
        return 0, np.float16(-10000).view(np.uint16)
    cols = np.nonzero(v == np.nanmax(np.where(np.isnan(v), -np.inf, v)))[0]
    best = min(cols.tolist(), key=lambda c: (int(f"{c % 1024:010b}"[::-1], 2), c))
    return best, x[best]


@pytest.mark.parametrize("cols", [8, 1016, 8184, 8192, 8200, 65528, 65536, 65544, 128256, (1 << 20) - 8])
def test_argmax_of_halves(cols):
    from nanoflow_amd import kernels as K
    rng = np.random.default_rng(cols)
    rows = [rng.standard_normal(cols), np.round(rng.standard_normal(cols)), np.zeros(cols), np.full(cols, -20000.0), np.full(cols, -np.inf),
            np.full(cols, np.nan), np.full(cols, -3.0)]
    x = np.stack(rows).astype(np.float16).view(np.uint16)
    x[0, rng.integers(0, cols, 3)] = [0x7e00, 0x7d01, 0xfe00]                     # quiet and signalling NaN
    x[2, rng.integers(0, cols, cols // 2)] = 0x8000                               # -0 equals 0
    x[3, -1] = 0xf0e1                                                             # -9992, the smallest that wins
    x[5, cols // 2] = 0xfbff if cols > 8 else 0x0001
    x[6, [0, -1]] = 0x7c00
    arg, value = K.argmax(torch.from_numpy(x.view(np.float16).copy()).cuda())
    want = [literal(r) for r in x]
    assert arg.cpu().tolist() == [int(w[0]) for w in want]
    assert value.cpu().numpy().view(np.uint16).tolist() == [int(w[1]) for w in want]
