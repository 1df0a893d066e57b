"""Choices of the router by rank (up to 64 outputs, one a lane: csrc/kernels/layer_router.hip) against the general form, which takes the same scores beside 64
outputs that cannot be chosen: the same choices and the same bits of every weight, whatever the scores are."""
import ctypes as C

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def route(z, correction, top, always, groups, keep, scores, plain):
    from nanoflow_amd import kernels as K
    shares, rows, ld = z.shape
    outputs = correction.shape[0]
    per, e = top + always, outputs + always
    i32 = lambda n: torch.full((n,), -7, dtype=torch.int32, device="cuda")
    tiles = K.lib().nf_routing_max_tiles(rows * per, e, 64)
    t = dict(choice=i32(rows * per), weight=torch.full((rows * per,), -7.0, device="cuda"), place=i32(rows * per), row_of=i32(rows * per), offsets=i32(e + 1),
             tile_group=i32(tiles), tile_row=i32(tiles), n_tiles=i32(1))
    r = K.Routing(tile_rows=64, **{k: v.data_ptr() for k, v in t.items()})
    a = K.RouteArgs(z=z.data_ptr(), shares=shares, ld=ld, rows=rows, outputs=outputs, experts=outputs, top=top, always=always, groups=groups, keep_groups=keep,
                    correction=correction.data_ptr(), scale=2.0, scores=scores, always_plain=int(plain))
    assert K.lib().nf_route(C.byref(a), C.byref(r), torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    return t["choice"].view(rows, per).cpu(), t["weight"].view(rows, per).cpu()


@pytest.mark.parametrize("outputs,top,groups,keep", [(1, 1, 1, 1), (7, 7, 1, 1), (32, 4, 8, 4), (32, 5, 32, 5), (40, 5, 4, 1), (63, 8, 9, 2), (64, 8, 1, 1),
                                                     (64, 6, 2, 1)])
@pytest.mark.parametrize("scores", ["softmax", "sigmoid"])
@pytest.mark.parametrize("shares,always,plain", [(1, 0, True), (3, 1, True), (16, 2, False)])
def test_ranks_and_the_general_form(outputs, top, groups, keep, scores, shares, always, plain):
    from nanoflow_amd import kernels as K
    kind = K.SCORES_SOFTMAX if scores == "softmax" else K.SCORES_SIGMOID
    g = torch.Generator(device="cuda").manual_seed(outputs * 100 + shares)
    rows, size = 37, outputs // groups
    extra = (64 + size - 1) // size * size          # whole groups of outputs that are never chosen
    z = torch.randn((shares, rows, outputs + 1), generator=g, device="cuda")
    odd = torch.rand((shares, rows, outputs + 1), generator=g, device="cuda")
    z[:, 8:16] = z[:, 8:16].round()                 # equal scores
    for row, bad in ((20, float("nan")), (22, float("inf")), (24, float("-inf"))):
        z[:, row:row + 2] = torch.where(odd[:, row:row + 2] < 0.2, torch.full_like(z[:, row:row + 2], bad), z[:, row:row + 2])
    z[:, 26] = float("nan")
    z[0, 27] = float("-inf")
    correction = torch.randn((outputs,), generator=g, device="cuda") * 0.1
    wide = torch.full((shares, rows, outputs + extra + 1), float("-inf"), device="cuda")
    wide[1:, :, outputs:-1] = 0
    wide[:, :, :outputs], wide[:, :, -1] = z[:, :, :outputs], z[:, :, -1]
    never = torch.cat((correction, torch.full((extra,), float("-inf"), device="cuda")))
    got, want = (route(a, b, top, always, m, keep, kind, plain) for a, b, m in ((z, correction, groups), (wide, never, groups + extra // size)))
    assert torch.equal(got[0][:, :top], want[0][:, :top]) and torch.equal(got[0][:, top:], want[0][:, top:] - extra)
    assert bool(((got[1] == want[1]) | (got[1].isnan() & want[1].isnan())).all())
