"""Recurrences whose decays depend on the token, 64 tokens at a time (csrc/kernels/recurrence_token.h), against float64, and against the general form, which
rows that are no multiple of 16 bytes apart take.  An output may be off by its one rounding to bf16 and by fp32 sums of a chunk's 64 + 64 terms, which the
norm divides by the outputs' size: 128 roundings of 2^-24 of terms some ten times that size; a state by fp32 sums and the decays' exponents."""
import ctypes as C

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
D = 64


def operands(reqs, heads, mean, seed=0, shares=2):
    g = torch.Generator(device="cuda").manual_seed(seed)
    T = sum(n for _, n in reqs)
    rn = lambda *s: torch.randn(s, generator=g, device="cuda")
    return dict(rkvg=rn(4, T, heads, D).bfloat16(), z=rn(shares, T, heads, D) * 0.7, w0=rn(heads, D) * 0.3 + mean, u=rn(heads, D), norm=rn(heads, D) * 0.1 + 1,
                state=rn(len(reqs), heads, D, D))


def run(s, reqs, gate, pad):
    """(outputs, states) with rows of the outputs heads * D + 8 + pad elements apart: a pad of 4 takes the general form."""
    from nanoflow_amd import kernels as K
    T, heads = s["rkvg"].shape[1:3]
    out = torch.full((T, heads * D + 8 + pad), 9.0, dtype=torch.bfloat16, device="cuda")
    st = s["state"].clone()
    i32 = lambda a: torch.from_numpy(np.ascontiguousarray(a, dtype=np.int32)).cuda()
    lens = [n for _, n in reqs]
    indptr, slots = i32(np.concatenate([[0], np.cumsum(lens)])), i32(np.arange(len(reqs))[::-1])
    pos = i32(np.concatenate([np.arange(p, p + n) for p, n in reqs]))
    need = K.lib().nf_recurrence_workspace_bytes(heads, D, D, T, len(reqs))
    ws = torch.full((max(need, 16),), 0x7f, dtype=torch.uint8, device="cuda")
    ld, at = heads * D, [x.data_ptr() for x in s["rkvg"]]
    a = K.RecurrenceArgs(dtype=K.BF16, kind=K.TOKEN_DECAY, heads=heads, dim=D, vdim=D, eps=1e-5, state=st.data_ptr(), out=out.data_ptr(), out_ld=out.shape[1],
                         out_col=8, input_indptr=indptr.data_ptr(), positions=pos.data_ptr(), state_slots=slots.data_ptr(), total_rows=T,
                         workspace=ws.data_ptr(), workspace_bytes=need, q=at[0], k=at[1], v=at[2], g=at[3] if gate else None, q_ld=ld, k_ld=ld, v_ld=ld, g_ld=ld,
                         z=s["z"].data_ptr(), z_ld=ld, z_shares=len(s["z"]), w0=s["w0"].data_ptr(), u=s["u"].data_ptr(),
                         norm_weight=s["norm"].data_ptr() if gate else None, out_scale=0.5, req_begin=0, req_num=len(reqs), row_begin=0, rows=T)
    assert K.lib().nf_linear_recurrence(C.byref(a), torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    assert (out[:, :8] == 9.0).all() and (pad == 0 or bool((out[:, 8 + ld:] == 9.0).all()))
    return out[:, 8:8 + ld].float().view(T, heads, D), st


def wanted(s, reqs, gate):
    r, k, v, g = s["rkvg"].double()
    out, left, t = torch.empty_like(r), s["state"].double(), 0
    w = (-torch.exp(s["z"].sum(0) + s["w0"]).double()).clamp(min=-126 * np.log(2.0)).exp()
    for i, (p, n) in enumerate(reqs):
        S = left[len(reqs) - 1 - i] * (p > 0)
        for t in range(t, t + n):
            out[t] = (r[t][:, :, None] * S).sum(1) + (r[t] * k[t] * s["u"]).sum(1, keepdim=True) * v[t]
            S = S * w[t][:, :, None] + k[t][:, :, None] * v[t][:, None, :]
        left[len(reqs) - 1 - i], t = S, t + 1
    if not gate:
        return out * 0.5, left
    return out * 0.5 / torch.sqrt((out * out).mean(-1, keepdim=True) + 1e-5) * s["norm"] * g * torch.sigmoid(g), left


# rows at the edges of a wavefront's 16 tokens and of chunks; decays that reach 2^-100 over 16 tokens never, in some channels, in all
@pytest.mark.parametrize("reqs,heads", [([(0, 24)], 1), ([(5, 31)], 2), ([(0, 63), (9, 64), (0, 65)], 2), ([(0, 33)], 1), ([(3, 128)], 1), ([(1, 129), (0, 24)], 3),
                                        ([(0, 193), (7, 48)], 5)], ids=str)
@pytest.mark.parametrize("mean", [-2.0, 1.0, 4.0])
@pytest.mark.parametrize("gate", [True, False])
def test_against_float64_and_the_general_form(reqs, heads, mean, gate):
    s = operands(reqs, heads, mean)
    want, left = wanted(s, reqs, gate)
    for pad in (0, 4):
        got, st = run(s, reqs, gate, pad)
        assert bool(((got.double() - want).abs() <= 2.0 ** -8 * want.abs() + 4e-5 * want.abs().max()).all()), pad
        assert float((st.double() - left).abs().max() / left.abs().max()) < 4e-6, pad


# more chunks than the scan requests at once, with a remainder, ahead of another request; the shares of the decays
@pytest.mark.parametrize("reqs", [[(0, 449), (7, 322)], [(5, 321), (0, 24), (64, 257)]], ids=str)
@pytest.mark.parametrize("shares", [1, 3])
def test_many_chunks(reqs, shares):
    s = operands(reqs, 2, -3.0, shares=shares)
    want, left = wanted(s, reqs, True)
    for pad in (0, 4):
        got, st = run(s, reqs, True, pad)
        assert bool(((got.double() - want).abs() <= 2.0 ** -8 * want.abs() + 4e-5 * want.abs().max()).all()), pad
        assert float((st.double() - left).abs().max() / left.abs().max()) < 4e-6, pad


@pytest.mark.parametrize("bad", [float("nan"), float("inf"), float("-inf")])
@pytest.mark.parametrize("row", [0, 21, 70])
def test_what_is_not_finite_stays_with_its_tokens(bad, row):
    """Tokens of earlier sixteens do not see a value that is not finite, other columns never; a decay that is not finite is the largest, or none."""
    reqs = [(4, 100)]
    s = operands(reqs, 1, -1.0)
    clean, _ = run(s, reqs, False, 0)
    s["rkvg"][2, row, 0, 5] = bad
    got, st = run(s, reqs, False, 0)
    assert torch.equal(got[:row // 16 * 16], clean[:row // 16 * 16])
    assert not got[row + 1:, 0, 5].isfinite().any() and got[:, 0, :5].isfinite().all() and not st[0, 0, :, 5].isfinite().any() and st[0, 0, :, :5].isfinite().all()
    s = operands(reqs, 1, -1.0)
    s["z"][1, row, 0, 7] = bad
    got, st = run(s, reqs, False, 0)
    want, left = run(s, reqs, False, 4)
    assert bool(((got - want).abs() <= 2.0 ** -7 * want.abs() + 4e-5 * want.abs().max()).all())
    assert float((st - left).abs().max() / left.abs().max()) < 4e-6


@pytest.mark.parametrize("bad", [float("inf"), float("-inf")])
@pytest.mark.parametrize("row", [0, 16, 40, 48, 63, 70, 99])      # 16, 48: the first of sixteen; 63, 99: a chunk's last, whose key the state takes undecayed
@pytest.mark.parametrize("what", ["q", "k", "v", "state"])
@pytest.mark.parametrize("gate", [False, True])
def test_infinities_are_those_of_the_general_form(gate, what, row, bad):
    """Operands of eight significant bits or fewer beside them: all of q, k and v, and every fourth column of the state.  What is finite may differ by the bounds of
    both forms."""
    reqs = [(4, 100)]
    s = operands(reqs, 2, -2.0)
    s["state"][:, :, :, ::4] = s["state"][:, :, :, ::4].bfloat16().float()
    if what == "state":
        s["state"][0, 1, row % D, 5] = bad
    else:
        s["rkvg"]["qkv".index(what), row, 1, 5] = bad
    got, st = run(s, reqs, gate, 0)
    want, left = run(s, reqs, gate, 4)
    assert not want.isfinite().all()
    for x, y, off in ((got, want, 2.0 ** -7), (st, left, 0.0)):
        assert torch.equal(x[y.isinf()], y[y.isinf()]) and torch.equal(x.isfinite(), y.isfinite())
        ok = y.isfinite()
        assert bool(((x[ok] - y[ok]).abs() <= off * y[ok].abs() + 8e-5 * y[ok].abs().max()).all())
