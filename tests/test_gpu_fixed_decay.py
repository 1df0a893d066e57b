"""Recurrences under a fixed decay in 16-bit matrix instructions (csrc/kernels/recurrence_fixed.h) against float64, and against the general form, which
rows that are no multiple of 16 bytes apart take.  An output may be off by its one rounding to bf16 and by fp32 sums of a chunk's 128 + 128 terms,
a state by fp32 sums and the decays' exponents: both far below 4e-6 of the largest."""
import ctypes as C

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
D = 128


def run(qkv, state, reqs, decay, k_scale, out_scale, pad):
    """(outputs, states) with rows 3 heads * D + pad elements apart: a pad of 4 takes the general form."""
    from nanoflow_amd import kernels as K
    T, heads = qkv.shape[0], qkv.shape[2]
    rows = torch.zeros((T, 3 * heads * D + pad), dtype=torch.bfloat16, device="cuda")
    rows[:, :3 * heads * D] = qkv.reshape(T, -1)
    out = torch.full((T, heads * D + 8), 9.0, dtype=torch.bfloat16, device="cuda")
    st = state.clone()
    i32 = lambda a: torch.from_numpy(np.ascontiguousarray(a, dtype=np.int32)).cuda()
    lens = [n for _, n in reqs]
    indptr, slots = i32(np.concatenate([[0], np.cumsum(lens)])), i32(np.arange(len(reqs))[::-1])
    pos = i32(np.concatenate([np.arange(p, p + n) for p, n in reqs]))
    log2 = torch.tensor(decay, dtype=torch.float64).log2().float().cuda()
    need = K.lib().nf_recurrence_workspace_bytes(heads, D, D, T, len(reqs))
    ws = torch.full((max(need, 16),), 0x7f, dtype=torch.uint8, device="cuda")
    at = lambda i: rows.data_ptr() + 2 * i * heads * D
    a = K.RecurrenceArgs(dtype=K.BF16, kind=K.FIXED_DECAY, heads=heads, dim=D, vdim=D, eps=1e-5, state=st.data_ptr(), out=out.data_ptr(), out_ld=out.shape[1],
                         out_col=8, input_indptr=indptr.data_ptr(), positions=pos.data_ptr(), state_slots=slots.data_ptr(), total_rows=T,
                         workspace=ws.data_ptr(), workspace_bytes=need, q=at(0), k=at(1), v=at(2), q_ld=rows.shape[1], k_ld=rows.shape[1], v_ld=rows.shape[1],
                         k_scale=k_scale, log2_decay=log2.data_ptr(), out_scale=out_scale, req_begin=0, req_num=len(reqs), row_begin=0, rows=T)
    assert K.lib().nf_linear_recurrence(C.byref(a), torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    assert (out[:, :8] == 9.0).all()
    return out[:, 8:].float().view(T, heads, D), st


def wanted(qkv, state, reqs, decay, k_scale, out_scale):
    T, heads = qkv.shape[0], qkv.shape[2]
    out, st, first = torch.empty((T, heads, D), dtype=torch.float64, device="cuda"), state.double(), 0
    log2 = torch.tensor(decay, dtype=torch.float64).log2().float().double().cuda()[:, None, None]
    for r, (p, n) in enumerate(reqs):
        q, k, v = qkv[first:first + n].double().permute(1, 2, 0, 3).contiguous()
        k, s, i = k * k_scale, st[len(reqs) - 1 - r] * (p > 0), torch.arange(n, device="cuda")
        back = i[:, None] - i[None, :]
        scores = (q @ k.transpose(1, 2).contiguous()) * torch.exp2(log2 * back.clamp(min=0)) * (back >= 0)
        out[first:first + n] = ((scores @ v + (q * torch.exp2(log2 * (i + 1)[:, None])) @ s) * out_scale).transpose(0, 1)
        st[len(reqs) - 1 - r] = torch.exp2(log2 * n) * s + (k * torch.exp2(log2 * (n - 1 - i)[:, None])).transpose(1, 2).contiguous() @ v
        first += n
    return out, st


def operands(reqs, heads, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    T = sum(n for _, n in reqs)
    qkv = torch.randn((T, 3, heads, D), generator=g, device="cuda").bfloat16()
    return qkv, torch.randn((len(reqs), heads, D, D), generator=g, device="cuda")


# rows at the edges of a wavefront's 16 tokens, of halves of chunks and of chunks; the last runs on whole chunks for more heads than CUs
@pytest.mark.parametrize("reqs,heads", [([(0, 24)], 1), ([(5, 31)], 2), ([(0, 63), (9, 64), (0, 65)], 2), ([(0, 127)], 1), ([(3, 128)], 1), ([(1, 129), (0, 24)], 3),
                                        ([(0, 193)], 1), ([(7, 256), (0, 257)], 2), ([(0, 700), (11, 130)], 1), ([(2, 100), (0, 140)], 150)], ids=str)
@pytest.mark.parametrize("decay", [(0.97, 1.0), (1e-6, 0.5)])
def test_against_float64_and_the_general_form(reqs, heads, decay):
    qkv, state = operands(reqs, heads)
    d = np.linspace(*decay, heads)
    for k_scale, out_scale in ((1.0, 1.0), (0.31, 0.5)):
        want, left = wanted(qkv, state, reqs, d, k_scale, out_scale)
        top, tall = want.abs().amax((0, 2))[None, :, None], left.abs().max()
        for pad in (0, 4):
            got, st = run(qkv, state, reqs, d, k_scale, out_scale, pad)
            assert bool(((got.double() - want).abs() <= 2.0 ** -8 * want.abs() + 4e-6 * top).all()), pad
            assert float((st.double() - left).abs().max() / tall) < 4e-6, pad


@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
@pytest.mark.parametrize("row", [0, 40, 100, 150])
def test_what_is_not_finite_stays_with_its_tokens(bad, row):
    """Tokens of earlier sixteens do not see a value that is not finite, a state that is not finite is seen by all."""
    qkv, state = operands([(4, 200)], 1)
    qkv[row, 2, 0, 5] = bad
    got, st = run(qkv, state, [(4, 200)], [0.9], 1.0, 1.0, 0)
    clean, _ = run(qkv.nan_to_num(0, 0, 0), state, [(4, 200)], [0.9], 1.0, 1.0, 0)
    assert torch.equal(got[:row // 16 * 16], clean[:row // 16 * 16])
    assert not got[row:, 0, 5].isfinite().any() and got[:, 0, :5].isfinite().all() and not st[0, 0, :, 5].isfinite().any() and st[0, 0, :, :5].isfinite().all()
    qkv, state = operands([(4, 200)], 1)
    state[0, 0, 3, 5] = bad
    qkv[:, 0] = qkv[:, 0].abs() + 1
    got, _ = run(qkv, state, [(4, 200)], [0.9], 1.0, 1.0, 0)
    assert bool((got[:, 0, 5].isnan() if bad != bad else got[:, 0, 5] == bad).all()) and got[:, 0, :5].isfinite().all()


@pytest.mark.parametrize("bad", [float("inf"), float("-inf")])
@pytest.mark.parametrize("row", [0, 16, 50, 96, 127, 130, 199])      # 16, 96: the first of sixteen; 127, 199: a chunk's last, whose key the state takes undecayed
@pytest.mark.parametrize("what", ["q", "k", "v", "state"])
@pytest.mark.parametrize("k_scale", [1.0, 0.31])
def test_infinities_are_those_of_the_general_form(what, row, bad, k_scale):
    """Operands of eight significant bits or fewer beside them: all of q, k and v, and every fourth column of the state.  What is finite may differ by the bounds of
    both forms."""
    reqs, heads = [(4, 200)], 2
    qkv, state = operands(reqs, heads)
    state[:, :, :, ::4] = state[:, :, :, ::4].bfloat16().float()
    if what == "state":
        state[0, 1, row % D, 5] = bad
    else:
        qkv[row, "qkv".index(what), 1, 5] = bad
    got, st = run(qkv, state, reqs, [0.9, 0.97], k_scale, 0.5, 0)
    want, left = run(qkv, state, reqs, [0.9, 0.97], k_scale, 0.5, 4)
    assert not want.isfinite().all()
    for x, y, off in ((got, want, 2.0 ** -7), (st, left, 0.0)):
        assert torch.equal(x[y.isinf()], y[y.isinf()]) and torch.equal(x.isfinite(), y.isfinite())
        ok = y.isfinite()
        assert bool(((x[ok] - y[ok]).abs() <= off * y[ok].abs() + 8e-6 * y[ok].abs().max()).all())


def test_a_nan_of_its_lowest_bit_is_no_infinity():
    qkv, state = operands([(4, 40)], 1)
    state.view(torch.int32)[0, 0, 3, 5] = 0x7f800001
    got, st = run(qkv, state, [(4, 40)], [0.9], 1.0, 1.0, 0)
    assert got[:, 0, 5].isnan().all() and st[0, 0, 3, 5].isnan() and got[:, 0, :5].isfinite().all()
