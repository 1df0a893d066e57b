"""The layer operators' wrappers tell a kernel one element type for several tensors: one of another type is refused before anything is launched, for the
kernel would read or write past its end.  (The launch itself is replaced; the tensors are on the CPU.)"""
import pytest

torch = pytest.importorskip("torch")
from nanoflow_amd import kernels as K

BF16, F32 = torch.bfloat16, torch.float32
OTHER = {BF16: F32, F32: BF16}


@pytest.fixture
def launched(monkeypatch):
    calls = []
    monkeypatch.setattr(K, "_call", lambda name, *args: calls.append((name, args)))
    monkeypatch.setattr(K, "_p", lambda t: None if t is None else t.data_ptr())
    monkeypatch.setattr(K, "_stream", lambda: 0)
    return calls


def z(*shape, dtype=F32):
    return torch.zeros(shape, dtype=dtype)


def test_a_table_without_activations_has_its_own_type(launched):
    for dtype, number in ((BF16, K.BF16), (F32, K.F32)):
        K.residual_rows(None, z(3, 16), None, 16, table=z(5, 16, dtype=dtype), tokens=z(3, dtype=torch.int32))
        assert launched[-1][1][0]._obj.dtype == number
    K.residual_rows(z(2, 3, 16), z(3, 16), None, 16)
    assert launched[-1][1][0]._obj.dtype == K.F32


def calls(t):
    """name -> (call over tensors by name, the tensors' types); t: the operands' type."""
    i32 = lambda *s: z(*s, dtype=torch.int32)
    kv, lat = K.KVLayout(K.BF16 if t == BF16 else K.F32, 2, 2, 32, 16, 32, 16, 16, 1), K.LatentLayout(K.BF16 if t == BF16 else K.F32, 2, 8, 8, 8, 64, 16)
    batch = {n: i32(2) for n in ("input_indptr", "kv_indptr", "kv_indices", "rev_input_indptr", "positions", "state_slots")}
    pages = [batch[n] for n in ("kv_indptr", "kv_indices", "rev_input_indptr", "positions")]
    return {
        "residual_rows": (lambda x, act, table, add: K.residual_rows(None, x, act, 16, table=table, tokens=i32(3), add=add), dict(x=F32, act=t, table=t, add=F32)),
        "mixture_rows": (lambda y, identity, x, act: K.mixture_rows(y, K.Routing(), 2, identity, x, act, 16), dict(y=t, identity=t, x=F32, act=t)),
        "norm": (lambda weight, bias: K.norm(K.NORM_LAYER, weight, bias), dict(weight=F32, bias=F32)),
        "gated_norm_rows": (lambda o, g, weight: K.gated_norm_rows(o, g, weight, 16, 1e-5), dict(o=t, g=t, weight=F32)),
        "gemm_nk": (lambda a, b, bias: K.gemm_nk(a, b, bias=bias), dict(a=t, b=t, bias=t)),
        "embed_rows": (lambda embed, pos: K.embed_rows(i32(3), i32(3), embed, pos), dict(embed=t, pos=t)),
        "gemm_grouped_heads": (lambda a, b, d: K.gemm_grouped_heads(a, b[None], d, 0, 0), dict(a=t, b=t, d=t)),
        "gemm_grouped_experts": (lambda a, b, d, limits: K.gemm_grouped_experts(a, b[None], d, K.Routing(), 3, True, gated=(1.0, 0.0, limits)), dict(a=t, b=t, d=t, limits=F32)),
        "token_shift": (lambda x, state, mu: K.token_shift(x, state, mu, i32(2), i32(3), i32(3), i32(1), t), dict(x=F32, state=F32, mu=F32)),
        "short_conv": (lambda weight, state: K.short_conv(weight, state, i32(2), i32(1)), dict(weight=t, state=t)),
        "qkv_append": (lambda proj, weight, pool: K.qkv_append(kv, proj, (0, 0, 0), weight, None, 1e-5, K.Rotation(), pool, *pages), dict(proj=t, weight=F32, pool=t)),
        "window_attention": (lambda q, pool, gate, sink: K.window_attention(kv, q, pool, batch, window=0, keep_first=0, scale=1.0, gate=gate, sink=sink),
                             dict(q=t, pool=t, gate=t, sink=F32)),
        "latent_append": (lambda proj, weight, q, pool: K.latent_append(lat, proj, (0, 0), weight, 1e-5, K.Rotation(), q, pool, batch), dict(proj=t, weight=F32, q=t, pool=t)),
        "latent_attention": (lambda q, pool: K.latent_attention(lat, q, pool, batch, scale=1.0), dict(q=t, pool=t)),
        "linear_recurrence": (lambda q, k, v, g, state, w: K.linear_recurrence(K.FIXED_DECAY, q, k, v, g, 1, 16, 16, state, batch, eps=1e-5, log2_decay=w, norm_weight=w),
                              dict(q=t, k=t, v=t, g=t, state=F32, w=F32)),
    }


@pytest.mark.parametrize("t", [BF16, F32], ids=str)
@pytest.mark.parametrize("name", sorted(calls(F32)))
def test_one_tensor_of_another_type_is_refused(launched, name, t):
    call, types = calls(t)[name]
    given = {n: z(3, 16, dtype=d) for n, d in types.items()}
    call(**given)
    after = len(launched)
    for n, d in types.items():
        with pytest.raises(TypeError):
            call(**{**given, n: given[n].to(OTHER[d])})
    assert len(launched) == after
