"""Decoder layers as a serving iteration runs them, through the operators of nanoflow_amd.kernels: what a server spends its
time on, from one decoding request to a full 2048-token iteration.

A case is one layer of a model (or the head behind the last one) on a batch of requests that decode, portions of prompts,
or both.  As the serving pipelines do, the sequence of operators is recorded once and replayed from a graph for every
iteration of the same make-up; `prepare` holds what stays on the device (weights, paged cache, states, workspaces, the recorded
graph) and `run` is one replay.

  llama, llama-e4m3   a layer of the 8B shape (4096 wide, 32 query and 8 kv heads of 128, feed-forward 14336) in fp16, [N][K]
                      weights, or with fp8 weights
  head                the rows to be sampled: gather, norm, product with a vocabulary of 128256, argmax
  parallel            window attention beside a token-decay recurrence, dense squared-ReLU feed-forward         } 2048 wide, bf16,
  lightning, latent   fixed-decay recurrence / attention over latents, 32 GELU experts and 8 identity experts  } the layer-stack
  differential        difference of two attentions behind short convolutions, 32 experts in groups, a shared one } designs of the
  chunked             attention in chunks with turned values, 32 gated experts weighed at their input, a shared one } stack benchmark
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from nanoflow_amd import kernels as K
from nanoflow_amd import synth

PAGE = 16
KINDS = ("llama", "llama-e4m3", "head", "parallel", "lightning", "latent", "differential", "chunked")
# the 8B shape
H, HQ, HKV, D, FF, VOCAB, THETA = 4096, 32, 8, 128, 14336, 128256, 5e5
KQV = (HQ + 2 * HKV) * D
# the layer-stack designs
W, N, G, SFF = 2048, 16, 4, 8192            # width, heads of 128, kv heads, dense feed-forward
EXPERTS, EFF = 32, SFF // 4
RANK, ROT = 512, 64                         # of the latents
RN, RD, LORA = W // 64, 64, 64              # token-decay heads, their size, the decay's inner size
WINDOW, KEEP, CHUNK, CAP, DIFF = 512, 16, 1536, 30.0, 0.4
TABLE = 32768                               # embedding rows
POSITIONS = 4096
EPS = 1e-5
MOE = {"lightning": dict(identity=8, top=5, scale=2.0, act=K.ACT_GELU),
       "latent": dict(identity=8, top=5, scale=2.0, act=K.ACT_GELU),
       "differential": dict(top=4, groups=8, keep=4, always=1, act=K.ACT_SQUARED_RELU),
       "chunked": dict(top=4, always=1, act=K.ACT_GATED)}


# ---------------------------------------------------------------- cases

def listed():
    return [
        # one conversation: the time between two tokens, where every launch counts
        dict(name="one request", layer="llama", decode=1, context=1000, prompts=0, prompt=0, history=0),
        # a lightly loaded server
        dict(name="64 requests", layer="llama", decode=64, context=1024, prompts=0, prompt=0, history=0),
        # the offline benchmark's iteration: decoding requests beside the next ones' prompts in portions; the largest
        dict(name="serving iteration", layer="llama", decode=681, context=1535, prompts=3, prompt=484, history=400),
        # fp8 weights, few requests
        dict(name="fp8 16 requests", layer="llama-e4m3", decode=16, context=1024, prompts=0, prompt=0, history=0),
        # fp8 weights, prompts as they arrive
        dict(name="fp8 prompts", layer="llama-e4m3", decode=0, context=0, prompts=2, prompt=1001, history=0),
        # what every iteration ends in
        dict(name="head of 200", layer="head", decode=200, context=0, prompts=0, prompt=0, history=0),
        # the designs of the layer stack: decoding
        dict(name="parallel 64 requests", layer="parallel", decode=64, context=1024, prompts=0, prompt=0, history=0),
        dict(name="differential 256 requests", layer="differential", decode=256, context=777, prompts=0, prompt=0, history=0),
        # a prompt arrives where others are decoding
        dict(name="latent 48 and a prompt", layer="latent", decode=48, context=1500, prompts=1, prompt=700, history=300),
        # prompts: two of the benchmark's length, one that fills the iteration to an odd number, four short ones
        dict(name="parallel 2 prompts", layer="parallel", decode=0, context=0, prompts=2, prompt=1024, history=0),
        dict(name="lightning prompt", layer="lightning", decode=0, context=0, prompts=1, prompt=2047, history=0),
        dict(name="chunked 4 prompts", layer="chunked", decode=0, context=0, prompts=4, prompt=530, history=0),
    ]


def draw(rng):
    span = lambda lo, hi: int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    c = dict(layer=rng.choice(KINDS), decode=0, context=0, prompts=0, prompt=0, history=0)
    if c["layer"] == "head":
        c["decode"] = span(1, 700)
        return c
    what = rng.choice(("decode", "decode", "prompts", "both"))
    if what != "prompts":
        c["decode"], c["context"] = span(1, 256), span(32, 1535)
    if what != "decode":
        c["prompts"] = rng.randint(1, 4)
        c["prompt"] = span(16, (2048 - c["decode"]) // c["prompts"])
        c["history"] = rng.choice((0, 0, span(16, 1024)))
    return c


def requests(case):
    """(positions held before, rows brought) of the requests, decoding ones first; of uneven lengths."""
    decode = [(case["context"] - i * 37 % (case["context"] // 3 + 1), 1) for i in range(case["decode"])] if case["context"] else []
    return decode + [(case["history"] - j * 53 % (case["history"] // 2 + 1), case["prompt"] - j * 29 % (case["prompt"] // 4 + 1))
                     for j in range(case["prompts"])]


def rows_of(case):
    return case["decode"] if case["layer"] == "head" else sum(n for _, n in requests(case))


# ---------------------------------------------------------------- inputs

class Box:
    """A bag of named things."""

    def __init__(self, **kw):
        self.__dict__.update(kw)


def decays(heads):
    return [1.0 - 2.0 ** (-5 - 3.0 * h / heads) for h in range(heads)]


def turns(dims, base):
    """fp32 (cos, sin) pairs [positions, dims / 2, 2]."""
    angle = torch.arange(POSITIONS, dtype=torch.float64, device="cuda")[:, None] * base ** (-torch.arange(0, dims, 2, dtype=torch.float64, device="cuda") / dims)
    return torch.stack((angle.cos(), angle.sin()), -1).float().contiguous()


def inputs(case, seed):
    """Everything on the device, from the seed alone: weights of the usual scales, caches and states as earlier iterations
    would have left them."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kind, T = case["layer"], rows_of(case)
    s = Box(case=case, kind=kind, T=T)
    half = torch.float16 if kind in ("llama", "llama-e4m3", "head") else torch.bfloat16

    def normal(*shape, std=1.0, mean=0.0, dtype=half):
        return torch.empty(shape, dtype=dtype, device="cuda").normal_(mean, std, generator=gen)

    weight = lambda *shape: normal(*shape, std=shape[-1] ** -0.5)
    f32 = lambda *shape, std=0.1, mean=1.0: normal(*shape, std=std, mean=mean, dtype=torch.float32)
    i32 = lambda a: torch.from_numpy(np.ascontiguousarray(a, dtype=np.int32)).cuda()
    if kind == "head":
        # the rows behind the last layer: every request's last row is sampled
        s.rows, s.norm, s.head = normal(T, H), normal(H, std=0.1, mean=1.0), weight(VOCAB, H)
        s.indptr = i32(np.arange(T + 1))
        return s
    held = requests(case)
    b = synth.make_batch([p for p, n in held[:case["decode"]]], held[case["decode"]:], TABLE, seed=seed)
    s.requests, s.decode, s.pages = held, case["decode"], b.num_pages
    s.tokens, s.indptr, s.rev, s.positions = i32(b.input_tokens), i32(b.input_indptr), i32(b.rev_input_indptr), i32(b.per_token_offset)
    s.kv_indptr, s.kv_indices, s.kv_last = i32(b.kv_indptr), i32(b.kv_indices), i32(b.kv_last_page_len)
    s.page_lists = [b.kv_indices[b.kv_indptr[r]:b.kv_indptr[r + 1]] for r in range(len(held))]
    s.slots = i32(np.random.default_rng(seed).permutation(len(held)))
    if kind.startswith("llama"):
        s.table = normal(TABLE, H)
        s.norm1, s.norm2 = normal(H, std=0.1, mean=1.0), normal(H, std=0.1, mean=1.0)
        s.kqv, s.o, s.gate, s.up, s.down = weight(KQV, H), weight(H, HQ * D), weight(FF, H), weight(FF, H), weight(H, FF)
        if kind == "llama-e4m3":
            for name in ("kqv", "o", "gate", "up", "down"):
                setattr(s, name, quantised(getattr(s, name)))
        s.kv = normal(s.pages, 2, PAGE, HKV, D)
        return s
    # a layer of the stack
    s.table = normal(TABLE, W)
    moe = MOE.get(kind)
    if moe:
        e = EXPERTS + moe.get("always", 0)
        s.router = weight(40, W)        # rows beyond the outputs and the gate of the shared expert stay unused
        s.eup = weight(e, EFF * (2 if kind == "chunked" else 1), W)
        s.edown = weight(e, W, EFF)
        if "identity" in moe:
            s.correction = f32(EXPERTS + moe["identity"], std=0.02, mean=0.0)
        if kind == "chunked":
            s.limits = torch.full((e,), 7.0, device="cuda")
    else:
        s.up, s.down = weight(SFF, W), weight(W, SFF)
    for name in ("norm1", "norm2"):
        setattr(s, name, f32(W))
        setattr(s, name + "b", f32(W, mean=0.0))
    if kind in ("parallel", "differential", "chunked"):
        s.layout = K.kv_layout(half, N, G, 64 if kind == "differential" else D, D, 2 if kind == "differential" else 1)
        s.kv = normal(s.pages, K.lib().nf_kv_page_elements(C.byref(s.layout)))
        s.qkv = weight((N + 2 * G) * D, W)
    if kind == "parallel":
        s.pos = normal(POSITIONS, W, std=0.1)
        s.qnorm, s.knorm, s.sink, s.rot = f32(D), f32(D), f32(N, std=0.5, mean=0.0), turns(D, 1e4)
        s.mu = torch.rand((5, W), generator=gen, device="cuda")
        s.rkvg = [weight(RN * RD, W) for _ in range(4)]
        s.w1, s.w2 = weight(LORA, W), weight(RN * RD, LORA)
        s.w0 = torch.rand((RN * RD,), generator=gen, device="cuda") * 6 - 7
        s.u, s.rnorm = f32(RN * RD, std=0.5, mean=0.0), f32(RN * RD)
        s.state, s.shift = f32(len(held), RN, RD, RD, std=1.0, mean=0.0), f32(len(held), W, std=1.0, mean=0.0)
        s.out = weight(W, N * D + RN * RD)
    elif kind == "lightning":
        s.qkv, s.g, s.out, s.gnorm = weight(3 * N * D, W), weight(N * D, W), weight(W, N * D), f32(N * D)
        s.log2 = torch.tensor(decays(N), dtype=torch.float64).log2().float().cuda()
        s.state = f32(len(held), N, D, D, std=1.0, mean=0.0)
    elif kind == "latent":
        s.lay = K.latent_layout(half, N, RANK, ROT)
        s.proj = weight(N * (D + ROT) + RANK + ROT, W)
        s.uk, s.uv = weight(N, D, RANK), weight(N, D, RANK)
        s.to_latent = s.uk.transpose(1, 2).contiguous()                     # [heads][rank][dim]
        s.expand = torch.cat((s.uk.reshape(-1, RANK), s.uv.reshape(-1, RANK))).contiguous()
        s.lnorm, s.rot, s.out = f32(RANK), turns(ROT, 1e4), weight(W, N * D)
        s.kv = normal(s.pages, PAGE, s.lay.row_ld)
        s.kv[..., RANK + ROT:] = 0
    elif kind == "differential":
        s.conv_w, s.conv = normal(4, s.qkv.shape[0], std=0.5), normal(len(held), 3, s.qkv.shape[0])
        s.rot, s.out = turns(64, 5e5), weight(W, N * D)
    elif kind == "chunked":
        s.qnorm, s.knorm, s.sink = f32(D), f32(D), f32(N, std=0.5, mean=0.0)
        s.rot, s.vrot, s.out = turns(64, 5e5), turns(D, 5e5), weight(W, N * D)
    return s


def quantised(w):
    """(e4m3 bytes [N, K], fp32 scale per row) of fp16 weights."""
    scale = w.float().abs().amax(1) / 448.0
    return (w.float() / scale[:, None]).to(torch.float8_e4m3fn).view(torch.uint8), scale


# ---------------------------------------------------------------- the path

def do(name, *args):
    rc = getattr(K.lib(), name)(*args, torch.cuda.current_stream().cuda_stream)
    if rc != 0:
        raise RuntimeError(f"{name}: {K.lib().nf_last_error().decode()}")


def llama_layer(s):
    T, nd, np_ = s.T, s.decode, s.case["prompts"]
    f8 = s.kind == "llama-e4m3"
    x = K.embedding(s.tokens, s.table)
    if f8:
        _, hq, hs = K.rmsnorm_quantize_e4m3(x, s.norm1, EPS)
        kqv = K.gemm_f8q(hq, hs, *s.kqv)
    else:
        kqv, _ = K.gemm_ws(K.rmsnorm(x, s.norm1, EPS), s.kqv, b_col_major=True)
    q = K.rope_append(kqv, s.kv, s.kv_indices, s.kv_indptr, s.rev, s.positions, HQ, HKV, rope_theta=THETA)
    a = torch.empty_like(q)

    def attend(first, n, rows, causal):
        K.attention_paged(q, s.indptr[first:first + n + 1], s.kv, s.kv_indptr[first:first + n + 1], s.kv_indices, s.kv_last[first:first + n],
                          HQ, HKV, causal=causal, out=a, batch=n, max_qo_rows=rows)

    main = torch.cuda.current_stream()
    if np_ and nd:          # the prompts' attention beside the decode attention
        s.side.wait_stream(main)
        with torch.cuda.stream(s.side):
            attend(nd, np_, T - nd, True)
        attend(0, nd, nd, False)
        main.wait_stream(s.side)
    else:
        attend(0, nd or np_, T, nd == 0)
    if f8:
        o = K.gemm_f8w(a, *s.o, Cmat=x, beta=1.0)
        _, hq, hs = K.rmsnorm_quantize_e4m3(o, s.norm2, EPS)
        y = K.gemm_f8w(K.dual_swiglu_f8q(hq, hs, *s.gate, *s.up), *s.down, Cmat=o, beta=1.0)
    else:
        o, _ = K.gemm_ws(a, s.o, Cmat=x, beta=1.0, b_col_major=True)
        f, _ = K.dual_swiglu_ws(K.rmsnorm(o, s.norm2, EPS), s.gate, s.up, b_col_major=True)
        y, _ = K.gemm_ws(f, s.down, Cmat=o, beta=1.0, b_col_major=True)
    return {"x": y, "kv": s.kv}


def head(s):
    rows = K.keep_token(s.rows, s.indptr, s.T)
    logits, _ = K.gemm_ws(K.rmsnorm(rows, s.norm, EPS), s.head, b_col_major=True)
    _, top = K.argmax(logits)
    return {"logits": logits, "top": top}


def product(s, a, w, **kw):
    need = max(K.lib().nf_gemm_nk_workspace_bytes_upto(a.shape[0], *w.shape), 16)
    return K.gemm_nk(a, w, workspace=torch.empty((need,), dtype=torch.uint8, device="cuda"), **kw)


def back(s, a, w):
    """A projection to the residual width, for the operator that ends a sublayer: fp32 sums where it is split over K or the rows
    are few."""
    if s.T > 512 and K.lib().nf_gemm_nk_sums_shares(s.T, *w.shape, 16) < 2:
        return K.gemm_nk(a, w)
    return K.gemm_nk_sums(a, w, 16)


def groups_of(s):
    """(first request, requests, first row, rows, decode) of the two launches of an operator over requests."""
    nd, n = s.decode, len(s.requests)
    return [g for g in ((0, nd, 0, nd, 1), (nd, n - nd, nd, s.T - nd, 0)) if g[1]]


def attention(s, layout, q, kv, indices, out, parts, rot=None, **kw):
    a = K.WindowAttentionArgs(kv=layout, out_rot=rot or K.Rotation(), out_scale=1.0, q=q.data_ptr(), out=out.data_ptr(), out_ld=out.shape[1],
                              kv_data=kv.data_ptr(), input_indptr=s.indptr.data_ptr(), kv_indptr=s.kv_indptr.data_ptr(), kv_indices=indices.data_ptr(),
                              rev_input_indptr=s.rev.data_ptr(), positions=s.positions.data_ptr(), **kw)
    for a.req_begin, a.req_num, a.row_begin, a.max_rows, a.decode in parts:
        do("nf_window_attention", C.byref(a))


def recurrence(s, kind, heads, d, out, **kw):
    need = K.lib().nf_recurrence_workspace_bytes(heads, d, d, s.T, len(s.requests))
    ws = torch.empty((max(need, 16),), dtype=torch.uint8, device="cuda")
    a = K.RecurrenceArgs(dtype=K.BF16, kind=kind, heads=heads, dim=d, vdim=d, eps=EPS, state=s.state.data_ptr(), out=out.data_ptr(), out_ld=out.shape[1],
                         input_indptr=s.indptr.data_ptr(), positions=s.positions.data_ptr(), state_slots=s.slots.data_ptr(), total_rows=s.T,
                         workspace=ws.data_ptr(), workspace_bytes=need, **kw)
    for a.req_begin, a.req_num, a.row_begin, a.rows, _ in groups_of(s):
        do("nf_linear_recurrence", C.byref(a))


def append(s, rot, qnorm=None, knorm=None, **kw):
    return K.qkv_append(s.layout, product(s, s.act, s.qkv), (0, N * D, (N + G) * D), qnorm, knorm, EPS, K.rotation(rot, rot.shape[1] * 2, True),
                        s.kv, s.kv_indptr, s.kv_indices, s.rev, s.positions, **kw)


def parallel_mixer(s):
    heads = torch.empty((s.T, N * D + RN * RD), dtype=torch.bfloat16, device="cuda")
    main = torch.cuda.current_stream()
    s.side.wait_stream(main)
    with torch.cuda.stream(s.side):     # two mixers that read the same rows
        attention(s, s.layout, append(s, s.rot, s.qnorm, s.knorm), s.kv, s.kv_indices, heads, groups_of(s), window=WINDOW, keep_first=KEEP,
                  scale=D ** -0.5, sink=s.sink.data_ptr())
    mixed = K.token_shift(s.x, s.shift, s.mu, s.indptr, s.rev, s.positions, s.slots, torch.bfloat16)
    r, k, v, g = (product(s, mixed[i], s.rkvg[i]) for i in range(4))
    z = K.gemm_nk_sums(K.tanh_rows(K.gemm_nk_sums(mixed[4], s.w1, 16), torch.bfloat16), s.w2, 1)
    ld = RN * RD
    recurrence(s, K.TOKEN_DECAY, RN, RD, heads, q=r.data_ptr(), k=k.data_ptr(), v=v.data_ptr(), g=g.data_ptr(), q_ld=ld, k_ld=ld, v_ld=ld, g_ld=ld,
               z=z.data_ptr(), z_ld=ld, z_shares=1, w0=s.w0.data_ptr(), u=s.u.data_ptr(), norm_weight=s.rnorm.data_ptr(), out_scale=0.5, out_col=N * D,
               shift_x=s.x.data_ptr(), shift_state=s.shift.data_ptr(), shift_ld=W)
    main.wait_stream(s.side)
    return heads


def lightning_mixer(s):
    heads = torch.empty((s.T, N * D), dtype=torch.bfloat16, device="cuda")
    qkv, g = product(s, s.act, s.qkv, act=K.ACT_SILU), product(s, s.act, s.g)
    at = lambda i: qkv.data_ptr() + 2 * i * N * D
    recurrence(s, K.FIXED_DECAY, N, D, heads, q=at(0), k=at(1), v=at(2), q_ld=3 * N * D, k_ld=3 * N * D, v_ld=3 * N * D, k_scale=1.0,
               log2_decay=s.log2.data_ptr(), out_scale=1.0)
    K.gated_norm_rows(heads, g, s.gnorm, N * D, EPS)
    return heads


def latent_mixer(s):
    new = lambda *shape: torch.empty(shape, dtype=torch.bfloat16, device="cuda")
    T, nd, lay, scale = s.T, s.decode, s.lay, (D + ROT) ** -0.5
    heads, proj = new(T, N * D), product(s, s.act, s.proj)
    q, rot = new(max(nd, 1), N, lay.row_ld), K.rotation(s.rot, ROT, True)
    do("nf_latent_append", C.byref(lay), proj.data_ptr(), proj.shape[1], N * D, N * (D + ROT), s.lnorm.data_ptr(), EPS, C.byref(rot), q.data_ptr(),
       s.kv.data_ptr(), s.kv_indptr.data_ptr(), s.kv_indices.data_ptr(), s.rev.data_ptr(), s.positions.data_ptr(), T, nd)
    if nd < T:              # prompts: keys and values of all heads written out
        first = int(s.first_page)
        pages = (s.last_page - first + 63) // 64 * 64
        kv = K.kv_layout(torch.bfloat16, N, N, D + ROT, D)
        rows, ids, packed = new(pages * PAGE, RANK), torch.empty_like(s.kv_indices), new(pages, K.lib().nf_kv_page_elements(C.byref(kv)))
        a = K.LatentExpandArgs(layout=lay, kv=kv, dim_pad=D, kv_data=s.kv.data_ptr(), kv_indptr=s.kv_indptr.data_ptr(), kv_indices=s.kv_indices.data_ptr(),
                               req_begin=nd, req_end=len(s.requests), max_pages=pages, rows=rows.data_ptr(), page_ids=ids.data_ptr(),
                               ld=2 * N * D, k_col=0, v_col=N * D, pages=packed.data_ptr())
        do("nf_latent_gather", C.byref(a))
        products = product(s, rows, s.expand)
        a.products = products.data_ptr()
        do("nf_latent_pack", C.byref(a))
        qp = new(T, N, kv.k_pad)
        do("nf_latent_queries", C.byref(kv), D, proj.data_ptr(), proj.shape[1], N * D, ROT, C.byref(rot), s.positions.data_ptr(), qp.data_ptr(), nd, T - nd)
        attention(s, kv, qp, packed, ids, heads, [g for g in groups_of(s) if not g[4]], scale=scale)
    if nd:                  # decoding: over the latents
        K.gemm_grouped_heads(proj[:nd], s.to_latent, q.view(nd, -1), D, lay.row_ld)
        out = new(nd, N, RANK)
        ws = torch.empty((max(K.lib().nf_latent_workspace_bytes(C.byref(lay), nd), 16),), dtype=torch.uint8, device="cuda")
        a = K.LatentAttentionArgs(layout=lay, scale=scale, q=q.data_ptr(), out=out.data_ptr(), kv_data=s.kv.data_ptr(), input_indptr=s.indptr.data_ptr(),
                                  kv_indptr=s.kv_indptr.data_ptr(), kv_indices=s.kv_indices.data_ptr(), rev_input_indptr=s.rev.data_ptr(),
                                  positions=s.positions.data_ptr(), req_begin=0, req_num=nd, row_begin=0, max_rows=nd, decode=1,
                                  workspace=ws.data_ptr(), workspace_bytes=ws.numel())
        do("nf_latent_attention", C.byref(a))
        K.gemm_grouped_heads(out.view(nd, -1), s.uv, heads[:nd], RANK, D)
    return heads


def attention_mixer(s):
    heads = torch.empty((s.T, N * D), dtype=torch.bfloat16, device="cuda")
    if s.kind == "differential":
        q = append(s, s.rot, conv=K.short_conv(s.conv_w, s.conv, s.indptr, s.slots))
        attention(s, s.layout, q, s.kv, s.kv_indices, heads, groups_of(s), window=WINDOW, scale=64 ** -0.5, softcap=CAP, map_weight=DIFF, head_norm=1,
                  head_eps=EPS)
    else:
        turn = K.rotation(s.vrot, D, True)
        q = append(s, s.rot, s.qnorm, s.knorm, value_norm=True, value_rot=turn)
        attention(s, s.layout, q, s.kv, s.kv_indices, heads, groups_of(s), turn, chunk=CHUNK, scale=D ** -0.5, sink=s.sink.data_ptr())
    return heads


def mixture(s, next_norm, y_norm):
    m, T = MOE[s.kind], s.T
    always, per, e = m.get("always", 0), m["top"] + m.get("always", 0), EXPERTS + m.get("always", 0)
    outputs, slots = EXPERTS + m.get("identity", 0), T * per
    z = K.gemm_nk_sums(s.act, s.router, 16)
    tile = K.lib().nf_grouped_tile_rows(K.BF16, slots, e)
    i32 = lambda n: torch.empty((n,), dtype=torch.int32, device="cuda")
    f32 = lambda n: torch.empty((n,), dtype=torch.float32, device="cuda")
    tiles = K.lib().nf_routing_max_tiles(slots, e, tile)
    t = dict(choice=i32(slots), weight=f32(slots), place=i32(slots), row_of=i32(slots), offsets=i32(e + 1), tile_group=i32(tiles), tile_row=i32(tiles),
             n_tiles=i32(1))
    weigh = s.kind == "chunked"
    if weigh:
        t["row_weight"] = f32(slots)
    r = K.Routing(tile_rows=tile, **{k: v.data_ptr() for k, v in t.items()})
    a = K.RouteArgs(z=z.data_ptr(), shares=z.shape[0], ld=z.shape[2], rows=T, outputs=outputs, experts=EXPERTS, top=m["top"], always=always,
                    groups=m.get("groups", 1), keep_groups=m.get("keep", 1), correction=s.correction.data_ptr() if "identity" in m else None,
                    scale=m.get("scale", 1.0), scores=K.SCORES_SIGMOID if weigh else K.SCORES_SOFTMAX, always_plain=int(weigh))
    do("nf_route", C.byref(a), C.byref(r))
    mid, out = (torch.empty((slots, n), dtype=torch.bfloat16, device="cuda") for n in (EFF, W))
    K.gemm_grouped_experts(s.act, s.eup, mid, r, slots, True, m["act"], weigh=weigh, gated=(1.702, 1.0, s.limits) if weigh else (1.0, 0.0, None))
    K.gemm_grouped_experts(mid, s.edown, out, r, slots, False)
    K.mixture_rows(out, r, per, s.act if "identity" in m else None, s.x, s.act, W, next_norm, y_norm=y_norm, plain=weigh)
    s.hold = (t, mid, out, z)


def stack_layer(s):
    rms = lambda w: K.norm(K.NORM_RMS, w, None, EPS)
    layer = lambda w, b: K.norm(K.NORM_LAYER, w, b, EPS)
    if s.kind == "parallel":        # sublayers add their normed output
        s.x, s.act = K.embed_rows(s.tokens, s.positions, s.table, s.pos)
        K.residual_rows(back(s, parallel_mixer(s), s.out), s.x, s.act, W, rms(s.norm1))
        K.residual_rows(back(s, product(s, s.act, s.up, act=K.ACT_SQUARED_RELU), s.down), s.x, s.act, W, rms(s.norm2))
        return {"x": s.x, "act": s.act, "kv": s.kv, "state": s.state, "shift": s.shift}
    pre = layer if s.kind in ("lightning", "latent") else (lambda w, b: rms(w))
    s.x, _ = K.embed_rows(s.tokens, s.positions, s.table, None)
    s.act = K.norm_rows(s.x, None, pre(s.norm1, s.norm1b), W, torch.bfloat16)
    heads = {"lightning": lightning_mixer, "latent": latent_mixer}.get(s.kind, attention_mixer)(s)
    after = rms(s.norm1b) if s.kind == "chunked" else None           # a norm behind the sublayer, scaled per column
    K.residual_rows(back(s, heads, s.out), s.x, s.act, W, after, pre(s.norm2, s.norm2b))
    mixture(s, pre(s.norm1, s.norm1b), rms(s.norm2b) if s.kind == "chunked" else None)
    own = {"lightning": ("state",), "differential": ("kv", "conv")}.get(s.kind, ("kv",))
    return {"x": s.x, "act": s.act, **{n: getattr(s, n) for n in own}}


def layer(s):
    return head(s) if s.kind == "head" else llama_layer(s) if s.kind.startswith("llama") else stack_layer(s)


def prepare(case, seed):
    s = inputs(case, seed)
    s.side = torch.cuda.Stream()
    if s.kind == "latent":
        s.first_page, s.last_page = sum(map(len, s.page_lists[:s.decode])), sum(map(len, s.page_lists))
    carried = {n: getattr(s, n).clone() for n in ("state", "shift", "conv") if hasattr(s, n)}
    layer(s)                            # loads the kernels
    for n, t in carried.items():
        getattr(s, n).copy_(t)
    torch.cuda.synchronize()
    s.graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(s.graph):
        s.outputs = layer(s)
    return s


def run(state):
    state.graph.replay()
    return state.outputs


# ---------------------------------------------------------------- what a pass cannot do without

def seen(case, position):
    """Positions that a row at `position` attends to."""
    kind = case["layer"]
    if kind in ("parallel", "differential"):
        return min(position + 1, WINDOW + (KEEP if kind == "parallel" else 0))
    return position % CHUNK + 1 if kind == "chunked" else position + 1


def work(case):
    kind, T = case["layer"], rows_of(case)
    if kind == "head":
        return {"bytes": VOCAB * H * 2 + T * (H * 4 + VOCAB * 2), "flops": 2 * T * VOCAB * H}
    held = requests(case)
    pairs = sum(seen(case, p + i) for p, n in held for i in range(n))
    read = sum(min(p, seen(case, p + n - 1) + n) for p, n in held)      # cached positions
    if kind.startswith("llama"):
        weights = H * KQV + HQ * D * H + 3 * H * FF
        return {"bytes": weights * (1 if kind == "llama-e4m3" else 2) + read * 2 * HKV * D * 2 + T * (2 * H + 2 * HKV * D) * 2,
                "flops": 2 * T * weights + pairs * HQ * D * 4}
    moe = MOE.get(kind)
    per_token, stored, cached, attend = 0, 0, 0, 0
    if kind in ("parallel", "differential", "chunked"):
        per_token += W * (N + 2 * G) * D
        cached, attend = 2 * G * D * 2, N * D * (6 if kind == "differential" else 4)
    if kind == "parallel":
        per_token += W * (4 * RN * RD + LORA) + LORA * RN * RD + W * RN * RD + 2 * RN * RD * RD
        stored += len(held) * RN * RD * RD * 4 * 2
    elif kind == "lightning":
        per_token += W * 4 * N * D + 2 * N * D * D
        stored += len(held) * N * D * D * 4 * 2
    elif kind == "latent":
        per_token += W * (N * (D + ROT) + RANK + ROT) + 2 * N * D * RANK
        cached, attend = (RANK + ROT) * 2, N * (2 * D + ROT) * 2
    per_token += W * N * D
    weights = per_token - {"parallel": 2 * RN * RD * RD, "lightning": 2 * N * D * D}.get(kind, 0)
    if moe:
        expert = W * EFF * (3 if kind == "chunked" else 2)
        outputs = EXPERTS + moe.get("identity", 0)
        per_token += W * outputs + expert * (moe["top"] * EXPERTS / outputs + moe.get("always", 0))
        weights += W * outputs + expert * (EXPERTS * (1 - (1 - moe["top"] / outputs) ** T) + moe.get("always", 0))
    else:
        per_token += 2 * W * SFF
        weights += 2 * W * SFF
    return {"bytes": 2 * weights + stored + read * cached + T * (cached + W * (2 + 4 + 2)), "flops": 2 * T * per_token + pairs * attend}


def tolerance(case):
    # About four times one layer's rounding, measured against `exact`: fp16 4e-4, logits 3e-4, bf16 4.5e-3, a mixture 8e-3 (a token
    # whose choice is close may go to another expert); with fp8 weights the activations are rounded to e4m3 (2.5e-2 off `exact`, which
    # does not round them; less between two that do).
    return {"llama": {"rel": 0.002}, "head": {"rel": 0.0012}, "llama-e4m3": {"rel": 0.02}, "parallel": {"rel": 0.015}}.get(case["layer"], {"rel": 0.02})


# ---------------------------------------------------------------- the same in 64 bits

def d64(t):
    return t.double()


def rms64(x, w=None, dim=-1):
    y = x / (x.square().mean(dim, keepdim=True) + EPS).sqrt()
    return y if w is None else y * d64(w)


def norm64(s, x, w, b):
    if s.kind in ("lightning", "latent"):
        x = x - x.mean(-1, keepdim=True)
        return rms64(x, w) + d64(b)
    return rms64(x, w)


def times(x, w):
    """x . w^T, the weights widened a part at a time."""
    return torch.cat([x @ d64(p).t() for p in w.split(16384)], -1)


def turned(x, table, positions, back=False):
    """x [T, heads, d]: neighbours 2i, 2i + 1 of the first columns turned by the table's angles."""
    n = table.shape[1] * 2
    c, s = (d64(table[positions.long(), :, i])[:, None] for i in (0, 1))
    s = -s if back else s
    u, v = x[..., 0:n:2], x[..., 1:n:2]
    return torch.cat((torch.stack((u * c - v * s, v * c + u * s), -1).flatten(-2), x[..., n:]), -1)


def attend64(q, k, v, positions, scale, mask=None, sink=None, cap=0.0):
    """q [n, heads, d], k [L, kv heads, d], v [L, kv heads, e] -> [n, heads, e]."""
    L, per = k.shape[0], q.shape[1] // k.shape[1]
    i, j = positions.long()[:, None], torch.arange(L, device="cuda")[None]
    see = (j <= i) if mask is None else (j <= i) & mask(i, j)
    out = torch.empty((q.shape[0], q.shape[1], v.shape[2]), dtype=torch.float64, device="cuda")
    for g in range(k.shape[1]):
        z = torch.matmul(q[:, g * per:(g + 1) * per].transpose(0, 1), k[:, g].t().contiguous()) * scale     # [per, n, L]
        z = cap * torch.tanh(z / cap) if cap else z
        z = z.masked_fill(~see, -math.inf)
        top = z.amax(-1, keepdim=True)
        if sink is not None:
            top = torch.maximum(top, d64(sink)[g * per:(g + 1) * per, None, None])
        p = (z - top).exp()
        den = p.sum(-1, keepdim=True)
        if sink is not None:
            den = den + (d64(sink)[g * per:(g + 1) * per, None, None] - top).exp()
        out[:, g * per:(g + 1) * per] = torch.matmul(p / den, v[:, g].contiguous()).transpose(0, 1)
    return out


def by_request(s, q, k, v, cache, store, one):
    """For each request: its cached (k, v), the new rows behind them, `one`(q, k, v, positions); new rows go to the cache."""
    out, at = [], 0
    for r, (held, n) in enumerate(s.requests):
        rows = slice(at, at + n)
        at += n
        pages = torch.from_numpy(s.page_lists[r].astype(np.int64)).cuda()
        old_k, old_v = cache(pages)
        kk, vv = torch.cat((old_k[:held], k[rows])), torch.cat((old_v[:held], v[rows]))
        where = torch.arange(held, held + n, device="cuda")
        store(pages[where // PAGE], where % PAGE, k[rows], v[rows])
        out.append(one(q[rows], kk, vv, s.positions[rows]))
    return torch.cat(out)


def llama64(s):
    f8 = s.kind == "llama-e4m3"
    if f8:
        wide = lambda w: d64(w[0].view(torch.float8_e4m3fn).float()) * d64(w[1])[:, None]
        mul = lambda x, w: x @ wide(w).t()
    else:
        mul = times
    x, pool = d64(s.table[s.tokens.long()]), d64(s.kv)
    kqv = mul(rms64(x, s.norm1), s.kqv)
    k, v, q = (t.reshape(s.T, -1, D) for t in kqv.split((HKV * D, HKV * D, HQ * D), 1))

    def rope(t):
        angle = d64(s.positions)[:, None, None] * THETA ** (-torch.arange(0, D, 2, dtype=torch.float64, device="cuda") / D)
        u, w = t[..., :D // 2], t[..., D // 2:]
        return torch.cat((u * angle.cos() - w * angle.sin(), w * angle.cos() + u * angle.sin()), -1)

    def store(pages, rows, kk, vv):
        pool[pages, 0, rows], pool[pages, 1, rows] = kk, vv

    a = by_request(s, rope(q), rope(k), v, lambda p: (pool[p, 0].flatten(0, 1), pool[p, 1].flatten(0, 1)), store,
                   lambda q, k, v, p: attend64(q, k, v, p, D ** -0.5))
    o = x + mul(a.flatten(1), s.o)
    h = rms64(o, s.norm2)
    gate = mul(h, s.gate)
    return {"x": o + mul(gate * torch.sigmoid(gate) * mul(h, s.up), s.down), "kv": pool}


def paged64(s, q, k, v, maps, one):
    """Attention over the stack's pages: keys [kv heads][maps][16][dim], values [kv heads][vdim][16]."""
    d = s.layout.k_pad
    cut = G * maps * PAGE * d
    pool = d64(s.kv)
    pk, pv = pool[:, :cut].view(-1, G, maps, PAGE, d), pool[:, cut:].view(-1, G, D, PAGE)

    def cache(p):
        return pk[p].permute(0, 3, 1, 2, 4).reshape(-1, G, maps * d), pv[p].permute(0, 3, 1, 2).reshape(-1, G, D)

    def store(p, r, kk, vv):
        pk[p, :, :, r], pv[p, :, :, r] = kk.view(-1, G, maps, d), vv

    out = by_request(s, q, k.flatten(2) if maps > 1 else k, v, cache, store, one)
    return out, pool


def split_qkv(h, s):
    return (t.reshape(s.T, -1, D) for t in h.split((N * D, G * D, G * D), 1))


def parallel64(s, x):
    mask = lambda i, j: (i - j < WINDOW) | (j < KEEP)
    q, k, v = split_qkv(times(x, s.qkv), s)
    q, k = turned(rms64(q, s.qnorm), s.rot, s.positions), turned(rms64(k, s.knorm), s.rot, s.positions)
    left, pool = paged64(s, q, k, v, 1, lambda q, k, v, p: attend64(q, k, v, p, D ** -0.5, mask, s.sink))
    first = s.positions.new_zeros(s.T, dtype=torch.bool)
    first[s.indptr[:-1].long()] = True
    shift, state = d64(s.shift), d64(s.state)
    slot = s.slots.long()
    prev = torch.cat((x[:1], x[:-1]))
    prev[s.indptr[:-1].long()] = shift[slot]
    prev = torch.where((s.positions == 0)[:, None], torch.zeros_like(prev), prev)
    mixed = [x + (prev - x) * d64(m) for m in s.mu]
    r, k, v, g = (times(mixed[i], s.rkvg[i]) for i in range(4))
    decay = torch.exp(-torch.exp(times(torch.tanh(times(mixed[4], s.w1)), s.w2) + d64(s.w0))).view(s.T, RN, RD)
    r, k, v = (t.view(s.T, RN, RD) for t in (r, k, v))
    uk, o = d64(s.u).view(RN, RD) * k, torch.empty_like(r)

    def step(S, t):
        o[t] = (S * r[t][..., None]).sum(-2) + (r[t] * uk[t]).sum(-1, keepdim=True) * v[t]
        return decay[t][..., None] * S + k[t][..., None] * v[t][..., None, :]

    if s.decode:
        rows = torch.arange(s.decode, device="cuda")
        old = torch.where((s.positions[:s.decode] == 0).view(-1, 1, 1, 1), 0.0, state[slot[:s.decode]])
        state[slot[:s.decode]] = step(old, rows)
    at = s.decode
    for i, (held, n) in enumerate(s.requests[s.decode:], s.decode):
        S = state[slot[i]] if held else torch.zeros_like(state[0])
        for t in range(at, at + n):
            S = step(S, t)
        state[slot[i]] = S
        at += n
    shift[slot] = x[s.indptr[1:].long() - 1]
    right = (rms64(o).flatten(1) * d64(s.rnorm)) * (g * torch.sigmoid(g))
    return torch.cat((left.flatten(1), 0.5 * right), 1), {"kv": pool, "state": state, "shift": shift}


def lightning64(s, h):
    qkv = times(h, s.qkv)
    q, k, v = ((t * torch.sigmoid(t)).view(s.T, N, D).transpose(0, 1) for t in qkv.split(N * D, 1))     # [N, T, D]
    state, out, at = d64(s.state), torch.empty((N, s.T, D), dtype=torch.float64, device="cuda"), 0
    log = d64(s.log2)[:, None]
    for i, (held, n) in enumerate(s.requests):
        rows, t = slice(at, at + n), torch.arange(n, device="cuda")
        at += n
        slot = int(s.slots[i])
        S = state[slot] if held else torch.zeros_like(state[0])
        for head in range(N):
            fade = torch.where(t[:, None] >= t, torch.exp2(log[head] * (t[:, None] - t)), 0.0)
            kk, vv, qq = k[head, rows], v[head, rows], q[head, rows]
            out[head, rows] = (qq @ kk.t() * fade) @ vv + torch.exp2(log[head] * (t + 1))[:, None] * (qq @ S[head])
            state[slot, head] = torch.exp2(log[head] * n) * S[head] + (kk * torch.exp2(log[head] * (n - 1 - t))[:, None]).t() @ vv
    o = out.transpose(0, 1).reshape(s.T, N * D)
    return rms64(o, s.gnorm) * torch.sigmoid(times(h, s.g)), {"state": state}


def latent64(s, h):
    q, qr, latent, kr = times(h, s.proj).split((N * D, N * ROT, RANK, ROT), 1)
    latent = rms64(latent, s.lnorm)
    qr, kr = turned(qr.view(s.T, N, ROT), s.rot, s.positions), turned(kr[:, None], s.rot, s.positions)[:, 0]
    pool = d64(s.kv)

    def store(p, r, kk, vv):
        pool[p, r, :RANK], pool[p, r, RANK:RANK + ROT] = vv, kk

    def one(q, kr, c, p):       # the heads' keys and values written out
        kk = torch.cat((torch.matmul(c, d64(s.uk).transpose(1, 2).contiguous()), kr[None].expand(N, -1, -1)), -1).transpose(0, 1)
        vv = torch.matmul(c, d64(s.uv).transpose(1, 2).contiguous()).transpose(0, 1)
        return attend64(q, kk, vv, p, (D + ROT) ** -0.5)

    o = by_request(s, torch.cat((q.view(s.T, N, D), qr), -1), kr, latent, lambda p: (pool[p].flatten(0, 1)[:, RANK:RANK + ROT], pool[p].flatten(0, 1)[:, :RANK]),
                   store, one)
    return o.flatten(1), {"kv": pool}


def differential64(s, h):
    raw, conv = times(h, s.qkv), d64(s.conv)
    mixed, at = torch.empty_like(raw), 0
    for i, (held, n) in enumerate(s.requests):
        slot = int(s.slots[i])
        before = [conv[slot, p % 3] if p >= 0 else torch.zeros_like(raw[0]) for p in range(held - 3, held)]
        line = torch.cat((torch.stack(before), raw[at:at + n]))
        mixed[at:at + n] = sum(line[j:j + n] * d64(s.conv_w[j]) for j in range(4))
        for p in range(max(held, held + n - 3), held + n):
            conv[slot, p % 3] = raw[at + p - held]
        at += n
    q, k, v = split_qkv(mixed, s)
    turn = lambda t: turned(t.reshape(s.T, -1, 64), s.rot, s.positions)
    mask = lambda i, j: i - j < WINDOW

    def one(q, k, v, p):
        q, k = q.view(-1, N, 2, 64), k.view(-1, G, 2, 64)
        a, b = (attend64(q[:, :, m], k[:, :, m], v, p, 64 ** -0.5, mask, None, CAP) for m in (0, 1))
        return rms64(a - DIFF * b)

    o, pool = paged64(s, turn(q), turn(k).view(s.T, G, 2, 64), v, 2, one)
    return o.flatten(1), {"kv": pool, "conv": conv}


def chunked64(s, h):
    q, k, v = split_qkv(times(h, s.qkv), s)
    q, k = turned(rms64(q, s.qnorm), s.rot, s.positions), turned(rms64(k, s.knorm), s.rot, s.positions)
    v = turned(rms64(v), s.vrot, s.positions)
    mask = lambda i, j: i // CHUNK == j // CHUNK
    o, pool = paged64(s, q, k, v, 1, lambda q, k, v, p: attend64(q, k, v, p, D ** -0.5, mask, s.sink))
    return turned(o, s.vrot, s.positions, back=True).flatten(1), {"kv": pool}


def mixture64(s, h):
    m = MOE[s.kind]
    always, outputs = m.get("always", 0), EXPERTS + m.get("identity", 0)
    z = times(h, s.router)
    score = torch.sigmoid(z[:, :outputs]) if s.kind == "chunked" else torch.softmax(z[:, :outputs], -1)
    by = score + d64(s.correction) if "identity" in m else score
    if "groups" in m:
        best = score.view(s.T, m["groups"], -1).amax(-1)
        shut = torch.ones_like(best, dtype=torch.bool).scatter_(1, best.topk(m["keep"], 1).indices, False)
        by = by.masked_fill(shut.repeat_interleave(outputs // m["groups"], 1), -math.inf)
    chosen = by.topk(m["top"], 1).indices
    weight = torch.zeros_like(score).scatter_(1, chosen, score.gather(1, chosen) * m.get("scale", 1.0))
    y = weight[:, EXPERTS:].sum(1, keepdim=True) * h if "identity" in m else torch.zeros_like(h)
    for e in range(EXPERTS + always):
        rows = torch.arange(s.T, device="cuda") if e >= EXPERTS else weight[:, e].nonzero()[:, 0]
        if not len(rows):
            continue
        w = weight[rows, e, None] if e < EXPERTS else torch.sigmoid(z[rows, outputs, None])
        a = h[rows] @ d64(s.eup[e]).t()
        if s.kind == "chunked":
            a = a * w if e < EXPERTS else a
            gate, up = a[:, 0::2].clamp(max=7.0), a[:, 1::2].clamp(-7.0, 7.0)
            y[rows] += (gate * torch.sigmoid(1.702 * gate) * (up + 1.0)) @ d64(s.edown[e]).t()
        else:
            a = torch.nn.functional.gelu(a) if "identity" in m else a.clamp(min=0).square()
            y[rows] += w * (a @ d64(s.edown[e]).t())
    return y


def stack64(s):
    x = d64(s.table[s.tokens.long()])
    if s.kind == "parallel":
        x = x + d64(s.pos[s.positions.long()])
        heads, kept = parallel64(s, x)
        x = x + rms64(times(heads, s.out), s.norm1)
        x = x + rms64(times(times(x, s.up).clamp(min=0).square(), s.down), s.norm2)
        return {"x": x, "act": x, **kept}
    mix = {"lightning": lightning64, "latent": latent64, "differential": differential64, "chunked": chunked64}[s.kind]
    heads, kept = mix(s, norm64(s, x, s.norm1, s.norm1b))
    y = times(heads, s.out)
    x = x + (rms64(y, s.norm1b) if s.kind == "chunked" else y)
    y = mixture64(s, norm64(s, x, s.norm2, s.norm2b))
    x = x + (rms64(y, s.norm2b) if s.kind == "chunked" else y)
    return {"x": x, "act": norm64(s, x, s.norm1, s.norm1b), **kept}


def exact(case, seed):
    s = inputs(case, seed)
    if s.kind == "head":
        logits = times(rms64(d64(s.rows), s.norm), s.head)
        return {"logits": logits, "top": logits.amax(1)}
    return llama64(s) if s.kind.startswith("llama") else stack64(s)
