"""Decode attention with several workgroups on a request and kv head (csrc/kernels/attention.hip): bit for bit what one workgroup
gives, which a capped launch keeps."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("causal,rows", [(False, None), (True, [0, 3, 1, 0, 0, 2, 1, 0, 0])])
@pytest.mark.parametrize("batch,Hkv", [(1, 1), (1, 8), (7, 8), (8, 8), (9, 8), (16, 8), (3, 5), (64, 1), (65, 1), (21, 3), (43, 3)])
@pytest.mark.parametrize("group", [1, 2, 4, 8])
def test_shared_heads(group, batch, Hkv, causal, rows):
    from nanoflow_amd import kernels as K
    gen = torch.Generator().manual_seed(batch * 100 + Hkv * 10 + group)
    edges = [1, 15, 16, 17, 31, 32, 33, 63, 64, 65, 128, 129, 255, 257, 400, 1000]
    lengths = [edges[int(i)] for i in torch.randint(0, len(edges), (batch,), generator=gen)]
    rows = [1] * batch if rows is None else [min(r, n) for r, n in zip((rows * batch)[:batch], lengths)]
    pages = [(n + 15) // 16 for n in lengths]
    indptr = lambda c: torch.tensor([0] + c).cumsum(0).int().cuda()
    total = sum(pages)
    kv = torch.randn((total, 2, 16, Hkv, 128), generator=gen).half()
    where = torch.randperm(total, generator=gen)
    at = 0
    for n, p in zip(lengths, pages):                                    # behind a request's last key: not a number
        if n % 16:
            kv[where[at + p - 1], :, n % 16:] = float("nan")
        at += p
    q = torch.randn((max(sum(rows), 1), Hkv * group, 128), generator=gen).half().cuda()
    args = (q, indptr(rows), kv.cuda(), indptr(pages), where.int().cuda(), torch.tensor([(n - 1) % 16 + 1 for n in lengths]).int().cuda(),
            Hkv * group, Hkv)
    out = [K.attention_paged(*args, causal=causal, max_qo_rows=batch, num_blocks=b) for b in (0, 100000)]
    assert bool(torch.isfinite(out[1]).all()) and torch.equal(*out)
