"""Rules that choose between two forms of a launch, where one of them once was much the slower: against the other form, on the same operands in turns.  The two
have the same bits."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def medians(calls, copies, turns=15):
    """Median time in us of each call(copy), taken in turns from graphs over all copies."""
    graphs = []
    for call in calls:
        call(0)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            for i in range(copies):
                call(i)
        graph.replay()
        graphs.append(graph)
    times = [[] for _ in calls]
    for _ in range(turns):
        for graph, taken in zip(graphs, times):
            begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            begin.record()
            graph.replay()
            end.record()
            torch.cuda.synchronize()
            taken.append(begin.elapsed_time(end) * 1e3 / copies)
    return [sorted(t)[turns // 2] for t in times]


# 256 x 256 tiles on four or eight wavefronts (a launch with a chosen tile has four): deep contractions of [K][N] weights on part of the chip
# take 1.11 to 1.14 of the time on eight
@pytest.mark.parametrize("M,N,Kd", [(1503, 6144, 14336), (1024, 10240, 8192)])
def test_deep_products_on_part_of_the_chip(M, N, Kd):
    from nanoflow_amd import kernels as K
    a, b = ([torch.randn(shape, device="cuda").half() for _ in range(6)] for shape in ((M, Kd), (Kd, N)))
    out = torch.empty((M, N), dtype=torch.float16, device="cuda")
    assert torch.equal(K.gemm(a[0], b[0]), K.gemm_tiled(a[0], b[0], (256, 256)))
    rule, four = medians([lambda i: K.gemm(a[i], b[i], out=out), lambda i: K.gemm_tiled(a[i], b[i], (256, 256), out=out)], 6)
    assert rule <= 1.06 * four, (rule, four)
