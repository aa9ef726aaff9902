"""Sums of one to four 4-byte values per entry through tiles of records (csrc/value_tiles.h) at the sizes where it can go wrong:
tiles of 1024 entries and their multiples, more tiles than a workgroup has lanes, a bucket of more entries than one round holds,
entries outside [0, N), batches, out given, counts for a mean. Sums of int32 are exact, floats against torch in 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
CASES = [("even", 1, 2048, 300), ("even", 1, 8191, 5), ("even", 1, 40961, 2000), ("even", 1, 100000, 3), ("hub", 1, 49150, 900),
         ("hub", 1, 60001, 4000), ("hub", 1, 1100000, 60000), ("outside", 1, 30001, 700), ("even", 3, 5000, 333),
         ("even", 1, 524289, 130000), ("even", 1, 4000000, 150001)]


def _index(kind, E, N, g):
    index = torch.randint(0, N, (E,), generator=g, device=DEV)
    if kind == "hub":
        index[torch.randperm(E, generator=g, device=DEV)[:E // 3]] = N // 3
    elif kind == "outside":
        index[::3] += N
        index[1::7] = -1 - index[1::7]
    return index


@pytest.mark.parametrize("K", [1, 2, 3, 4])
@pytest.mark.parametrize("kind,B,E,N", CASES)
def test_value_tiles(kind, B, E, N, K, monkeypatch):
    from pytorch_scatter_amd import capi
    monkeypatch.setenv("TS_SCATTER_BINNED", "2")
    g = torch.Generator(device=DEV).manual_seed(E + K)
    index = torch.stack([_index(kind, E, N, g) for _ in range(B)])
    ok = (index >= 0) & (index < N)
    rows = (index + torch.arange(B, device=DEV).view(B, 1) * N)[ok]
    for dtype in (torch.int32, torch.float32):
        src = torch.randint(-50, 51, (B, E, K), generator=g, device=DEV).to(dtype)
        given = torch.randint(-50, 51, (B, N, K), generator=g, device=DEV).to(dtype)
        if dtype == torch.float32:
            src, given = src + torch.randn(src.shape, generator=g, device=DEV), given + 0.5
        # (on the CPU: additions in 64 bits to one address take seconds on the device)
        total = torch.zeros((B * N, K), dtype=torch.float64).index_add_(0, rows.cpu(), src[ok].double().cpu()).to(DEV)
        size = torch.zeros((B * N, K), dtype=torch.float64).index_add_(0, rows.cpu(), src[ok].double().abs().cpu()).to(DEV)
        n = torch.bincount(rows, minlength=B * N)
        for out_given in (False, True):
            out, count = given.clone(), torch.full((B * N,), -3, dtype=torch.int32, device=DEV)
            capi.scatter_with_workspace(src, index, out, None, B, E, K, N, E, 1, 0, capi.SUM, out_given)
            want = total + given.view(B * N, K).double() if out_given else total
            # sums in 64 bits, rounded once; those of a large bucket once per 8192 entries and once more where these meet
            bound = 2 ** -24 * want.abs() + 1e-13 * size if dtype == torch.float32 else 0 * size
            if dtype == torch.float32 and (kind == "hub" or N < 10):
                parts = torch.minimum(n, torch.full_like(n, E // 8192 + 1)).view(B * N, 1)
                bound = bound + (2 * parts + 1) * 2 ** -24 * (size + given.view(B * N, K).double().abs())
            assert bool(((out.view(B * N, K).double() - want).abs() <= bound).all())
            out = given.clone()
            capi.scatter_sum_count_with_workspace(src, index, out, count, B, E, K, N, E, 1, out_given)
            assert bool(((out.view(B * N, K).double() - want).abs() <= bound).all())
            assert torch.equal(count.long(), n)


def test_value_tiles_under_graph_replay(monkeypatch):
    """A captured sum, replayed over even, skewed and sorted indices: each verdict of the sample leaves the call to other kernels."""
    import pytorch_scatter_amd as ts
    monkeypatch.setenv("TS_SCATTER_BINNED", "2")
    g = torch.Generator(device=DEV).manual_seed(2)
    E, N = 300000, 20000
    index, x = _index("even", E, N, g), torch.randint(-9, 10, (E, 3), generator=g, device=DEV, dtype=torch.int32)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        ts.scatter(x, index, dim=0, dim_size=N)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = ts.scatter(x, index, dim=0, dim_size=N)
    for kind in ("even", "sorted", "hub", "one row", "even"):
        new = _index(kind, E, N, g)
        index.copy_(new.sort()[0] if kind == "sorted" else torch.full_like(new, 7) if kind == "one row" else new)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, torch.zeros((N, 3), dtype=torch.int32, device=DEV).index_add_(0, index, x))
