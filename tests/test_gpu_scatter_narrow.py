"""Sums and means of narrow rows over entries sorted by row (GS_SUM in csrc/group_rows.h): widths of one column to 60 bytes, empty
rows among and behind the others, hubs over many tiles, entries outside [0, N), batches. Whole numbers: exact."""
import pytest
import torch

from test_gpu_group_order import DEV, _index

pytestmark = pytest.mark.gpu

CASES = [("even", 1, 9001, 1, 700), ("even", 2, 5003, 3, 9000), ("even", 1, 20000, 5, 900), ("hub", 1, 60001, 2, 500),
         ("hub", 1, 20011, 7, 30000), ("one group", 1, 9000, 6, 4), ("sorted", 1, 30000, 7, 2100), ("sorted", 2, 9001, 1, 50),
         ("outside", 2, 9003, 4, 300), ("nobody", 1, 8200, 3, 20), ("even", 1, 9000, 15, 90)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("kind,B,E,K,N", CASES)
def test_sums_and_means(kind, B, E, K, N, dtype, monkeypatch):
    import pytorch_scatter_amd as ts
    from pytorch_scatter_amd import capi
    monkeypatch.setenv("TS_SCATTER_NARROW", "2")
    K = min(K, 60 // dtype.itemsize)
    g = torch.Generator(device=DEV).manual_seed(E + K)
    index = _index(kind, E, N, g)
    ok = (index >= 0) & (index < N)
    # 16-bit types: at most 200 ones to a row (bf16 counts to 256), the others small numbers
    if dtype.itemsize == 2:
        few = torch.rand(E, generator=g, device=DEV) < 200 / max(200, int(torch.bincount(index[ok], minlength=1).max()) * 1.3)
        src = few.view(1, E, 1).expand(B, E, K).to(dtype).contiguous()
    else:
        src = torch.randint(-9, 10, (B, E, K), generator=g, device=DEV).to(dtype)
    want = torch.zeros((B, N, K), dtype=torch.float64, device=DEV).index_add_(1, index[ok], src[:, ok].double())
    assert dtype.itemsize > 2 or float(want.max()) <= 256
    out = ts.scatter_sum(src, index, dim=1, dim_size=N)
    assert capi.scatter_last_route() == "sum: narrow rows, entries sorted by row"
    assert torch.equal(out.double(), want)
    n = torch.bincount(index[ok], minlength=N).clamp(min=1).view(1, N, 1).to(dtype)
    mean = ts.scatter_mean(src, index.expand(B, E), dim=1, dim_size=N)
    assert torch.equal(mean, out / n)
    # a given out takes the kernels that add to it
    base = torch.ones((B, N, K), dtype=dtype, device=DEV)
    if dtype.itemsize > 2:
        assert torch.equal(ts.scatter_sum(src, index, dim=1, out=base.clone()).double(), want + 1)
