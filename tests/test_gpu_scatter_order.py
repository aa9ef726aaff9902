"""Scatter of wide rows that keeps its order for the backward pass (ts_scatter_ordered, csrc/row_sort.h, rows_spread_kernel in
csrc/group_rows.h): gradients of entries sorted by row, of widths that fill no vector, in and outside [0, N), over batches.
Every gradient is one value of grad_out, divided once for the mean: exact."""
import pytest
import torch

from test_gpu_group_order import DEV, _index

pytestmark = pytest.mark.gpu

CASES = [("even", 1, 3001, 16, 250), ("even", 2, 900, 40, 80), ("even", 1, 5, 64, 3), ("even", 1, 700, 272, 900),
         ("hub", 1, 20000, 24, 300), ("one group", 1, 9001, 32, 3), ("sorted", 1, 5000, 48, 700), ("sorted", 2, 1201, 128, 7),
         ("outside", 2, 1001, 32, 50), ("nobody", 1, 300, 32, 20)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("kind,B,E,K,N", CASES)
def test_gradients(kind, B, E, K, N, dtype, monkeypatch):
    import pytorch_scatter_amd as ts
    from pytorch_scatter_amd import capi
    monkeypatch.setenv("TS_SCATTER_BINNED", "2")
    monkeypatch.setenv("TS_SCATTER_ORDER", "2")
    monkeypatch.setenv("TS_SCATTER_SMALL", "0")
    g = torch.Generator(device=DEV).manual_seed(E + K)
    index = _index(kind, E, N, g)
    ok = (index >= 0) & (index < N)
    count = torch.bincount(index[ok], minlength=N).clamp(min=1).view(1, N, 1).to(dtype)
    grad = torch.randn((B, N, K), generator=g, device=DEV, dtype=torch.float64).to(dtype)
    for odd in (0, 1):  # a width that fills no vector: sums alone
        src = torch.randint(-8, 9, (B, E, K + odd), generator=g, device=DEV).to(dtype).requires_grad_()
        go = torch.cat([grad, grad[:, :, :1]], 2) if odd else grad
        for op in (ts.scatter_sum, ts.scatter_mean) + (() if odd else (ts.scatter_max, ts.scatter_min)):
            out = op(src, index.expand(B, E), dim=1, dim_size=N)
            assert "segmented" in capi.scatter_last_route() or src[0, 0].nbytes < 64
            want = torch.zeros((B, E, K + odd), dtype=dtype, device=DEV)
            if isinstance(out, tuple):
                out, arg = out
                rows = go.transpose(0, 1)[index[ok]].transpose(0, 1)
                here = arg.transpose(0, 1)[index[ok]].transpose(0, 1) == torch.nonzero(ok).view(1, -1, 1)
                want[:, ok] = torch.where(here, rows, torch.zeros_like(rows))
            else:
                want[:, ok] = (go / count if op is ts.scatter_mean else go)[:, index[ok]]
            got, = torch.autograd.grad(out, src, go)
            assert torch.equal(got, want), (op.__name__, odd)


def test_order_is_kept_only_where_it_is_needed(monkeypatch):
    """Without a gradient nothing is saved, and a hook that moves the order off its border leaves the gradient as it is."""
    import pytorch_scatter_amd as ts
    monkeypatch.setenv("TS_SCATTER_BINNED", "2")
    monkeypatch.setenv("TS_SCATTER_ORDER", "2")
    monkeypatch.setenv("TS_SCATTER_SMALL", "0")
    g, E, K, N = torch.Generator(device=DEV).manual_seed(7), 5000, 32, 400
    index = torch.randint(0, N, (E,), generator=g, device=DEV)
    src = torch.randn((E, K), generator=g, device=DEV, requires_grad=True)
    go = torch.randn((N, K), generator=g, device=DEV)
    seen = []

    def moved(t):
        seen.append(t.dtype)
        return torch.cat([t[:1], t])[1:] if t.dtype == torch.uint8 else t

    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, moved):
        out = ts.scatter_sum(src, index, dim=0, dim_size=N)
        got, = torch.autograd.grad(out, src, go)
    assert torch.uint8 in seen and torch.equal(got, go[index])
    kept = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: kept.append(t) or t, lambda t: t):
        ts.scatter_sum(src.detach(), index, dim=0, dim_size=N)
    assert kept == []
