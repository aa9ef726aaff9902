"""Scatter sum, mean, min and max of small inputs in one launch (csrc/scatter_small.h) at the sizes where it can go wrong: 512 entries
a step, 8192 at most, rows and columns of a workgroup, all entries in one row, entries outside [0, N), more rows than entries,
batches, strides, an index shared by all batches, out given. Expected values: torch in 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
CASES = [("even", 1, 1, 1, 1), ("even", 1, 511, 8, 40), ("even", 1, 512, 8, 40), ("even", 1, 513, 33, 7), ("even", 1, 3010, 64, 128),
         ("even", 1, 8191, 3, 900), ("even", 1, 8192, 1, 5), ("one row", 1, 2000, 64, 3), ("one row", 1, 8192, 1, 1),
         ("outside", 1, 3001, 16, 300), ("even", 1, 100, 4, 60000), ("even", 3, 1000, 20, 50), ("even", 8, 40, 130, 600),
         ("even", 1, 40, 3000, 9), ("sorted", 1, 5000, 24, 513), ("nobody", 1, 50, 4, 6)]


def _index(kind, E, N, g):
    index = torch.randint(0, N, (E,), generator=g, device=DEV)
    if kind == "one row":
        index.fill_(N // 2)
    elif kind == "sorted":
        index = index.sort()[0]
    elif kind == "outside":
        index[::3] += N
        index[1::7] = -1 - index[1::7]
    elif kind == "nobody":
        index += N
    return index


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("kind,B,E,K,N", CASES)
def test_scatter_small(kind, B, E, K, N, dtype, monkeypatch):
    from pytorch_scatter_amd import capi
    monkeypatch.setenv("TS_SCATTER_SMALL", "2")
    assert capi.scatter_small_applies(B, E, K, N, dtype, capi.SUM)
    g = torch.Generator(device=DEV).manual_seed(E + K)
    rows = torch.stack([_index(kind, E, N, g) for _ in range(B)])
    for shared in (False, True):
        index = rows[:1].expand(B, E) if shared else rows
        src = torch.randn((B, E, K), generator=g, device=DEV, dtype=torch.float64).to(dtype)
        given = torch.randn((B, N, K), generator=g, device=DEV, dtype=torch.float64).to(dtype)
        n, total = torch.zeros((B, N), device=DEV, dtype=torch.float64), torch.zeros((B, N, K), device=DEV, dtype=torch.float64)
        size = torch.zeros_like(total)
        for b in range(B):
            ok = (index[b] >= 0) & (index[b] < N)
            n[b] = torch.bincount(index[b][ok], minlength=N)
            total[b].index_add_(0, index[b][ok], src[b][ok].double())
            size[b].index_add_(0, index[b][ok], src[b][ok].double().abs())
        # sums are held in 64 bits and rounded once, a mean once more
        eps, tiny = torch.finfo(dtype).eps, 2.0 ** -24 if dtype == torch.float16 else 0.0
        c = n.clamp(min=1).unsqueeze(-1)
        for reduce, out_given in ((capi.SUM, False), (capi.SUM, True), (capi.MEAN, False), (capi.MEAN, True)):
            out, count = given.clone(), torch.full((B, N), -3, device=DEV, dtype=torch.float64).to(dtype)
            capi.scatter_small(src, index, out, count, None, B, E, K, N, 0 if shared else E, 1, reduce, out_given)
            want = total + given.double() if out_given else total
            want = want / c if reduce == capi.MEAN else want
            bound = 2 * eps * want.abs() + 4e-16 * size * n.clamp(min=1).unsqueeze(-1).sqrt() + tiny
            if dtype in (torch.bfloat16, torch.float16) and reduce == capi.MEAN:
                bound = bound + eps * want.abs()  # the count is rounded to the element type as well
            assert bool(((out.double() - want).abs() <= bound).all())
            assert torch.equal(count, n.clamp(min=1).to(dtype))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("kind,B,E,K,N", CASES)
def test_scatter_small_min_max(kind, B, E, K, N, dtype, monkeypatch):
    """Against the kernels that other sizes take, exactly: values with many ties, both zeros, NaN, infinities, the limits."""
    from pytorch_scatter_amd import capi
    monkeypatch.setenv("TS_SCATTER_SMALL", "2")
    assert capi.scatter_small_applies(B, E, K, N, dtype, capi.MAX)
    g = torch.Generator(device=DEV).manual_seed(E + K)
    index = torch.stack([_index(kind, E, N, g) for _ in range(B)])
    src = torch.randint(-3, 4, (B, E, K), generator=g, device=DEV).to(dtype)
    odd = torch.tensor([-0.0, float("nan"), float("inf"), -float("inf"), torch.finfo(dtype).min, torch.finfo(dtype).max],
                       device=DEV, dtype=dtype)
    src.view(-1)[::7] = odd[torch.randint(0, 6, (src.view(-1)[::7].numel(),), generator=g, device=DEV)]
    given = torch.randint(-3, 4, (B, N, K), generator=g, device=DEV).to(dtype)
    given.view(-1)[::11] = float("nan")
    for reduce in (capi.MIN, capi.MAX):
        for out_given in (False, True):
            out, want = given.clone(), given.clone()
            arg, want_arg = (torch.full((B, N, K), -5, dtype=torch.int64, device=DEV) for _ in range(2))
            capi.scatter_small(src, index, out, None, arg, B, E, K, N, E, 1, reduce, out_given)
            capi.scatter(src, index, want, want_arg, B, E, K, N, E, 1, 0, reduce, out_given)
            bits = torch.int32 if dtype == torch.float32 else torch.int16
            assert torch.equal(out.view(bits), want.view(bits)) and torch.equal(arg, want_arg)


def test_scatter_small_operator():
    """Through the operators: strides, dims, autograd of the mean, an integer mean and a large call beside it."""
    import pytorch_scatter_amd as ts
    g = torch.Generator(device=DEV).manual_seed(1)
    wide = torch.randint(0, 50, (700, 2), generator=g, device=DEV)
    index = wide[:, 1]
    x = torch.randn((700, 12), generator=g, device=DEV, requires_grad=True)
    for reduce in ("sum", "mean"):
        out = ts.scatter(x, index, dim=0, dim_size=60, reduce=reduce)
        want = torch.zeros((60, 12), device=DEV).index_add(0, index, x)
        n = torch.bincount(index, minlength=60).clamp(min=1).view(-1, 1)
        want = want / n if reduce == "mean" else want
        assert torch.allclose(out, want, rtol=1e-5, atol=1e-5)
        go = torch.randn_like(out)
        assert torch.allclose(torch.autograd.grad(out, x, go)[0], torch.autograd.grad(want, x, go)[0], rtol=1e-6, atol=1e-7)
        y = torch.randn((4, 700, 3), generator=g, device=DEV)
        out = ts.scatter(y, index, dim=1, dim_size=60, reduce=reduce)
        want = torch.zeros((4, 60, 3), device=DEV).index_add(1, index, y)
        assert torch.allclose(out, want / n if reduce == "mean" else want, rtol=1e-5, atol=1e-5)
        last = ts.scatter(y.transpose(1, 2), index, dim=-1, dim_size=60, reduce=reduce)
        assert torch.allclose(last, out.transpose(1, 2), rtol=1e-5, atol=1e-5)
    ints = torch.randint(-9, 9, (700, 2), generator=g, device=DEV)
    want = torch.zeros((60, 2), dtype=torch.int64, device=DEV).index_add(0, index, ints)
    assert torch.equal(ts.scatter(ints, index, dim=0, dim_size=60, reduce="mean"), torch.div(want, n, rounding_mode="floor"))
    given = torch.ones((60, 12), device=DEV)
    out = ts.scatter_mean(x.detach(), index, 0, given)
    want = (torch.ones((60, 12), device=DEV).index_add(0, index, x.detach())) / n
    assert torch.allclose(out, want, rtol=1e-5, atol=1e-5) and torch.equal(given, out)


def test_scatter_small_declines(monkeypatch):
    from pytorch_scatter_amd import capi
    for dtype, sizes, reduce in ((torch.float32, (1, 8193, 1, 10), capi.MEAN), (torch.float32, (1, 8192, 64, 10), capi.MAX),  # 2^19 values
                                 (torch.int32, (1, 100, 4, 10), capi.SUM), (torch.float64, (1, 100, 4, 10), capi.MIN),
                                 (torch.float32, (1, 100, 4, 10), capi.MUL)):
        assert not capi.scatter_small_applies(*sizes, dtype, reduce)
    assert capi.scatter_small_applies(1, 100, 4, 10, torch.float32, capi.SUM)
    monkeypatch.setenv("TS_SCATTER_SMALL", "0")
    assert not capi.scatter_small_applies(1, 100, 4, 10, torch.float32, capi.SUM)
