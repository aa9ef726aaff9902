"""Group statistics over entries sorted by group (csrc/group_rows.h) at the sizes where they can go wrong: rows of one column
to several column slices, widths that fill no vector, workers that begin and end inside a group, groups over several workers
and tiles, empty groups, entries outside [0, N), batches. Expected values: torch in 64 bits."""
import pytest
import torch

from test_gpu_group_order import DEV, _index, _softmax64

pytestmark = pytest.mark.gpu

WIDTHS = [("even", 2, 700, K, 60) for K in (1, 2, 3, 4, 5, 7, 33, 64, 65, 130)] + [
    ("even", 1, 3001, 100, 150), ("even", 1, 1, 3, 1), ("even", 1, 9, 256, 40), ("even", 1, 5000, 8, 20000),
    ("hub", 1, 20000, 8, 900), ("hub", 1, 3000, 50, 70), ("hub", 2, 6001, 1, 50), ("one group", 1, 5001, 6, 7),
    ("one group", 1, 1300, 72, 2), ("one group", 1, 255, 64, 1), ("sorted", 1, 6000, 9, 900), ("sorted", 2, 1201, 41, 40),
    ("outside", 1, 4000, 12, 300), ("outside", 2, 1001, 101, 50), ("nobody", 1, 300, 8, 20),
    # from 16 MB on the tiles for an index in order come first
    ("sorted", 1, 600000, 9, 70000), ("one descent", 2, 300000, 8, 35000)]
TYPES = [torch.float32, torch.float64, torch.bfloat16, torch.float16]


def _case(kind, B, E, K, N, dtype, monkeypatch):
    monkeypatch.setenv("TS_GROUP_ORDER", "2")
    g = torch.Generator(device=DEV).manual_seed(E * 7 + K)
    index = _index(kind, E, N, g)
    src, grad = ((torch.randn((B, n, K), generator=g, device=DEV, dtype=torch.float64) * 3).to(dtype) for n in (E, E))
    return index, (index >= 0) & (index < N), src, grad, torch.finfo(dtype).eps


def _sums(ix, x, N):
    return torch.zeros((x.size(0), N, x.size(2)), dtype=torch.float64, device=DEV).index_add(1, ix, x)


def _within(got, want, bound):
    bad = (got.double() - want).abs() - bound
    assert bad.numel() == 0 or float(bad.max()) <= 0, float(bad.max())


@pytest.mark.parametrize("dtype", TYPES)
@pytest.mark.parametrize("kind,B,E,K,N", WIDTHS)
def test_softmax(kind, B, E, K, N, dtype, monkeypatch):
    from pytorch_scatter_amd import capi
    index, ok, src, grad, eps = _case(kind, B, E, K, N, dtype, monkeypatch)
    ix = index[ok]
    n = torch.bincount(ix, minlength=N)[ix].view(1, -1, 1)
    tiny = 2.0 ** -23 if dtype == torch.float16 else 1e-30  # fp16 results below 2^-14: absolute spacing 2^-24
    for log_space in (False, True):
        out, grad_in = (torch.full((B, E, K), 7, dtype=dtype, device=DEV) for _ in range(2))
        order = capi.group_softmax_ordered(src, index, out, B, E, K, N, 0, 1, log_space)
        z, want = _softmax64(src[:, ok].double(), ix, N, log_space)
        # roundings: of z (its size times eps, in the exponential), of exp, sum and quotient or logarithm and difference
        bound = eps * (4 + want.abs() + z.abs()) if log_space else eps * (4 + z.abs()) * want
        if dtype == torch.float64:  # the same roundings on either side, and n additions
            bound = 2 * bound + eps * n * (1 if log_space else want)
        _within(out[:, ok], want, bound + tiny)
        capi.group_softmax_ordered_backward(out, grad, index, grad_in, B, E, K, N, 0, 1, log_space, order)
        y, go = out[:, ok].double(), grad[:, ok].double()
        terms = go if log_space else y * go
        s, spread = _sums(ix, terms, N)[:, ix], _sums(ix, terms.abs(), N)[:, ix]
        want = go - y.exp() * s if log_space else y * (go - s)
        # every term and the sum rounded once, then two or three operations on the whole
        size = go.abs() + y.exp() * spread if log_space else y.abs() * (go.abs() + spread)
        bound = 8 * eps * size
        if dtype == torch.float64:  # n additions on either side
            bound = 2 * bound + eps * n * (y.exp() if log_space else y) * spread
        _within(grad_in[:, ok], want, bound + tiny)
        assert not bool(out[:, ~ok].any()) and not bool(grad_in[:, ~ok].any())


@pytest.mark.parametrize("dtype", TYPES)
@pytest.mark.parametrize("kind,B,E,K,N", WIDTHS)
def test_logsumexp(kind, B, E, K, N, dtype, monkeypatch):
    from pytorch_scatter_amd import capi
    index, ok, src, grad, eps = _case(kind, B, E, K, N, dtype, monkeypatch)
    ix, x = index[ok], src[:, ok].double()
    n = torch.bincount(ix, minlength=N).view(1, -1, 1)
    out, grad_in = torch.full((B, N, K), 7, dtype=dtype, device=DEV), torch.full((B, E, K), 7, dtype=dtype, device=DEV)
    order = capi.group_reduce_ordered(src, index, out, None, None, B, E, K, N, 0, 1)
    full = ix.view(1, -1, 1).expand_as(x)
    top = torch.full((B, N, K), -float("inf"), dtype=torch.float64, device=DEV).scatter_reduce_(1, full, x, "amax")
    want = torch.where(n > 0, (_sums(ix, (x - top[:, ix]).exp(), N) + 1e-12).log() + top, 0)
    # roundings: of every z (|x| and the maximum at most 18: 36 eps in the exponential), of the exponentials and their sum, of
    # the logarithm and the sum with the maximum
    bound = eps * (2 + 36 + 2 * want.abs() + 8) + (eps * n if dtype == torch.float64 else 0)
    _within(out, want, bound.expand_as(want))
    go = grad[:, :1].expand(B, N, K).contiguous()
    capi.group_reduce_ordered_backward(src, index, out, None, None, go, grad_in, B, E, K, N, 0, 1, order)
    z = x - out.double()[:, ix]
    want = go.double()[:, ix] * z.exp()
    # the difference and the exponential in 32 bits (64 bits: as wide as the reference), then the element type
    e32 = max(eps, 2.0 ** -23) if dtype != torch.float64 else eps
    _within(grad_in[:, ok], want, want.abs() * (2 * eps + e32 * (4 + 2 * z.abs())) + (2.0 ** -23 if dtype == torch.float16 else 1e-30))
    assert not bool(grad_in[:, ~ok].any())


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64, torch.bfloat16])
@pytest.mark.parametrize("kind,B,E,K,N", WIDTHS)
def test_std(kind, B, E, K, N, dtype, monkeypatch):
    from pytorch_scatter_amd import capi
    if kind in ("one group", "hub") and dtype == torch.bfloat16:
        pytest.skip("a sum of squares over hundreds of entries, rounded to 16 bits, is not meaningful")
    index, ok, src, grad, eps = _case(kind, B, E, K, N, dtype, monkeypatch)
    ix, x = index[ok], src[:, ok].double()
    n = torch.bincount(ix, minlength=N)
    total, out = (torch.full((B, N, K), 7, dtype=dtype, device=DEV) for _ in range(2))
    count, grad_in = torch.full((B, N), -7, dtype=torch.int32, device=DEV), torch.full((B, E, K), 7, dtype=dtype, device=DEV)
    order = capi.group_reduce_ordered(src, index, out, total, count, B, E, K, N, 0, 1)
    assert torch.equal(count.long(), n.expand(B, N))
    sums, size = _sums(ix, x, N), _sums(ix, x.abs(), N)
    # the tiles for an index in order add in the element type: a lane at most twelve entries, half an eps of what it has each
    adds = 6 * eps if kind == "sorted" and E * K * src.element_size() >= 1 << 24 else 1e-13
    assert bool(((total.double() - sums).abs() <= eps * sums.abs() + adds * size).all())
    c = n.clamp(min=1).view(1, N, 1).double()
    mean, div = sums / c, (c - 1).clamp(min=1) + 1e-6
    want = (_sums(ix, (x - mean[:, ix]) ** 2, N) / div).sqrt()
    # roundings of the deviation and its square, of sum, quotient and root: 4 eps of the result; the mean is off by
    # 2 eps of itself, times the root of n / (n - 1) <= 2 in the result
    bound = (4 * eps + adds) * want + 4 * eps * mean.abs() + 2 * adds * size / c + 1e-6 * eps
    if dtype == torch.float64:  # n additions of squares on either side: n / 2 eps of the sum each, half that of its root
        bound = bound + eps * c / 2 * want
    _within(out, want, bound)
    go = grad[:, :1].expand(B, N, K).contiguous()
    capi.group_reduce_ordered_backward(src, index, out, total, count, go, grad_in, B, E, K, N, 0, 1, order)
    # (from the deviation that the call was given; groups of one entry have no gradient)
    w = go.double() / (out.double() * div)
    want = (w[:, ix] * (x - (total.double() / c)[:, ix]))
    some = (out != 0)[:, ix]
    # the divisor, its product, the quotient, the mean (2 eps of itself) and the difference; then the element type
    bound = eps * (8 * want.abs() + 4 * (w * mean).abs()[:, ix])
    _within(grad_in[:, ok][some], want[some], bound[some] + 1e-30)
    assert not bool(grad_in[:, ~ok].any())


def test_special_values(monkeypatch):
    """The lowest value, infinities and NaN: as the passes that do not sort give them."""
    import pytorch_scatter_amd as ts
    g, E, K, N = torch.Generator(device=DEV).manual_seed(3), 20000, 6, 900
    index = torch.randint(0, N, (E,), generator=g, device=DEV)
    src = torch.randn((E, K), generator=g, device=DEV)
    flat = src.view(-1)
    flat[:800] = torch.finfo(torch.float32).min
    flat[800:900] = float("inf")
    flat[950] = float("nan")
    flat[1000:3000] = -float("inf")
    for op in (ts.scatter_softmax, ts.scatter_log_softmax, ts.scatter_logsumexp, ts.scatter_std):
        got, want = [], []
        for outs, mode in ((got, "2"), (want, "0")):
            monkeypatch.setenv("TS_GROUP_ORDER", mode)
            x = src.clone().requires_grad_()
            y = op(x, index, dim=0, dim_size=N)
            outs += [y.detach(), torch.autograd.grad(y, x, torch.ones_like(y))[0]]
        for a, b in zip(got, want):
            assert torch.allclose(a, b, rtol=2e-5, atol=2e-5, equal_nan=True)
