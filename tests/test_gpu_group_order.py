"""Softmax over entries sorted by group first (the ordered tiles of csrc/group_fused.h) at the sizes where it can go wrong:
tiles of 256 to 2048 entries, rows of one 16-byte unit to several column slices, groups inside a tile, across one border
and over many tiles, an index in order, entries outside [0, N), batches and strides. Expected values: torch in 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _index(kind, E, N, g):
    index = torch.randint(0, N, (E,), generator=g, device=DEV)
    if kind == "one group":
        index.fill_(N // 2)
    elif kind == "hub":
        index[torch.randperm(E, generator=g, device=DEV)[:E // 2]] = N // 3
    elif kind == "sorted":
        index = index.sort()[0]
    elif kind == "one descent":
        index = index.sort()[0]
        index[E // 2] = 0
    elif kind == "outside":
        index[::3] += N
        index[1::7] = -1 - index[1::7]
    elif kind == "nobody":
        index += N
    return index


def _softmax64(x, index, N, log_space):
    """x [B, E, K], every index in [0, N): the group maximum, what the exponential is taken of, and the result."""
    B, E, K = x.shape
    full = index.view(1, E, 1).expand(B, E, K)
    top = torch.full((B, N, K), -float("inf"), dtype=torch.float64, device=DEV).scatter_reduce_(1, full, x, "amax")
    z = x - top.gather(1, full)
    s = torch.zeros((B, N, K), dtype=torch.float64, device=DEV).index_add_(1, index, z.exp()).gather(1, full)
    return z, z - (s + 1e-12).log() if log_space else z.exp() / s


CASES = [("even", 1, 255, 8, 30), ("even", 1, 3001, 8, 400), ("even", 2, 2049, 24, 100), ("even", 1, 5000, 16, 500),
         ("even", 1, 1500, 64, 100), ("even", 1, 700, 200, 50), ("hub", 1, 9001, 8, 300), ("hub", 1, 3000, 72, 20),
         ("one group", 1, 5001, 8, 7), ("one group", 1, 600, 136, 1), ("sorted", 1, 6000, 8, 900), ("sorted", 2, 1201, 40, 90),
         ("sorted", 1, 2500, 72, 40), ("outside", 1, 4000, 8, 300), ("outside", 2, 1001, 104, 50), ("nobody", 1, 300, 8, 20),
         ("even", 1, 1, 8, 1), ("even", 1, 20000, 8, 30000), ("hub", 1, 40000, 8, 70000),
         # from 16 MB on the tiles for an index in order come first
         ("sorted", 1, 600000, 8, 70000), ("even", 1, 600000, 8, 70000), ("one descent", 1, 600000, 16, 70000)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("kind,B,E,K,N", CASES)
def test_ordered_softmax(kind, B, E, K, N, dtype, monkeypatch):
    from pytorch_scatter_amd import capi
    monkeypatch.setenv("TS_GROUP_ORDER", "2")
    g = torch.Generator(device=DEV).manual_seed(E * 7 + K)
    index = _index(kind, E, N, g)
    ok = (index >= 0) & (index < N)
    src = (torch.randn((B, E, K), generator=g, device=DEV, dtype=torch.float64) * 3).to(dtype)
    grad = torch.randn((B, E, K), generator=g, device=DEV, dtype=torch.float64).to(dtype)
    eps = torch.finfo(dtype).eps
    tiny = 2.0 ** -23 if dtype == torch.float16 else 1e-30  # fp16 results below 2^-14: absolute spacing 2^-24
    for log_space in (False, True):
        out = torch.full((B, E, K), 7, dtype=dtype, device=DEV)
        order = capi.group_softmax_ordered(src, index, out, B, E, K, N, 0, 1, log_space)
        z, want = _softmax64(src[:, ok].double(), index[ok], N, log_space)
        # roundings: of z (its size times eps, in the exponential), of exp, sum and quotient or logarithm and difference
        bound = eps * (4 + want.abs() + z.abs()) if log_space else eps * (4 + z.abs()) * want
        if dtype == torch.float64:  # the same roundings on either side, and n additions
            n = torch.bincount(index[ok], minlength=N)[index[ok]].view(1, -1, 1)
            bound = 2 * bound + eps * n * (1 if log_space else want)
        bad = (out[:, ok].double() - want).abs() - bound - tiny
        assert bad.numel() == 0 or float(bad.max()) <= 0
        assert not bool(out[:, ~ok].any())
        if K * src.element_size() > 64:  # the backward pass of wider rows does not take the order
            continue
        grad_in = torch.full((B, E, K), 7, dtype=dtype, device=DEV)
        capi.group_softmax_ordered_backward(out, grad, index, grad_in, B, E, K, N, 0, 1, log_space, order)
        y, go, ix = out[:, ok].double(), grad[:, ok].double(), index[ok]
        terms = go if log_space else y * go
        zero = torch.zeros((B, N, K), dtype=torch.float64, device=DEV)
        s, spread = zero.index_add(1, ix, terms)[:, ix], zero.index_add(1, ix, terms.abs())[:, ix]
        want = go - y.exp() * s if log_space else y * (go - s)
        # every term and the sum rounded once, then two or three operations on the whole
        size = go.abs() + y.exp() * spread if log_space else y.abs() * (go.abs() + spread)
        if dtype == torch.float64:  # n additions on either side
            bound = 16 * eps * size + eps * n * (y.exp() if log_space else y) * spread
        else:
            bound = 8 * eps * size
        bad = (grad_in[:, ok].double() - want).abs() - bound - tiny
        assert bad.numel() == 0 or float(bad.max()) <= 0
        assert not bool(grad_in[:, ~ok].any())


@pytest.mark.parametrize("mode", ["2", "3"])
def test_ordered_softmax_layouts(mode, monkeypatch):
    """An index with strides of its own, the lowest value, infinities and NaN; src and gradients off their 16-byte border."""
    from pytorch_scatter_amd import capi
    import pytorch_scatter_amd as ts
    g = torch.Generator(device=DEV).manual_seed(3)
    E, N, K = 600000, 40000, 8
    wide = torch.randint(0, N, (E, 3), generator=g, device=DEV)
    flat = torch.randn(E * K + 1, generator=g, device=DEV)
    flat[:800] = torch.finfo(torch.float32).min
    flat[800:900] = float("inf")
    flat[950] = float("nan")
    flat[1000:1200] = -float("inf")
    go = torch.randn(E * K + 1, generator=g, device=DEV)
    for index in (wide[:, 1], wide[:, 1].sort()[0]):
        ref, want = torch.empty((1, E, K), device=DEV), torch.empty((1, E, K), device=DEV)
        for off in (0, 1):  # elements behind a 16-byte border
            src, grad = flat[off:off + E * K].view(E, K), go[off:off + E * K].view(E, K)
            monkeypatch.setenv("TS_GROUP_ORDER", "0")
            capi.group_softmax(src.clone(), index.contiguous(), ref, 1, E, K, N, 0, 1, False)
            capi.group_softmax_backward(ref, grad.clone().view(1, E, K), index.contiguous(), want, 1, E, K, N, 0, 1, False)
            monkeypatch.setenv("TS_GROUP_ORDER", mode)
            x = src.detach().requires_grad_()
            assert x.data_ptr() % 16 == 4 * off
            y = ts.scatter_softmax(x, index, dim=0, dim_size=N)
            assert torch.allclose(y, ref[0], rtol=2e-6, atol=0, equal_nan=True)
            got, = torch.autograd.grad(y, x, grad)
            assert torch.allclose(got, want[0], rtol=1e-5, atol=1e-6, equal_nan=True)


@pytest.mark.parametrize("E,N", [(20000, 900), (600000, 40000)])
def test_ordered_softmax_under_graph_replay(E, N, monkeypatch):
    """A captured forward and backward pass, replayed over other indices, in order and not."""
    import pytorch_scatter_amd as ts
    monkeypatch.setenv("TS_GROUP_ORDER", "2")
    g, K = torch.Generator(device=DEV).manual_seed(5), 8
    index, x, go = _index("even", E, N, g), torch.randn((E, K), generator=g, device=DEV), torch.randn((E, K), generator=g, device=DEV)
    x.requires_grad_()

    def step():
        y = ts.scatter_softmax(x, index, dim=0, dim_size=N)
        return y.detach(), torch.autograd.grad(y, x, go)[0]

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        outs = step()
    for kind in ("even", "sorted", "one group", "sorted", "hub", "outside"):
        index.copy_(_index(kind, E, N, g))
        graph.replay()
        torch.cuda.synchronize()
        for got, want in zip(outs, step()):
            assert torch.allclose(got, want, rtol=1e-5, atol=1e-6)


def test_ordered_softmax_checks(monkeypatch):
    from pytorch_scatter_amd import capi
    sizes = tuple(map(capi._i, (1, 1 << 20, 8, 1 << 17)))
    assert capi.lib().ts_group_order_bytes(*sizes, capi.DTYPE[torch.float32]) > 0
    assert capi.lib().ts_group_order_bytes(*sizes, capi.DTYPE[torch.int32]) == 0
    assert capi.lib().ts_group_order_bytes(*map(capi._i, (1, 1 << 20, 7, 1 << 17)), capi.DTYPE[torch.float32]) == 0
    monkeypatch.setenv("TS_GROUP_ORDER", "0")
    assert capi.lib().ts_group_order_bytes(*map(capi._i, (1, 1 << 24, 8, 1 << 20)), capi.DTYPE[torch.float32]) == 0
    x, ix = torch.zeros((1, 8, 4), device=DEV), torch.zeros(8, dtype=torch.int64, device=DEV)
    with pytest.raises(RuntimeError):
        capi.group_softmax_ordered(x, ix, x.clone(), 1, 8, 4, 2, 0, 1, False)
