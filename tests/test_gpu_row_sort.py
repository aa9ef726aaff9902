"""Scatter of wide rows through the sort of the index by row (csrc/row_sort.h) at the sizes where it can go wrong: tiles
of 1024 to 8192 entries, buckets at and above what one sorting workgroup holds (8192 entries, 16384 from 4 M entries on), buckets
of one row and of 8192 rows, entries outside [0, N), an index in order. Sums of int32 are exact; min / max must give the
first position of equal values. The expected results come from torch on the same device."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _index(kind, E, N, g):
    index = torch.randint(0, N, (E,), generator=g, device=DEV)
    if kind == "one row":
        index.fill_(N // 2)
    elif kind.startswith("hub"):  # exactly so many entries in one row, the others elsewhere
        n = int(kind[3:])
        index = torch.where(index == N // 3, (N // 3 + 1) % N, index)
        index[torch.randperm(E, generator=g, device=DEV)[:n]] = N // 3
    elif kind == "sorted":
        index = index.sort()[0]
    elif kind == "pieces":  # in order but for pieces of 5000 entries: a bucket's entries in one or two tiles
        index = index.sort()[0]
        index = index[(torch.arange(E, device=DEV) // 5000 + torch.rand(E, generator=g, device=DEV, dtype=torch.float64)).argsort()]
    elif kind == "outside":
        index[::3] += N
        index[1::7] = -1 - index[1::7]
    return index


CASES = [("even", 8191, 300), ("even", 8192, 300), ("even", 8193, 300), ("one row", 8192, 5), ("one row", 8193, 5),
         ("one row", 50001, 1), ("hub8191", 20000, 40), ("hub8192", 20000, 40), ("hub8193", 20000, 40),
         ("hub30000", 60001, 100000), ("even", 30000, 600001), ("sorted", 30001, 7000), ("outside", 30001, 7000),
         ("even", 1, 1), ("even", 4194303, 70001), ("even", 4194305, 70001), ("hub16384", 4194305, 2000003),
         ("hub16385", 4194305, 2000003), ("hub1000000", 4194304, 1000),
         ("hub200001", 600001, 8400007), ("even", 600001, 8400007),
         # a lane more in place from 524288 entries on; more than 1024 tiles: the runs of a bucket in two rounds
         ("even", 524288, 5000), ("even", 524289, 5000), ("pieces", 60001, 3000), ("pieces", 8500001, 400000),
         ("hub40000", 8500001, 40000), ("outside", 8388609, 40000)]


@pytest.mark.parametrize("kind,E,N", CASES)
def test_row_sort(kind, E, N, monkeypatch):
    from pytorch_scatter_amd import capi
    monkeypatch.setenv("TS_SCATTER_BINNED", "2")
    g = torch.Generator(device=DEV).manual_seed(E + N)
    K = 16 if E > 100000 or N > 1000000 else 32
    index = _index(kind, E, N, g)
    ok = (index >= 0) & (index < N)
    src = torch.randint(-50, 51, (E, K), generator=g, device=DEV, dtype=torch.int32)
    out = torch.full((N, K), 9, dtype=torch.int32, device=DEV)
    capi.scatter_with_workspace(src, index, out, None, 1, E, K, N, 0, 1, 0, capi.SUM, 0)
    want = torch.zeros((N, K), dtype=torch.int32, device=DEV).index_add_(0, index[ok], src[ok])
    assert torch.equal(out, want)
    arg = torch.empty((N, K), dtype=torch.int64, device=DEV)
    capi.scatter_with_workspace(src, index, out, arg, 1, E, K, N, 0, 1, 0, capi.MAX, 0)
    idx = index[ok].view(-1, 1).expand(-1, K)
    top = torch.full((N, K), -1000, dtype=torch.int32, device=DEV).scatter_reduce_(0, idx, src[ok], "amax")
    pos = torch.nonzero(ok).expand(-1, K)
    first = torch.where(src[ok] == top.gather(0, idx), pos, E)
    want_arg = torch.full((N, K), E, dtype=torch.int64, device=DEV).scatter_reduce_(0, idx, first, "amin")
    assert torch.equal(out, torch.where(want_arg < E, top, 0))
    assert torch.equal(arg, want_arg)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("kind,B,E,K,N", [("even", 1, 3000, 33, 250), ("even", 2, 900, 130, 80), ("sorted", 1, 3001, 200, 7),
                                          ("outside", 1, 20000, 64, 900), ("one row", 1, 30001, 32, 3),
                                          ("hub500", 1, 2000, 513, 300), ("even", 1, 1, 64, 1), ("even", 1, 200, 64, 5000)])
def test_std_rows(kind, B, E, K, N, dtype, monkeypatch):
    """Standard deviation over entries sorted by group: every error against 64 bits within the roundings of the element
    type: root, quotient, and the mean, whose rounding shifts all deviations of a group alike."""
    from pytorch_scatter_amd import capi
    if kind in ("one row", "hub500") and dtype in (torch.bfloat16, torch.float16):
        pytest.skip("a sum of squares over hundreds of entries, rounded to 16 bits, is not meaningful")
    monkeypatch.setenv("TS_SCATTER_BINNED", "2")
    monkeypatch.setenv("TS_GROUP_BINS", "0")
    g = torch.Generator(device=DEV).manual_seed(E + K)
    index = _index(kind, E, N, g)
    ok = (index >= 0) & (index < N)
    src = (torch.randn((B, E, K), generator=g, device=DEV, dtype=torch.float64) * 3 + 1).to(dtype)
    total, out = (torch.full((B, N, K), 7, dtype=dtype, device=DEV) for _ in range(2))
    count = torch.full((B, N), -7, dtype=torch.int32, device=DEV)
    capi.group_std_forward(src, index, total, count, out, B, E, K, N, 0, 1, True)
    idx, x = index[ok], src[:, ok].double()
    n = torch.bincount(idx, minlength=N)
    assert torch.equal(count.long(), n.expand(B, N))
    zero = torch.zeros((B, N, K), dtype=torch.float64, device=DEV)
    sums, size = zero.index_add(1, idx, x), zero.index_add(1, idx, x.abs())
    eps = torch.finfo(dtype).eps
    assert bool(((total.double() - sums).abs() <= eps * sums.abs() + 1e-13 * size).all())
    c = n.clamp(min=1).view(1, N, 1).double()
    mean = sums / c
    want = (zero.index_add(1, idx, (x - mean[:, idx]) ** 2) / ((c - 1).clamp(min=1) + 1e-6)).sqrt()
    # roundings of the deviation and its square, of sum, quotient and root: 4 eps of the result; the mean is off by
    # 2 eps of itself, times the root of n / (n - 1) <= 2 in the result
    bound = 4 * eps * want + 4 * eps * mean.abs() + 1e-6 * eps
    if dtype == torch.float64:  # n additions of squares on either side: n / 2 eps of the sum each, half that of its root
        bound = bound + eps * c / 2 * want
    if dtype == torch.float16:
        bound = bound + 2.0 ** -12  # squares below 2^-14 are subnormal: 2^-25 apiece, 2^-12.5 under the root
    bad = (out.double() - want).abs() > bound
    assert not bool(bad.any()), float(((out.double() - want).abs() - bound).max())


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64, torch.bfloat16])
@pytest.mark.parametrize("kind,B,E,K,N", [("even", 1, 3000, 33, 250), ("even", 2, 900, 136, 80), ("sorted", 1, 3001, 200, 7),
                                          ("outside", 1, 20000, 64, 900), ("outside", 2, 1001, 300, 50),
                                          ("one row", 1, 9001, 64, 3), ("even", 1, 1, 64, 1), ("even", 1, 200, 520, 5000)])
def test_arg_backward_rows(kind, B, E, K, N, dtype, monkeypatch):
    """Backward of max over entries sorted by row: every element exactly, zeros for entries outside [0, N)."""
    import ctypes
    from pytorch_scatter_amd import capi
    monkeypatch.setenv("TS_SCATTER_BINNED", "2")
    g = torch.Generator(device=DEV).manual_seed(E + K)
    index = _index(kind, E, N, g)
    src = torch.randint(-9, 10, (B, E, K), generator=g, device=DEV).to(dtype)
    out = torch.empty((B, N, K), dtype=dtype, device=DEV)
    arg = torch.empty((B, N, K), dtype=torch.int64, device=DEV)
    capi.scatter_with_workspace(src, index, out, arg, B, E, K, N, 0, 1, 0, capi.MAX, 0)
    ok = (index >= 0) & (index < N)
    full, x = index[ok].view(1, -1, 1).expand(B, -1, K), src[:, ok].double()
    top = torch.full((B, N, K), -100.0, dtype=torch.float64, device=DEV).scatter_reduce_(1, full, x, "amax")
    first = torch.where(x == top.gather(1, full), torch.nonzero(ok).view(1, -1, 1).expand(B, -1, K), E)
    want_arg = torch.full((B, N, K), E, device=DEV).scatter_reduce_(1, full, first, "amin")
    assert torch.equal(arg, want_arg) and torch.equal(out.double(), torch.where(want_arg < E, top, 0.0))
    grad = torch.randn((B, N, K), generator=g, device=DEV).to(dtype)
    want = torch.zeros((B, E + 1, K), dtype=dtype, device=DEV).scatter_(1, arg, grad)[:, :E]
    got = torch.full((B, E, K), 7, dtype=dtype, device=DEV)
    code, i = capi.DTYPE[dtype], ctypes.c_int64
    nbytes = int(capi.lib().ts_arg_backward_rows_workspace_bytes(i(B), i(E), i(K), i(N), code))
    ws = torch.empty(nbytes, dtype=torch.uint8, device=DEV)
    p = lambda x: ctypes.c_void_p(x.data_ptr())
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    capi._check(capi.lib().ts_arg_backward_rows(p(grad), p(arg), p(index), p(got), i(B), i(N), i(E), i(K), i(0), i(1), code,
                                                p(ws), ctypes.c_size_t(nbytes), stream))
    assert torch.equal(got, want)


def test_rows_that_were_given_up_are_reported(monkeypatch):
    """The wait for the tiles before a row's last one is bounded. With the bound forced to "never wait" from the host
    (TS_CSR_SPIN=-1; every kernel exits normally) the rows that cross tiles are given up: the status words say so and the
    operators raise. Without the override the words stay clean and the values are right."""
    import pytorch_scatter_amd as ts
    from pytorch_scatter_amd import capi
    monkeypatch.setenv("TS_SCATTER_BINNED", "2")
    monkeypatch.setenv("TS_GROUP_BINS", "0")
    E, N, K = 30001, 3, 64  # rows of thousands of entries
    g = torch.Generator(device=DEV).manual_seed(1)
    index = torch.randint(0, N, (E,), generator=g, device=DEV)
    src = torch.randint(-50, 51, (E, K), generator=g, device=DEV).float()
    sums = torch.zeros((N, K), device=DEV, dtype=torch.float64).index_add_(0, index, src.double()).float()  # exact
    out, total = torch.empty((N, K), device=DEV), torch.empty((N, K), device=DEV)
    arg = torch.empty((N, K), dtype=torch.long, device=DEV)
    count = torch.empty(N, dtype=torch.int32, device=DEV)
    i = capi._i
    std_bytes = int(capi.lib().ts_group_std_workspace_bytes(i(1), i(E), i(K), i(N), 0))

    def words(reduce):
        monkeypatch.setattr(capi, "CHECK_STATUS", False)
        ws = capi.scatter_with_workspace(src, index, out, arg if reduce == capi.MAX else None, 1, E, K, N, 0, 1, 0, reduce, 0)
        nbytes = capi.lib().ts_scatter_workspace_bytes(i(1), i(E), i(K), i(N), 0, reduce)
        monkeypatch.setattr(capi, "CHECK_STATUS", True)
        return capi.status_word(ws, nbytes)

    monkeypatch.setenv("TS_CSR_SPIN", "-1")
    assert words(capi.SUM) == 1 and bool((out == 0).all())
    assert words(capi.MAX) == 1 and bool((out == 0).all()) and bool((arg == E).all())
    with pytest.raises(capi.TsError, match="given up"):
        capi.group_std_forward(src, index, total, count, out, 1, E, K, N, 0, 1, True)
    with pytest.raises(capi.TsError, match="given up"):
        capi.scatter_sum_count_with_workspace(src, index, out, count, 1, E, K, N, 0, 1, False)
    for op in (ts.scatter_sum, ts.scatter_mean, ts.scatter_max, ts.scatter_std):
        with pytest.raises(RuntimeError, match="given up"):
            op(src, index, dim=0, dim_size=N)
    monkeypatch.delenv("TS_CSR_SPIN")
    assert std_bytes >= capi.STATUS_BYTES
    assert words(capi.SUM) == 0 and torch.equal(out, sums)
    assert words(capi.MAX) == 0 and torch.equal(out.max(0)[0], src.max(0)[0])
    for op in (ts.scatter_sum, ts.scatter_mean, ts.scatter_max, ts.scatter_std):
        op(src, index, dim=0, dim_size=N)


@pytest.mark.parametrize("K,taken", [(64, False), (130, True)])
def test_std_of_a_src_off_its_border(K, taken):
    """ts_group_std_forward with the workspace that its query reports, src one element off a 16-byte border: rows that the
    buckets then hold no longer (64 lanes) are refused as unsupported, not as a workspace too small; others are served."""
    import ctypes
    from pytorch_scatter_amd import capi
    E, N = (1 << 22) // max(1, K // 16), 70_001
    g = torch.Generator(device=DEV).manual_seed(K)
    index = torch.randint(0, N, (E,), generator=g, device=DEV)
    src = torch.randn(E * K + 1, generator=g, device=DEV)[1:].view(E, K)
    assert src.data_ptr() % 16 == 4
    total, out = torch.empty((N, K), device=DEV), torch.empty((N, K), device=DEV)
    count = torch.empty(N, dtype=torch.int32, device=DEV)
    i, p = capi._i, capi._p
    nbytes = int(capi.lib().ts_group_std_workspace_bytes(i(1), i(E), i(K), i(N), 0))
    assert nbytes > 0
    ws = torch.empty(nbytes, dtype=torch.uint8, device=DEV)
    rc = capi.lib().ts_group_std_forward(p(src), p(index), p(total), p(count), p(out), i(1), i(E), i(K), i(N), i(0), i(1), 0, 1,
                                         p(ws), ctypes.c_size_t(nbytes), capi._stream(out))
    assert rc == (0 if taken else 2)  # TS_OK, TS_ERR_UNSUPPORTED
    import pytorch_scatter_amd as ts
    got = ts.scatter_std(src, index, dim=0, dim_size=N)
    want = ts.scatter_std(src.double(), index, dim=0, dim_size=N)
    for x in [got] + ([out] if taken else []):
        assert torch.allclose(x.double(), want, rtol=1e-5, atol=1e-6)


class _NoGradient(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x):
        return x.clone()

    @staticmethod
    def backward(ctx, g):
        return None


@pytest.mark.parametrize("op", ["scatter_sum", "scatter_mean", "scatter_min", "scatter_max"])
def test_no_gradient_from_above_is_zero(op):
    """A function behind the call that hands no gradient back: the gradient of src is zeros, not missing."""
    import pytorch_scatter_amd as ts
    src = torch.randn((40, 3), dtype=torch.float64, device=DEV, requires_grad=True)
    out = getattr(ts, op)(src, torch.arange(40, device=DEV) % 7, 0)
    y = _NoGradient.apply(out[0] if isinstance(out, tuple) else out)
    (grad,) = torch.autograd.grad(y.sum(), src)
    assert grad.dtype == src.dtype and torch.equal(grad, torch.zeros_like(src))


def _special_values(shape, dtype, rng):
    """Small whole numbers (many ties) and, one in twenty, the values that trip a comparison: the limits of the type and, for
    floating types, infinities, NaN and -0.0."""
    x = torch.from_numpy(rng.integers(0 if dtype == torch.uint8 else -8, 9, size=shape)).to(dtype)
    if dtype.is_floating_point:
        info = torch.finfo(dtype)
        extra = torch.tensor([info.min, info.max, float("inf"), -float("inf"), float("nan"), -0.0], dtype=dtype)
    else:
        info = torch.iinfo(dtype)
        extra = torch.tensor([info.min, info.max, info.min + 1, info.max - 1], dtype=dtype)
    pick = torch.from_numpy(rng.integers(0, len(extra), size=shape))
    return torch.where(torch.from_numpy(rng.random(shape) < 0.05), extra[pick], x)


def _index_layout(layout, B, E, N, kind, rng):
    """[B, E] rows on the CPU; the device tensor that holds them and the strides of a batch and an entry in it."""
    own = layout != "shared"
    rows = rng.integers(0, N, size=(B if own else 1, E))
    if kind == "hub":  # half of the entries in one row: more than 32 tiles of the reduction
        rows = np.where(rng.random(rows.shape) < 0.5, N // 3, rows)
    if kind == "sorted":
        rows = np.sort(rows, axis=1)
    rows = torch.from_numpy(rows)
    if layout == "every second":
        held = torch.full((rows.shape[0], 2 * E), -5, dtype=torch.long)
        held[:, ::2] = rows
        return rows.expand(B, E), held.to(DEV), 2 * E, 2
    return rows.expand(B, E), rows.to(DEV), E if own else 0, 1


LAYOUTS = [("even", "shared", 1, 3000, 250), ("hub", "shared", 1, 40001, 40), ("hub", "every second", 1, 9001, 300),
           ("even", "own", 3, 3001, 90), ("sorted", "own", 3, 2500, 90), ("even", "every second", 2, 2500, 700)]


@pytest.mark.parametrize("reduce", ["min", "max"])
@pytest.mark.parametrize("dtype", [torch.float64, torch.int64, torch.float32, torch.bfloat16, torch.int32, torch.uint8])
@pytest.mark.parametrize("K", [64, 33, 520])
@pytest.mark.parametrize("kind,layout,B,E,N", LAYOUTS)
def test_minmax_rows(oracle, kind, layout, B, E, N, K, dtype, reduce, monkeypatch):
    """Values and positions of min / max as the oracle has them, for every accumulator width (8-byte carries of values and
    positions among them), 33 single columns, 520 columns in more than four column chunks, with and without an initial out."""
    from pytorch_scatter_amd import capi
    monkeypatch.setenv("TS_SCATTER_BINNED", "2")
    if K * (torch.finfo(dtype) if dtype.is_floating_point else torch.iinfo(dtype)).bits < 512:
        pytest.skip("rows under 64 bytes are not sorted")
    if K == 520:
        B, E = 1, min(E, 6000)
    if kind == "hub" and K != 33:
        E = min(E, 12001)
    rng = np.random.default_rng(E + K)
    rows, held, sb, se = _index_layout(layout, B, E, N, kind, rng)
    src = _special_values((B, E, K), dtype, rng)
    full = rows.unsqueeze(-1).expand(B, E, K)
    for given in (False, True):
        want = _special_values((B, N, K), dtype, rng) if given else None
        out = want.to(DEV) if given else torch.empty((B, N, K), dtype=dtype, device=DEV)
        arg = torch.empty((B, N, K), dtype=torch.long, device=DEV)
        want, want_arg = oracle.scatter(src, full, 1, want, None if given else N, reduce)
        capi.scatter_with_workspace(src.to(DEV), held, out, arg, B, E, K, N, sb, se, 0, capi.REDUCE[reduce], given)
        assert capi.scatter_last_route().startswith("min/max: buckets or segmented")
        assert torch.equal(arg.cpu(), want_arg), given
        got = out.cpu()
        same = (got == want) | ((got != got) & (want != want))
        assert bool(same.all()), given


@pytest.mark.parametrize("dtype", [torch.int32, torch.int64, torch.float32, torch.bfloat16])
@pytest.mark.parametrize("kind,layout,B,E,N", LAYOUTS[2:])
def test_sum_and_std_layouts(kind, layout, B, E, N, dtype, monkeypatch):
    """Sums (of whole numbers: exact) and standard deviations under an index of its own per batch and with strides."""
    from pytorch_scatter_amd import capi
    monkeypatch.setenv("TS_SCATTER_BINNED", "2")
    monkeypatch.setenv("TS_GROUP_BINS", "0")
    K = 40
    rng = np.random.default_rng(E)
    rows, held, sb, se = _index_layout(layout, B, E, N, kind, rng)
    # (bf16: at most 4500 ones and zeros to a row, which a partial sum in more than 16 bits rounds once at the end)
    src = torch.from_numpy(rng.integers(0, 2, size=(B, E, K)) if dtype == torch.bfloat16 else rng.integers(-9, 10, size=(B, E, K)))
    want = torch.zeros((B, N, K), dtype=torch.long).scatter_add_(1, rows.unsqueeze(-1).expand(B, E, K), src)
    for given in (False, True):
        out = torch.full((B, N, K), 3, dtype=dtype, device=DEV)
        capi.scatter_with_workspace(src.to(dtype).to(DEV), held, out, None, B, E, K, N, sb, se, 0, capi.SUM, given)
        assert capi.scatter_last_route().startswith("sum: buckets or segmented")
        assert torch.equal(out.cpu(), (want + (3 if given else 0)).to(dtype)), given
    if dtype == torch.float32:
        total, out = (torch.empty((B, N, K), device=DEV) for _ in range(2))
        count = torch.empty((B, N), dtype=torch.int32, device=DEV)
        capi.group_std_forward(src.to(dtype).to(DEV), held, total, count, out, B, E, K, N, sb, se, True)
        n = torch.zeros((B, N), dtype=torch.long).scatter_add_(1, rows, torch.ones((B, E), dtype=torch.long))
        assert torch.equal(count.cpu().long(), n) and torch.equal(total.cpu().long(), want)
        full = rows.unsqueeze(-1).expand(B, E, K)
        c = n.clamp(min=1).unsqueeze(-1).double()
        dev = (src - (want / c).gather(1, full)) ** 2
        exact = (torch.zeros((B, N, K), dtype=torch.double).scatter_add_(1, full, dev) / ((c - 1).clamp(min=1) + 1e-6)).sqrt()
        # roundings as in test_std_rows; the mean is at most 9
        assert bool(((out.cpu().double() - exact).abs() <= 2.0 ** -23 * (4 * exact + 36) + 1e-12).all())


def test_more_than_1024_buckets(monkeypatch):
    """From 12.6 M entries the buckets outnumber the lanes of the workgroup that turns their totals into starts; one of them is
    a hub of many chunks."""
    from pytorch_scatter_amd import capi
    monkeypatch.setenv("TS_SCATTER_BINNED", "2")
    E, N, K = 16_000_001, 1_500_007, 16
    g = torch.Generator(device=DEV).manual_seed(3)
    index = torch.randint(0, N, (E,), generator=g, device=DEV)
    index[::9] = 77_777
    src = torch.randint(-50, 51, (E, K), generator=g, device=DEV, dtype=torch.int32)
    out = torch.full((N, K), 9, dtype=torch.int32, device=DEV)
    capi.scatter_with_workspace(src, index, out, None, 1, E, K, N, 0, 1, 0, capi.SUM, 0)
    want = torch.zeros((N, K), dtype=torch.int32, device=DEV).index_add_(0, index, src)
    assert torch.equal(out, want)


@pytest.mark.parametrize("op", ["scatter_max", "scatter_min"])
@pytest.mark.parametrize("layout", ["expanded", "per batch", "every second", "full"])
def test_arg_backward_through_autograd(op, layout, monkeypatch):
    """Gradients of the operators through the rows in order (forced at this size); a full index keeps the other route."""
    import pytorch_scatter_amd as ts
    monkeypatch.setenv("TS_SCATTER_BINNED", "2")
    B, E, N, K = 2, 3001, 70, 64
    rng = np.random.default_rng(E)
    rows, held, _, _ = _index_layout("every second" if layout == "every second" else "shared" if layout == "expanded" else "own",
                                     B, E, N, "even", rng)
    index = held[:, ::2] if layout == "every second" else held[0] if layout == "expanded" else held
    if layout == "full":
        index = index.unsqueeze(-1).expand(B, E, K).contiguous()
    elif layout != "expanded":
        index = index.unsqueeze(-1)
    src = torch.from_numpy(rng.integers(-9, 10, size=(B, E, K))).double()
    grad = torch.randn((B, N, K), dtype=torch.double)
    full = rows.unsqueeze(-1).expand(B, E, K)
    # the first position of the best value of every row, from the values alone
    best = torch.zeros((B, N, K), dtype=torch.double).scatter_reduce_(1, full, src, "amax" if op == "scatter_max" else "amin", include_self=False)
    at = torch.arange(E).view(1, E, 1).expand(B, E, K)
    first = torch.full((B, N, K), E).scatter_reduce_(1, full, torch.where(src == best.gather(1, full), at, E), "amin")
    want = torch.where(first.gather(1, full) == at, grad.gather(1, full), 0.0)
    x = src.to(DEV).requires_grad_()
    out, arg = getattr(ts, op)(x, index, dim=1, dim_size=N)
    assert torch.equal(arg.cpu(), first) and torch.equal(out.detach().cpu(), best)
    (got,) = torch.autograd.grad(out, x, grad.to(DEV))
    assert torch.equal(got.cpu(), want)


def test_rows_under_graph_replay(monkeypatch):
    """A captured launch keeps its tag and its workspace: the readers of carries clear their flags, the totals of the sort are
    cleared by the call. Replays with another index each time (hubs over many tiles, one row, in order), eager calls in
    between, each against the eager result."""
    import pytorch_scatter_amd as ts
    monkeypatch.setenv("TS_SCATTER_BINNED", "2")
    monkeypatch.setenv("TS_GROUP_BINS", "0")
    E, N = 30001, 400
    g = torch.Generator(device=DEV).manual_seed(5)
    index = torch.randint(0, N, (E,), generator=g, device=DEV)
    wide, odd = (torch.zeros((E, K), device=DEV) for K in (32, 33))

    def step():
        return (ts.scatter_sum(wide, index, 0, dim_size=N), *ts.scatter_max(wide, index, 0, dim_size=N),
                ts.scatter_sum(odd, index, 0, dim_size=N), *ts.scatter_min(odd, index, 0, dim_size=N),
                ts.scatter_std(odd, index, 0, dim_size=N))

    for _ in range(2):
        step()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step()
    for kind in ("hub20000", "one row", "even", "sorted", "hub9000", "hub20000"):
        index.copy_(_index(kind, E, N, g))
        for x in (wide, odd):
            x.copy_(torch.randint(-50, 51, x.shape, generator=g, device=DEV))
        graph.replay()
        torch.cuda.synchronize()
        got = [t.clone() for t in out]
        for a, b in zip(got[:-1], step()[:-1]):
            assert torch.equal(a, b), kind
        assert torch.allclose(got[-1], step()[-1], rtol=1e-6, atol=0), kind  # sums of squares: another order of additions
        want = torch.zeros((N, 32), dtype=torch.float64, device=DEV).index_add_(0, index, wide.double())
        assert torch.equal(got[0].double(), want), kind
