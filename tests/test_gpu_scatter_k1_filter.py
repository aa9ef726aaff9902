"""min / max of one value per entry where hubs share a row of the workgroups' tables (csrc/scatter_k1.h): the ones that come late
go through the filter and the queues. Values repeat, so that positions decide among equal ones."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
ROWS = 8192  # rows of a table


@pytest.mark.parametrize("dtype", [torch.float32, torch.int32])
@pytest.mark.parametrize("how", ["random", "rising", "falling", "constant"])
@pytest.mark.parametrize("E,N,hubs", [(1 << 15, 2 * ROWS + 6, [0, ROWS, 2 * ROWS]), (300_001, 40_000, [5, 5 + ROWS, 5 + 2 * ROWS, 7]),
                                      (1_200_003, 64 * ROWS, [ROWS * k for k in range(64)])])
def test_hubs_that_share_a_table_row(E, N, hubs, how, dtype):
    import pytorch_scatter_amd as ts
    from pytorch_scatter_amd import capi
    g = torch.Generator(device=DEV).manual_seed(E)
    index = torch.randint(0, N, (E,), generator=g, device=DEV)
    some = torch.rand(E, generator=g, device=DEV) < 0.9
    index[some] = torch.tensor(hubs, device=DEV)[torch.randint(0, len(hubs), (int(some.sum()),), generator=g, device=DEV)]
    at = torch.arange(E, device=DEV)
    src = {"random": torch.randint(-500, 500, (E,), generator=g, device=DEV), "rising": at // 7, "falling": -(at // 7),
           "constant": torch.full_like(at, 3)}[how].to(dtype)
    for op, reduce in ((ts.scatter_max, "amax"), (ts.scatter_min, "amin")):
        out, arg = op(src, index, dim=0, dim_size=N)
        assert capi.scatter_last_route() == capi.lib().ts_scatter_route_name(14).decode()
        best = torch.zeros(N, dtype=dtype, device=DEV).scatter_reduce_(0, index, src, reduce, include_self=False)
        first = torch.full((N,), E, dtype=torch.long, device=DEV).scatter_reduce_(
            0, index, torch.where(src == best[index], at, E), "amin")
        assert torch.equal(out, best) and torch.equal(arg, first)
