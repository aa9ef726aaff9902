"""What is timed of this package: reductions over entries that share a row, through its public functions.

A case names an operator and a reduction, the number of entries and rows, the values per entry (``width``), the
element type, how the entries spread over the rows and in which order they come. ``train`` adds the backward pass.

* ``degrees``: ``even`` draws every entry's row uniformly (meshes, molecules, random sampling), ``web`` weights the rows
  log-normally (links, citations), ``hub`` by 1 / rank ** 1.2 (the most frequent row holds about a fifth of the entries).
* ``order``: ``sorted`` by row (batched graphs, compressed matrices) or ``shuffled`` (an edge list in any other order).
"""
import math

import torch

import pytorch_scatter_amd as ts

FLOAT, HALF, BF16 = "float32", "float16", "bfloat16"
GROUP_OPS = ("softmax", "log_softmax", "logsumexp", "std")
SIZE = {FLOAT: 4, "float64": 8, HALF: 2, BF16: 2, "int64": 8, "int32": 4}


def case(name, op, reduce, entries, rows, width, dtype=FLOAT, degrees="web", order="shuffled", train=False, batch=1):
    c = dict(op=op, reduce=reduce, entries=entries, rows=rows, width=width, dtype=dtype, degrees=degrees, order=order,
             train=train, batch=batch)
    return dict(c, name=name) if name else c


def listed():
    return [
        # mean readout of a mini-batch of 128 small graphs, a training step: nothing but latency
        case("readout", "scatter", "mean", 3_010, 128, 64, degrees="even", order="sorted", train=True),
        # sum of messages in one mid-sized graph, inference
        case("conv", "scatter", "sum", 200_000, 10_000, 16, degrees="even"),
        # neighbour mean over compressed rows, a training step
        case("csr-mean", "segment_csr", "mean", 467_488, 100_000, 64, order="sorted", train=True),
        # forces on atoms or points: three components per pair, each pair's row in no order
        case("forces", "scatter", "sum", 3_000_017, 150_001, 3, degrees="even"),
        # best score per node of a large skewed graph, with the position it came from
        case("best-score", "scatter", "max", 10_000_000, 100_000, 1, degrees="hub"),
        # attention of eight heads over the edges of a citation graph, a training step
        case("attention", "softmax", "", 2_313_294, 268_495, 8, train=True),
        # deviation of the messages, one of several aggregators side by side; a width that fills no vector
        case("deviation", "std", "", 1_000_003, 65_537, 33, train=True),
        # max pooling of messages, a training step
        case("max-pool", "scatter", "max", 2_312_497, 281_903, 64, train=True),
        # sum of messages in mixed precision, a training step
        case("conv-bf16", "scatter", "sum", 2_313_294, 268_495, 128, dtype=BF16, train=True),
        # a fixed mesh whose index was sorted once, a batch of four fields on it
        case("mesh-plan", "sorted_plan", "sum", 1_325_977, 220_000, 32, degrees="even", batch=4),
        # max over a large sorted edge list, with the positions
        case("coo-max", "segment_coo", "max", 8_997_792, 1_062_576, 128, degrees="even", order="sorted"),
        # node features to the edges of a large graph in mixed precision and their gradient back
        case("gather-bf16", "gather_csr", "", 21_005_389, 1_465_137, 128, dtype=BF16, order="sorted", train=True),
    ]


def draw(rng):
    op = rng.choice(["scatter"] * 6 + ["segment_csr", "segment_csr", "segment_coo", "segment_coo", "gather_csr", "gather_coo",
                                       "softmax", "softmax", "log_softmax", "logsumexp", "std", "sorted_plan"])
    reduce = "" if op in GROUP_OPS or op.startswith("gather") else rng.choice(["sum", "sum", "mean", "max", "max", "min"])
    dtype = rng.choice([FLOAT] * 5 + [BF16, BF16, HALF] + (["float64", "int64"] if op not in GROUP_OPS else []))
    degrees = rng.choice(["even", "even", "web", "web", "hub"])
    if degrees == "hub" and dtype in (BF16, HALF) and reduce in ("sum", "mean"):
        degrees = "web"  # millions of terms are not summed in 16 bits
    order = "shuffled" if op == "sorted_plan" else "sorted" if op.startswith(("segment", "gather")) else rng.choice(
        ["sorted", "shuffled", "shuffled"])
    train = not dtype.startswith("int") and rng.random() < 0.5
    if op == "std" and train:
        dtype = FLOAT  # two equal values in 16 bits: the gradient of their deviation is 0 / 0
    batch = rng.choice([1, 1, 1, 1, 2, 3, 8]) if op in ("scatter", "sorted_plan") else 1
    width = rng.choice([1, 1, 3, 4, 8, 16, 32, 64, 100, 128, 256, int(2 ** rng.uniform(0, 9)), int(2 ** rng.uniform(0, 9))])
    entries = int(math.exp(rng.uniform(math.log(1_000), math.log(20_000_000))))
    fewest = 6 if op == "std" else 1.5
    per_row = math.exp(rng.uniform(math.log(fewest), math.log(32 if dtype in (BF16, HALF) else 500)))
    # what a case moves stays well below the largest listed one, lower still where the rows come in no order
    most = 2.5e9 if order == "sorted" else 0.7e9
    entries = max(1_000, min(entries, int(most / (batch * (width * SIZE[dtype] + 8)))))
    rows = max(2, int(entries / per_row))
    return case("", op, reduce, entries, rows, width, dtype, degrees, order, train, batch)


def index_of(c, g):
    rows, dev = c["rows"], "cuda"
    if c["degrees"] == "even":
        index = torch.randint(0, rows, (c["entries"],), generator=g, device=dev)
    else:
        if c["degrees"] == "web":
            w = torch.randn(rows, generator=g, device=dev, dtype=torch.float64).exp_()
        else:
            w = torch.arange(1, rows + 1, device=dev, dtype=torch.float64).pow_(-1.2)
            w = w[torch.randperm(rows, generator=g, device=dev)]
        ends = w.cumsum(0)
        at = torch.rand(c["entries"], generator=g, device=dev, dtype=torch.float64) * ends[-1]
        index = torch.searchsorted(ends, at, right=True).clamp_(max=rows - 1)
    if c["op"] == "std":  # four entries in every row: the deviation of a single one has no gradient, that of two cancels
        index[:4 * rows] = torch.arange(4 * rows, device=dev) % rows
        index = index[torch.randperm(c["entries"], generator=g, device=dev)]
    return index.sort()[0] if c["order"] == "sorted" else index


def values(shape, dtype, g):
    kind = getattr(torch, dtype)
    if dtype.startswith("int"):
        return torch.randint(-100, 101, shape, generator=g, device="cuda", dtype=kind)
    return torch.randn(shape, generator=g, device="cuda", dtype=kind)


def prepare(case, seed):
    c = case
    g = torch.Generator(device="cuda").manual_seed(seed)
    index = index_of(c, g)
    lead = (c["batch"],) if c["batch"] > 1 else ()
    tail = (c["width"],) if c["width"] > 1 else ()
    per_entry, per_row = lead + (c["entries"],) + tail, lead + (c["rows"],) + tail
    gathers = c["op"].startswith("gather")
    state = dict(case=c, dim=len(lead), index=index, src=values(per_row if gathers else per_entry, c["dtype"], g))
    if c["op"].endswith("csr"):
        state["indptr"] = torch.searchsorted(index, torch.arange(c["rows"] + 1, device="cuda"))
        del state["index"]
    if c["op"] == "sorted_plan":
        state["plan"] = ts.SortedIndex(index, dim_size=c["rows"])
    if c["train"]:
        state["src"].requires_grad_()
        to_entries = gathers or c["op"] in ("softmax", "log_softmax")
        state["grad"] = values(per_entry if to_entries else per_row, c["dtype"], g)
    return state


def forward(state):
    """The call of the operator: its result, or the pair of values and positions."""
    c, src, dim, n = state["case"], state["src"], state["dim"], state["case"]["rows"]
    op, reduce = c["op"], c["reduce"]
    if op == "scatter":
        if reduce in ("min", "max"):
            return (ts.scatter_min if reduce == "min" else ts.scatter_max)(src, state["index"], dim=dim, dim_size=n)
        return ts.scatter(src, state["index"], dim=dim, dim_size=n, reduce=reduce)
    if op == "sorted_plan":
        return ts.scatter_sorted(src, state["plan"], dim=dim, reduce=reduce)
    if op == "segment_csr":
        if reduce in ("min", "max"):
            return (ts.segment_min_csr if reduce == "min" else ts.segment_max_csr)(src, state["indptr"])
        return ts.segment_csr(src, state["indptr"], reduce=reduce)
    if op == "segment_coo":
        if reduce in ("min", "max"):
            return (ts.segment_min_coo if reduce == "min" else ts.segment_max_coo)(src, state["index"], dim_size=n)
        return ts.segment_coo(src, state["index"], dim_size=n, reduce=reduce)
    if op == "gather_csr":
        return ts.gather_csr(src, state["indptr"])
    if op == "gather_coo":
        return ts.gather_coo(src, state["index"])
    call = {"softmax": ts.scatter_softmax, "log_softmax": ts.scatter_log_softmax, "logsumexp": ts.scatter_logsumexp,
            "std": ts.scatter_std}[op]
    return call(src, state["index"], dim=dim, dim_size=n)


def run(state):
    got = forward(state)
    outs = list(got) if isinstance(got, tuple) else [got]
    if state["case"]["train"]:
        outs += torch.autograd.grad(outs[0], state["src"], state["grad"])
    return [t.detach() for t in outs]


def work(case):
    c = case
    s, b = SIZE[c["dtype"]], c["batch"]
    entries, rows = b * c["entries"] * c["width"] * s, b * c["rows"] * c["width"] * s
    positions = b * c["rows"] * c["width"] * 8 if c["reduce"] in ("min", "max") else 0
    index = 8 * (c["rows"] + 1) if c["op"].endswith("csr") else 8 * c["entries"]
    if c["op"] == "sorted_plan":
        index = 4 * c["entries"] + 8 * (c["rows"] + 1)
    softmax = c["op"] in ("softmax", "log_softmax")
    moved = index + (2 * entries if softmax else entries + rows + positions)
    if c["train"]:  # softmax: result and gradient in; std, logsumexp: values, result and gradient; others: gradient (and positions)
        moved += (0 if positions else index) + entries + (
            2 * entries if softmax else entries + 2 * rows if c["op"] in GROUP_OPS else rows + positions)
    each = b * c["entries"] * c["width"]
    return {"bytes": moved, "flops": each * (4 if c["op"] in GROUP_OPS else 1) * (2 if c["train"] else 1)}


def tolerance(case):
    c = case
    if c["dtype"].startswith("int") or c["reduce"] in ("min", "max") or (c["op"].startswith("gather") and not c["train"]):
        return "exact"
    if c["dtype"] == "float64":
        return {"rel": 1e-13}
    if c["dtype"] == FLOAT:
        return {"rel": 1e-5}
    # a sum that is kept in 16 bits is rounded once per term
    kept = c["op"] == "scatter"
    return {"rel": (3e-2 if kept else 1.5e-2) * (1 if c["dtype"] == BF16 else 0.125)}
