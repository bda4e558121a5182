"""What the embedding table is asked to do in earnest, as cases that can be timed and whose results can be compared.

A case is one kind of program around the table.  A table of `rows` x `width` floats is a concatenation of `fields`
categorical fields, and a batch holds `hot` ids per field for each of `samples` samples (the layout of
hetuctr_amd.workloads, which also names most of the sizes used here).  Ids follow a truncated Zipf law with exponent
`alpha` over the field's own range (0: uniform); with `whole` every field draws over the whole table.

One pass is
  * "train":  two consecutive training steps on two batches A and B, each of them preprocess(ids) and then
              push_pull(gradients of the batch before, output).  The second step returns every row that the first one
              updated, and the batch before the first step of a pass is the B of the pass before (of `prepare`, at first);
  * "infer":  one look-up, preprocess(ids) and push_pull without gradients.
Options: `host_ids` the ids lie in ordinary host memory, as numpy hands them over; `pooled` the `hot` ids of a field are
one sum-pooled bag; `shards` the table is cut over that many shards of a loopback group, of which the first `feeding`
have batches of their own and keep the hottest `cache` of the other shards' rows, under the staleness bound `bound`.
"""
import itertools
import math

import numpy as np
import torch

from hetuctr_amd import capi, load_hetuCTR, workloads

_DEFAULTS = {"path": "train", "samples": 2048, "fields": 26, "hot": 1, "rows": 33_762_577, "width": 128, "alpha": 1.05,
             "whole": False, "host_ids": False, "pooled": False, "shards": 1, "feeding": 1, "cache": 0.0, "bound": 0}


def _case(name=None, **options):
    case = dict(_DEFAULTS, **options)
    assert set(case) == set(_DEFAULTS)
    if name:
        case["name"] = name
    return case


def listed():
    return [
        # serving: the rows of a request of 128 samples from the large table
        _case("serve_128", path="infer", samples=128),
        # the batch of the reference's own driver (2048 samples of 26 fields), ids in HBM, and as that driver has them: a
        # numpy array
        _case("train_2048"),
        _case("train_2048_host", host_ids=True),
        # a small table of short rows, uniform ids: little memory traffic, many keys
        _case("train_8192_narrow", samples=8192, rows=1_000_000, width=16, alpha=0.0, whole=True),
        # sizes nobody rounds: a row width that is no multiple of four, a ragged batch
        _case("train_5003_odd", samples=5003, fields=39, rows=2_000_003, width=37, alpha=1.1),
        # the headline training step: 65536 samples of 26 Zipf fields, 33.8 M rows of 128 floats; ids in HBM and in host
        # memory
        _case("train_65536", samples=65536),
        _case("train_65536_host", samples=65536, host_ids=True),
        # multi-hot fields: few rows hit very often, and nearly every id of the large fields distinct
        _case("multihot_zipf", samples=32768, hot=10, rows=50_000_000, width=64, alpha=1.4),
        _case("multihot_uniform", samples=32768, hot=10, rows=50_000_000, width=64, alpha=0.0),
        # the same multi-hot fields with every field's ids sum-pooled in the table
        _case("pooled_zipf", samples=32768, hot=10, rows=50_000_000, width=64, alpha=1.4, pooled=True),
        # one shard of eight with its hot-row cache, the owners of the other rows beside it on the GPU
        _case("shard_1_of_8", samples=65536, shards=8, feeding=1, cache=0.10),
        # four shards that all train, with caches and bounded staleness
        _case("shards_4_train", samples=2048, rows=4_000_000, width=32, shards=4, feeding=4, cache=0.10, bound=5),
    ]


_MOST_FLOATS = 32768 * 26 * 10 * 64   # of a batch's rows, in the largest listed cases


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["train", "train", "train_host", "infer", "multihot", "pooled", "sharded"])
    case = _case(samples=_log_uniform(rng, 64, 65536), rows=_log_uniform(rng, 100_000, 50_000_000),
                 fields=rng.choice([26, 26, 13, 39]), alpha=rng.choice([0.0, 1.05, 1.1, 1.2, 1.4]),
                 width=rng.choice([16, 32, 64, 128, 128, rng.randint(5, 160)]))
    case["host_ids"] = kind == "train_host"
    if kind == "infer":
        case["path"] = "infer"
    if kind in ("multihot", "pooled"):
        case["hot"] = rng.randint(2, 20)
        case["pooled"] = kind == "pooled"
    if kind == "sharded":
        case["shards"] = rng.choice([2, 4, 8])
        case["feeding"] = rng.choice([1, case["shards"]])
        case["cache"] = rng.choice([0.02, 0.10])
        case["bound"] = rng.choice([0, 5])
        case["rows"] = min(case["rows"], 4_000_000)
        case["samples"] = max(64, case["samples"] // (case["feeding"] * 2))
    per_sample = case["fields"] * case["hot"] * case["width"] * case["feeding"]
    case["samples"] = max(1, min(case["samples"], _MOST_FLOATS // per_sample, 8_000_000 // (case["fields"] * case["hot"])))
    return case


# ---- ids ------------------------------------------------------------------------------------------------------------
_HEAD = 2048  # ranks of a field whose Zipf weights are added up one by one; the sum over the ranks behind them is the integral


def _zipf_head(count, alpha):
    """Cumulative weights of the first ranks of a field of `count` ids, the weight of all of them."""
    head = np.cumsum(np.power(np.arange(1, min(count, _HEAD) + 1, dtype=np.float64), -alpha))
    tail = 0.0
    if count > _HEAD:
        tail = ((_HEAD + 0.5) ** (1 - alpha) - (count + 0.5) ** (1 - alpha)) / (alpha - 1)
    return head, head[-1] + tail


def _field_ids(count, n, alpha, gen):
    if alpha == 0.0:
        return torch.randint(count, (n,), device="cuda", generator=gen)
    head, total = _zipf_head(count, alpha)
    u = torch.rand(n, device="cuda", generator=gen, dtype=torch.float64) * total
    rank = torch.searchsorted(torch.from_numpy(head).cuda(), u)
    behind = u - head[-1]
    beyond = ((_HEAD + 0.5) ** (1 - alpha) - behind.clamp_min(0) * (alpha - 1)).pow(1 / (1 - alpha)) - 0.5
    return torch.where(rank < len(head), rank, beyond.long()).clamp_(0, count - 1)


def _layout(case):
    return workloads.KeyStream({"rows": case["rows"], "samples": case["samples"], "fields": case["fields"],
                                "hot": case["hot"], "alpha": case["alpha"], "single_field": case["whole"]}, seed=0)


def _batch(case, fields, gen):
    s, f, h = case["samples"], case["fields"], case["hot"]
    ids = torch.empty((s, f, h), dtype=torch.int64, device="cuda")
    for i in range(f):
        ids[:, i, :] = _field_ids(int(fields.card[i]), s * h, case["alpha"], gen).view(s, h) + int(fields.base[i])
    return ids.view(-1)


# ---- the program around the table -----------------------------------------------------------------------------------
_ports = itertools.count(24000)


class _Single:
    """One table, every row in it: the module the reference's scripts import, or its pooled call."""

    def __init__(self, case, seed):
        owner, stored = np.zeros(case["rows"], np.uint8), np.arange(case["rows"], dtype=np.int64)
        self.bag = case["hot"] if case["pooled"] else 1
        if case["pooled"]:
            capi.seed(seed)
            self.table = capi.Table(0, 1, 0, "127.0.0.1", next(_ports), case["rows"], case["width"], 0, 0, owner, stored,
                                    ("Normal", 0.0, 0.1), 0.05)
        else:
            m = load_hetuCTR()
            m.seed(seed)
            self.table = m.HetuTable(rank=0, nrank=1, device_id=0, ip="127.0.0.1", port=next(_ports), length=case["rows"],
                                     width=case["width"], pull_bound=0, push_bound=0,
                                     init=m.Initializer(m.InitType.Normal, 0.0, 0.1), learning_rate=0.05,
                                     root_arr=owner, storage_arr=stored, verbose=0)

    def batch(self, case, fields, gen):
        ids = _batch(case, fields, gen)
        return ids.cpu().numpy() if case["host_ids"] else ids

    def step(self, ids, grad, out):
        if isinstance(ids, np.ndarray):
            self.table.preprocess(ids.ctypes.data, ids.shape[0])
        else:
            self.table.preprocess(ids.data_ptr(), ids.numel())
        g = 0 if grad is None else grad.data_ptr()
        if self.bag > 1:
            self.table.push_pull_pooled(g, out.data_ptr(), self.bag)
        else:
            self.table.push_pull(g, out.data_ptr())


class _Group:
    """The shards of a loopback group, stepped by one caller."""
    bag = 1

    def __init__(self, case, seed):
        r, fields = case["shards"], _layout(case)
        owner, stored = workloads.shard_layout(fields, r, case["cache"], seed=0, cached_ranks=tuple(range(case["feeding"])))
        capi.seed(seed)
        port = next(_ports)
        self.tables = [capi.Table(i, r, 0, "127.0.0.1", port, case["rows"], case["width"], case["bound"], case["bound"], owner,
                                  stored[i], ("Normal", 0.0, 0.1), 0.05) for i in range(r)]
        self.idle = [0] * (r - case["feeding"])

    def batch(self, case, fields, gen):
        return [_batch(case, fields, gen) for _ in range(case["feeding"])]

    def step(self, ids, grad, out):
        capi.group_preprocess(self.tables, [x.data_ptr() for x in ids] + self.idle, [x.numel() for x in ids] + self.idle)
        g = [0] * len(self.tables) if grad is None else [x.data_ptr() for x in grad] + self.idle
        capi.group_push_pull(self.tables, g, [x.data_ptr() for x in out] + self.idle)


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    fields = _layout(case)
    program = _Single(case, seed) if case["shards"] == 1 else _Group(case, seed)
    n = case["samples"] * case["fields"] * case["hot"] // program.bag
    many = case["feeding"] if case["shards"] > 1 else 0

    def rows(make):
        return [make() for _ in range(many)] if many else make()

    state = {"program": program, "train": case["path"] == "train", "steps": []}
    for _ in range(2 if state["train"] else 1):
        state["steps"].append({
            "ids": program.batch(case, fields, gen),
            "grad": rows(lambda: torch.randn((n, case["width"]), device="cuda", generator=gen) * 1e-3) if state["train"] else None,
            "out": rows(lambda: torch.empty((n, case["width"]), device="cuda")),
        })
    torch.cuda.synchronize()
    last = state["steps"][-1]
    program.step(last["ids"], None, last["out"])
    return state


def run(state):
    before = state["steps"][-1]
    for s in state["steps"]:
        state["program"].step(s["ids"], before["grad"], s["out"])
        before = s
    return [s["out"] for s in state["steps"]]


# ---- what a pass cannot do without ------------------------------------------------------------------------------------
def _distinct(count, n, alpha):
    """Expected number of distinct ids among n draws of one field."""
    if alpha == 0.0:
        return -count * math.expm1(-n / count)
    _, total = _zipf_head(count, alpha)
    edges = np.unique(np.round(np.geomspace(1, count + 1, 400)))        # ranks in groups of about equal weight
    middle = np.sqrt(edges[:-1] * (edges[1:] - 1).clip(min=1))
    return float(np.sum((edges[1:] - edges[:-1]) * -np.expm1(-n * np.power(middle, -alpha) / total)))


def work(case):
    fields = _layout(case)
    n = case["samples"] * case["fields"] * case["hot"]
    if case["whole"]:
        unique = _distinct(case["rows"], n, case["alpha"])
    else:
        unique = sum(_distinct(int(c), case["samples"] * case["hot"], case["alpha"]) for c in fields.card)
    row, out = 4 * case["width"], n // (case["hot"] if case["pooled"] else 1)
    # a look-up: the ids, every distinct row read once, every output row written
    pull_bytes, pull_flops = 8 * n + row * (unique + out), case["width"] * (n - out)
    # a push: the gradient rows read, every distinct row and its 8-byte version read and written
    push_bytes, push_flops = row * out + unique * (2 * row + 16), case["width"] * (n + unique)
    if case["path"] == "infer":
        return {"bytes": int(pull_bytes), "flops": int(pull_flops)}
    steps = 2 * case["feeding"]
    return {"bytes": int(steps * (pull_bytes + push_bytes)), "flops": int(steps * (pull_flops + push_flops))}


def tolerance(case):
    if case["path"] == "infer":
        return "exact"   # rows of the table, copied
    # The gradient rows of an id are added up in fp32, and the error of that sum grows with the occurrences of the hottest
    # id.  Against the same updates summed in 64 bits (four passes) the pulled rows are off by 1.3e-7 at 2048 samples,
    # 2.8e-7 at 65536, 2.9e-6 with 10 ids per field and exponent 1.4, and 9e-6 where those are pooled; the worst value by
    # 3 to 14 times that.
    fields = _layout(case)
    n = case["samples"] * case["hot"] * (case["fields"] if case["whole"] else 1)
    hottest = max(n / (c if case["alpha"] == 0.0 else _zipf_head(int(c), case["alpha"])[1]) for c in fields.card)
    rel = (5e-7 + 1e-10 * float(hottest)) * (math.sqrt(case["hot"]) if case["pooled"] else 1)
    return {"rel": rel, "max": 12 * rel}
