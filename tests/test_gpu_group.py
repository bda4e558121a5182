"""Several shards on one GPU behind the in-process loopback: the reference's multi-GPU tests
(tests/test_update.py, tests/check.py) with their closed forms, plus step-by-step parity with the oracle
including cache hit / miss / refresh decisions and bounded staleness."""
import threading

import numpy as np
import pytest
import torch

from hetuctr_amd import capi
from tests.gpu_util import Pair, INT_ITEMS_PRE, INT_ITEMS_POST, assert_close
from tests.helpers import zipf_sampler

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)


def update_pair(nrank, length, width, bounds=(0, 0), init=("Zero", 0.0, 0.0), lr=-1.0, cache="lower", seed=0):
    rs = np.random.RandomState(seed)
    root = rs.randint(nrank, size=length).astype(np.uint8)
    if cache == "lower":      # tests/test_update.py:21
        storage = [np.where(root <= r)[0].astype(np.int64) for r in range(nrank)]
    elif cache == "none":     # tests/check.py:30
        storage = [np.where(root == r)[0].astype(np.int64) for r in range(nrank)]
    else:                     # a random third of the remote rows, shuffled
        storage = []
        for r in range(nrank):
            own, other = np.where(root == r)[0], np.where(root != r)[0]
            st = np.concatenate([own, rs.choice(other, other.shape[0] // 3, replace=False)])
            rs.shuffle(st)
            storage.append(st.astype(np.int64))
    return Pair(nrank, length, width, root, storage, init=init, lr=lr, bounds=bounds, seed=seed), root


@pytest.mark.parametrize("nrank", [2, 4])
def test_occurrence_count_closed_form(nrank):
    say("test_update::test_one nrank", nrank)
    length, width, bs = 1024, 128, 1024
    p, root = update_pair(nrank, length, width)
    rngs = [np.random.RandomState(r) for r in range(nrank)]
    store = np.zeros(length)
    p.preprocess([np.zeros(0, np.int64)] * nrank)
    prev = [np.zeros(0, np.int64)] * nrank
    for step in range(50):
        for r in range(nrank):
            np.add.at(store, prev[r], 1.0)
        keys = [rngs[r].randint(length, size=bs).astype(np.int64) for r in range(nrank)]
        p.preprocess(keys)
        out, ref = p.push_pull([np.ones((prev[r].shape[0], width), np.float32) for r in range(nrank)])
        for r in range(nrank):
            assert np.array_equal(out[r][:, 0], store[keys[r]].astype(np.float32)), (step, r)
            assert np.array_equal(out[r], ref[r])
        prev = keys
    p.compare_ints(INT_ITEMS_PRE + INT_ITEMS_POST)
    p.close()


def test_gradient_sum_closed_form():
    say("test_update::test_two")
    nrank, length, width, bs = 4, 1024, 16, 1024
    p, root = update_pair(nrank, length, width)
    rngs = [np.random.RandomState(100 + r) for r in range(nrank)]
    store = np.zeros((length, width))
    prev = [np.zeros(0, np.int64)] * nrank
    for step in range(50):
        grads = [rngs[r].rand(prev[r].shape[0], width).astype(np.float32) for r in range(nrank)]
        for r in range(nrank):
            np.add.at(store, prev[r], grads[r].astype(np.float64))
        keys = [rngs[r].randint(length, size=bs).astype(np.int64) for r in range(nrank)]
        p.preprocess(keys)
        out, ref = p.push_pull(grads)
        for r in range(nrank):
            assert np.max(np.abs(out[r] - store[keys[r]])) < 1e-4   # tests/test_update.py:70
            assert_close(out[r], ref[r], 1e-5, "step %d rank %d" % (step, r))
        prev = keys
    p.close()


@pytest.mark.parametrize("nrank,bounds,cache,width", [(4, (0, 0), "lower", 8), (4, (10, 10), "none", 128),
                                                      (3, (2, 3), "third", 20), (8, (1, 0), "third", 64),
                                                      (2, (0, 5), "lower", 3)])
def test_stepwise_parity_with_staleness(nrank, bounds, cache, width):
    say("stepwise", nrank, bounds, cache, width)
    length, bs = 3000, 2500
    p, root = update_pair(nrank, length, width, bounds=bounds, init=("Uniform", -1.0, 1.0), lr=0.5, cache=cache, seed=3)
    rng = np.random.default_rng(nrank * 10 + bounds[0])
    draw = zipf_sampler(length, 1.05, rng)
    prev_n = [0] * nrank
    for step in range(12):
        keys = [draw(bs - 7 * r) if step % 3 else rng.integers(0, length, bs - 7 * r).astype(np.int64) for r in range(nrank)]
        if step == 5:
            keys[0] = np.zeros(0, np.int64)       # one shard sits a step out
        p.preprocess(keys)
        p.compare_ints(INT_ITEMS_PRE, "step %d" % step)
        grads = [rng.normal(0, 0.1, size=(prev_n[r], width)).astype(np.float32) for r in range(nrank)]
        if step == 8:
            grads[1] = None                        # inference on one shard
        out, ref = p.push_pull(grads)
        p.compare_ints(INT_ITEMS_POST, "step %d" % step)
        for r in range(nrank):
            assert_close(out[r], ref[r], 1e-5, "dst step %d rank %d" % (step, r))
        p.compare_state(1e-5, "step %d" % step)
        prev_n = [k.shape[0] for k in keys]
    p.close()


@pytest.mark.parametrize("nrank,cache,width", [(3, "third", 20), (5, "lower", 128)])
def test_steps_without_a_look_at_the_index(nrank, cache, width):
    # Nothing is fetched between preprocess and push_pull, so push_pull finds the index of the current batches still
    # running and never waits for it on the host: the queries are placed and counted on the device, and the grids of
    # the query kernels are cut from what the step before had.  Batch sizes jump by orders of magnitude both ways,
    # shards sit steps out, one step has no keys at all.
    say("no look at the index", nrank, cache, width)
    length = 40_000
    p, root = update_pair(nrank, length, width, bounds=(1, 2), init=("Uniform", -1.0, 1.0), lr=0.5, cache=cache, seed=5)
    rng = np.random.default_rng(nrank)
    draw = zipf_sampler(length, 1.05, rng)
    sizes = [300, 120_000, 7, 60_000, 0, 1, 90_000, 2_000]
    prev_n = [0] * nrank
    for step, bs in enumerate(sizes):
        keys = [draw(max(bs - 5 * r, 0)) if step % 2 else rng.integers(0, length, max(bs - 5 * r, 0)).astype(np.int64)
                for r in range(nrank)]
        if step in (1, 6):
            keys[step % nrank] = np.zeros(0, np.int64)     # a shard sits out a large step
        p.preprocess(keys, device_keys=bool(step % 3))
        grads = [rng.normal(0, 0.1, size=(prev_n[r], width)).astype(np.float32) for r in range(nrank)]
        out, ref = p.push_pull(grads)
        p.compare_ints(INT_ITEMS_PRE + INT_ITEMS_POST, "step %d" % step)
        for r in range(nrank):
            assert_close(out[r], ref[r], 1e-5, "dst step %d rank %d" % (step, r))
        p.compare_state(1e-5, "step %d" % step)
        prev_n = [k.shape[0] for k in keys]
    p.close()


@pytest.mark.parametrize("bounds,cached", [((0, 0), (0,)), ((2, 3), tuple(range(8)))])
def test_partitioned_table_with_hot_row_cache(bounds, cached):
    # the 8-way partition of the Criteo-like table at 1/100 scale: uniform owners, the hottest 10 % of the remote
    # rows cached; either rank 0 alone feeds batches while the peers only serve, or every rank does
    from hetuctr_amd import workloads
    say("partitioned", bounds, cached)
    cfg = workloads.CONFIGS["cfg3"]
    ks = workloads.KeyStream(cfg, seed=0, scale=0.01)
    R, width = cfg["nrank"], cfg["width"]
    root, storage = workloads.shard_layout(ks, R, cfg["cache_frac"], cached_ranks=cached)
    p = Pair(R, ks.rows, width, root, storage, init=("Uniform", -0.1, 0.1), lr=cfg["lr"], bounds=bounds, seed=0)
    rng = np.random.default_rng(4)
    prev_n = [0] * R
    totals = np.zeros(6)
    for step in range(5):
        keys = [ks.batch() if r in cached else np.zeros(0, np.int64) for r in range(R)]
        p.preprocess(keys, device_keys=True)
        p.compare_ints(INT_ITEMS_PRE, "step %d" % step)
        out, ref = p.push_pull([rng.normal(0, 1e-2, size=(prev_n[r], width)).astype(np.float32) for r in range(R)])
        p.compare_ints(INT_ITEMS_POST, "step %d" % step)
        for r in cached:
            assert_close(out[r], ref[r], 1e-5, "dst step %d rank %d" % (step, r))
        for r in range(R):
            totals += p.tables[r].fetch(capi.STATS)[:6]
        prev_n = [k.shape[0] for k in keys]
    p.compare_state(1e-5, "end")
    hit, miss, refreshed, pushed, returned, received = totals
    assert hit > 0 and miss > 0 and pushed == received and returned == miss + refreshed
    assert refreshed > 0                            # at least the first fetch of every touched cached row
    p.close()


def test_layout_from_the_offline_partitioner():
    # the whole offline flow at 1/100 scale: click log -> partitioner (owners, cache candidates, samples per rank)
    # -> eight tables that train on their own samples; parity with the oracle, and fewer rows cross ranks than
    # with uniform owners and the hottest rows cached
    from hetuctr_amd import workloads
    say("layout from the partitioner")
    cfg = workloads.CONFIGS["cfg3"]
    R, width = cfg["nrank"], cfg["width"]
    ranks = tuple(range(R))
    ks = workloads.KeyStream(cfg, seed=0, scale=0.01)
    steps = 4
    root, storage, batches, info = workloads.partitioned_layout(ks, R, cfg["cache_frac"], R * ks.samples * (steps + 1),
                                                                ks.samples, rounds=3, cached_ranks=ranks)
    assert info["cost_per_round"][-1] < 0.8 * info["cost_per_round"][0]
    assert min(len(b) for b in batches.values()) >= steps
    for r in ranks:                                   # a rank stores what it owns and nothing twice
        assert np.array_equal(np.sort(storage[r][:int((root == r).sum())]), np.flatnonzero(root == r))
        assert np.unique(storage[r]).shape[0] == storage[r].shape[0]

    def run(root, storage, batches, check):
        p = Pair(R, ks.rows, width, root, storage, init=("Uniform", -0.1, 0.1), lr=cfg["lr"], bounds=(2, 3), seed=0)
        rng = np.random.default_rng(4)
        prev_n = [0] * R
        totals = np.zeros(6)
        for step in range(steps):
            keys = [batches[r][step] for r in range(R)]
            p.preprocess(keys, device_keys=True)
            if check:
                p.compare_ints(INT_ITEMS_PRE, "step %d" % step)
            out, ref = p.push_pull([rng.normal(0, 1e-2, size=(prev_n[r], width)).astype(np.float32) for r in range(R)])
            if check:
                p.compare_ints(INT_ITEMS_POST, "step %d" % step)
                for r in range(R):
                    assert_close(out[r], ref[r], 1e-5, "dst step %d rank %d" % (step, r))
            for r in range(R):
                totals += p.tables[r].fetch(capi.STATS)[:6]
            prev_n = [k.shape[0] for k in keys]
        if check:
            p.compare_state(1e-5, "end")
        p.close()
        return totals

    hit, miss, refreshed, pushed, returned, received = run(root, storage, batches, True)
    assert pushed == received and returned == miss + refreshed
    ks2 = workloads.KeyStream(cfg, seed=0, scale=0.01)
    root2, storage2 = workloads.shard_layout(ks2, R, cfg["cache_frac"], cached_ranks=ranks)
    plain = {r: [ks2.batch() for _ in range(steps)] for r in range(R)}
    _, miss2, refreshed2, pushed2, returned2, _ = run(root2, storage2, plain, False)
    say("  rows returned by owners: %d partitioned, %d uniform owners; pushed %d vs %d" %
        (returned, returned2, pushed, pushed2))
    assert returned < returned2 and pushed < pushed2


def test_hand_computed_staleness_scenario():
    # same scenario as tests/test_oracle_update.py::test_staleness_scenario_both_update, on the GPU
    root = np.array([0, 1], np.uint8)
    p = Pair(2, 2, 4, root, [np.array([0, 1]), np.array([1])], lr=-1.0, bounds=(1, 2))
    one = np.array([1], np.int64)
    r0, r1 = [], []
    n_prev = 0
    for step in range(4):
        p.preprocess([one, one])
        g = np.ones((n_prev, 4), np.float32)
        out, ref = p.push_pull([g, g]); n_prev = 1
        r0.append(float(out[0][0, 0])); r1.append(float(out[1][0, 0]))
    assert r0 == [0.0, 1.0, 4.0, 5.0] and r1 == [0.0, 1.0, 2.0, 6.0]
    assert p.tables[0].fetch(capi.STATS).tolist()[:3] == [1, 0, 0]
    p.close()


def test_per_shard_calls_from_threads():
    # the reference's per-process call pattern (tests/check.py:40-44), one thread per shard
    say("threads")
    nrank, length, width, bs = 4, 1024, 32, 512
    p, root = update_pair(nrank, length, width, bounds=(0, 0))
    rng = np.random.RandomState(5)
    steps = 6
    keys = [[rng.randint(length, size=bs).astype(np.int64) for _ in range(steps)] for _ in range(nrank)]
    outs = [[None] * steps for _ in range(nrank)]
    errors = []

    def worker(r):
        try:
            dst = torch.zeros((bs, width), device="cuda")
            grad = torch.ones((bs, width), device="cuda")
            torch.cuda.synchronize()
            for s in range(steps):
                p.tables[r].preprocess(keys[r][s].ctypes.data, bs)
                p.tables[r].push_pull(grad.data_ptr() if s else 0, dst.data_ptr())
                outs[r][s] = dst.cpu().numpy().copy()
        except Exception as e:  # pragma: no cover
            errors.append(e)

    ts = [threading.Thread(target=worker, args=(r,)) for r in range(nrank)]
    [t.start() for t in ts]
    [t.join(60) for t in ts]
    assert not errors, errors
    store = np.zeros(length)
    for s in range(steps):
        if s > 0:
            for r in range(nrank):
                np.add.at(store, keys[r][s - 1], 1.0)
        for r in range(nrank):
            assert np.array_equal(outs[r][s][:, 0], store[keys[r][s]].astype(np.float32)), (s, r)
    p.close()


def test_group_errors():
    root = np.array([0, 1], np.uint8)
    t0 = capi.Table(0, 2, 0, "10.0.0.1", 999, 2, 4, 0, 0, root, np.array([0]), ("Zero", 0, 0), 0.1)
    k = np.array([0], np.int64)
    with pytest.raises(RuntimeError, match="every rank|missing ranks"):
        capi.group_preprocess([t0], [k.ctypes.data], [1])
    with pytest.raises(RuntimeError, match="already exists"):
        capi.Table(0, 2, 0, "10.0.0.1", 999, 2, 4, 0, 0, root, np.array([0]), ("Zero", 0, 0), 0.1)
    t0.close()


@pytest.mark.parametrize("nrank", [33, 200])
def test_many_shards(nrank):
    """More shards than any benchmark uses (the owner-side kernels walk up to 256 sources per target row, the exchanges
    describe nrank * nrank segment pairs): three steps with caches and staleness against the oracle."""
    rng = np.random.default_rng(nrank)
    length, width = 5000, 12
    root = rng.integers(0, nrank, size=length).astype(np.uint8)
    storage = []
    for r in range(nrank):
        own, other = np.flatnonzero(root == r), np.flatnonzero(root != r)
        storage.append(np.concatenate([own, rng.choice(other, other.shape[0] // 4, replace=False)]).astype(np.int64))
    p = Pair(nrank, length, width, root, storage, init=("Uniform", -0.1, 0.1), lr=0.1, bounds=(1, 2))
    draw = zipf_sampler(length, 1.2, rng)
    prev = [0] * nrank
    for step in range(3):
        sizes = [int(rng.choice([0, 40, 400])) for _ in range(nrank)]
        keys = [draw(k) if k else np.zeros(0, np.int64) for k in sizes]
        p.preprocess(keys)
        p.compare_ints(INT_ITEMS_PRE, "step %d" % step)
        out, ref = p.push_pull([rng.normal(0, 0.1, size=(prev[r], width)).astype(np.float32) for r in range(nrank)])
        p.compare_ints(INT_ITEMS_POST, "step %d" % step)
        for r in range(nrank):
            assert_close(out[r], ref[r], 1e-5, "dst step %d rank %d" % (step, r))
        p.compare_state(1e-5, "step %d" % step)
        prev = sizes
    p.close()


@pytest.mark.parametrize("nrank,width", [(8, 16), (9, 5), (17, 8)])
def test_groups_of_more_shards_than_a_launch_serves(nrank, width):
    # the kernels on the shards' own batches serve eight shards per launch: exactly eight, one more, two full launches and
    # one; batches of very different sizes and empty ones side by side, in changing places; outputs and gradients of some
    # shards off by four bytes; a step without gradients in between
    say("group launches, shards", nrank, "width", width)
    p, _ = update_pair(nrank, 4_000, width, bounds=(2, 3), init=("Uniform", -0.1, 0.1), lr=0.05, cache="third", seed=nrank)
    rng = np.random.default_rng(nrank)
    draw = zipf_sampler(4_000, 1.2, rng)
    sizes = [0, 1, 300, 5_000, 40]
    prev = [0] * nrank
    for step in range(6):
        ns = [sizes[(r + 2 * step) % len(sizes)] for r in range(nrank)]
        keys = [draw(n) if n else np.zeros(0, np.int64) for n in ns]
        p.preprocess(keys, device_keys=True)
        p.compare_ints(INT_ITEMS_PRE, "step %d" % step)
        grads = [None if step == 3 else rng.normal(0, 1e-2, size=(n, width)).astype(np.float32) for n in prev]
        bufs, dst, gptr = [], [], []
        for r in range(nrank):
            off = (r + step) % 2
            d = torch.full((ns[r] * width + 1,), float("nan"), device="cuda")
            dst.append(d[off:off + ns[r] * width])
            g = torch.zeros(prev[r] * width + 1, device="cuda")
            if grads[r] is not None:
                g[off:off + prev[r] * width].copy_(torch.from_numpy(grads[r].reshape(-1)))
            gptr.append(0 if grads[r] is None or not prev[r] else g.data_ptr() + 4 * off)
            bufs += [d, g]
        torch.cuda.synchronize()
        capi.group_push_pull(p.tables, gptr, [d.data_ptr() if d.numel() else 0 for d in dst])
        ref = p.oracle.push_pull(grads)
        p.compare_ints(INT_ITEMS_POST, "step %d" % step)
        for r in range(nrank):
            assert_close(dst[r].cpu().numpy().reshape(-1, width), ref[r], 1e-5, "dst step %d rank %d" % (step, r))
        p.compare_state(1e-5, "step %d" % step)
        prev = ns
    p.close()


@pytest.mark.parametrize("sizes,width", [
    # tile-sorted batches of one shape in more shards than a launch serves, one-block ones and an empty one among them
    ([8193 + 431 * r for r in range(13)] + [8192, 40, 0, 2_500], 8),
    # three shapes of the index side by side: four and two keys per thread of a sort tile, and one block
    ([270_000, 9_000, 300], 5),
    # one large batch beside many small ones: a launch's blocks belong to very different numbers of rows
    ([120_000] + [60] * 8, 12)])
def test_batches_of_unequal_shape_in_shared_launches(sizes, width):
    nrank = len(sizes)
    say("shared launches, keys per shard", sizes, "width", width)
    p, _ = update_pair(nrank, 30_000, width, bounds=(1, 2), init=("Uniform", -0.1, 0.1), lr=0.05, cache="third", seed=nrank)
    rng = np.random.default_rng(nrank)
    draw = zipf_sampler(30_000, 1.1, rng)
    prev = [0] * nrank
    for step in range(4):
        ns = [sizes[(r + 2 * step) % nrank] for r in range(nrank)]
        keys = [draw(n) for n in ns]
        # the ids of every other shard lie in host memory
        dev = [None if (r + step) % 2 else torch.from_numpy(keys[r]).cuda() for r in range(nrank)]
        torch.cuda.synchronize()
        ptrs = [0 if not ns[r] else keys[r].ctypes.data if dev[r] is None else dev[r].data_ptr() for r in range(nrank)]
        capi.group_preprocess(p.tables, ptrs, ns)
        p.n = ns
        p.oracle.preprocess(keys)
        p.compare_ints(INT_ITEMS_PRE, "step %d" % step)
        out, ref = p.push_pull([rng.normal(0, 1e-2, size=(n, width)).astype(np.float32) for n in prev])
        p.compare_ints(INT_ITEMS_POST, "step %d" % step)
        for r in range(nrank):
            assert_close(out[r], ref[r], 1e-5, "dst step %d rank %d" % (step, r))
        p.compare_state(1e-5, "step %d" % step)
        prev = ns
    p.close()


@pytest.mark.parametrize("sizes", [(1, 2, 3), (16, 17, 18), (15, 33, 400), (289, 5000, 290), (5000, 0, 4999)])
def test_pushes_of_unequal_length_to_one_owner(sizes):
    # every source's range of ids between two rows of the longest segment is found by searches over segments of these lengths
    print("pushed segments", sizes, flush=True)
    rng = np.random.default_rng(3)
    length, R, width = 24_000, len(sizes), 8
    root = np.full(length, 2, np.uint8)                 # everything belongs to the last shard
    storage = [np.zeros(0, np.int64), np.zeros(0, np.int64), np.arange(length, dtype=np.int64)]
    p = Pair(R, length, width, root, storage, init=("Uniform", -0.01, 0.01), lr=0.05)
    prev = [0] * R
    for step in range(2):
        keys = [rng.permutation(length)[:n].astype(np.int64) for n in sizes]
        p.preprocess(keys, device_keys=True)
        out, ref = p.push_pull([rng.normal(0, 1e-2, size=(n, width)).astype(np.float32) for n in prev])
        for r in range(R):
            assert_close(out[r], ref[r], 1e-5, "dst step %d rank %d" % (step, r))
        p.compare_state(1e-5, "step %d" % step)
        p.compare_ints(INT_ITEMS_POST, "step %d" % step)
        prev = list(sizes)
    p.close()


@pytest.mark.parametrize("large", [0, 1])
def test_one_shard_reads_its_ids_by_word_and_the_other_by_event(large):
    # 2^21 + 1 keys are one block too many for the word that says the ids are read, so the call waits for one shard by an
    # event and for the other by the word; either may hold a bad id, and both buffers are the caller's when the call returns
    say("ids read by word and by event, large batch at", large)
    rng = np.random.default_rng(11)
    length, width, ns = 5_000, 1, [700, 700]
    ns[large] = (1 << 21) + 1
    root = rng.integers(0, 2, size=length).astype(np.uint8)
    p = Pair(2, length, width, root, [np.flatnonzero(root == r).astype(np.int64) for r in range(2)],
             init=("Uniform", -0.01, 0.01), lr=0.05)
    side = torch.cuda.Stream()
    bad = [None, large, None, 1 - large, None]
    for step, where in enumerate(bad):
        if where is not None:
            ids = [torch.full((n,), 3, dtype=torch.int64, device="cuda") for n in ns]
            ids[where][-1] = length
            torch.cuda.synchronize()
            with pytest.raises(RuntimeError, match="outside"):
                capi.group_preprocess(p.tables, [d.data_ptr() for d in ids], ns)
            continue
        p.preprocess([rng.integers(0, length, n) for n in ns], device_keys=True)
        with torch.cuda.stream(side):
            for d in p.keep:
                d.fill_(7)
        out, ref = p.push_pull([None, None])
        for r in range(2):
            assert_close(out[r], ref[r], 1e-5, "dst step %d rank %d" % (step, r))
    p.close()


def fill_the_gpu(leave):
    # holds of device memory after which at most `leave` bytes are free
    held = []
    torch.cuda.empty_cache()
    torch.cuda.synchronize()
    for piece in (1 << 30, 16 << 20):
        while torch.cuda.mem_get_info()[0] > leave + piece // 2:
            free = torch.cuda.mem_get_info()[0]
            try:
                held.append(torch.empty(max(free - (1 << 30), piece), dtype=torch.uint8, device="cuda"))
            except torch.OutOfMemoryError:
                break
    assert torch.cuda.mem_get_info()[0] <= leave + (16 << 20)
    return held


@pytest.mark.parametrize("repeats", [2, 20, 400])
def test_step_without_memory_for_its_push_plan(repeats):
    # The first step of a pair of batch buffers plans their push last, behind everything else it allocates.  No room for that plan:
    # the step fails, and the steps after it do what they do where there was room (nothing is pushed in the step that
    # fails and no row is cached: the tables are the same either way).
    n, width, leave = 20_000_000, 4, 48 << 20        # the plan asks for 90 MB at a time
    length = n // repeats
    say("no memory for a push plan", repeats)
    gen = torch.Generator(device="cuda")
    tables = []
    for short in (True, False):
        gen.manual_seed(repeats)
        root = (np.arange(length) % 2).astype(np.uint8)
        p = Pair(2, length, width, root, [np.nonzero(root == r)[0].astype(np.int64) for r in range(2)],
                 init=("Uniform", -0.01, 0.01), lr=0.05, with_oracle=False)
        tables.append(p.tables)
        dst = torch.empty((n, width), device="cuda")
        prev = 0
        for step in range(4):
            k = n if step < 2 else n // 4
            ids = torch.randperm(n, device="cuda", generator=gen)[:k] % length
            grad = torch.randn((prev, width), device="cuda", generator=gen) if step > 1 else None
            torch.cuda.synchronize()
            capi.group_preprocess(p.tables, [ids.data_ptr(), 0], [k, 0])
            args = (p.tables, [grad.data_ptr() if grad is not None else 0, 0], [dst.data_ptr(), 0])
            if short and step == 1:
                held = fill_the_gpu(leave)
                with pytest.raises(RuntimeError, match="out of memory"):
                    capi.group_push_pull(*args)
                del held
                torch.cuda.empty_cache()
            else:
                capi.group_push_pull(*args)
            prev = k
        del ids, grad, dst
    for r in range(2):
        for item in (capi.EMBEDDING, capi.VERSION):
            a, b = (t[r].fetch(item) for t in tables)
            assert np.array_equal(a, b), "shard %d item %d: %d of %d entries differ" % (r, item, (a != b).sum(), a.size)
    for t in tables[0] + tables[1]:
        t.close()


@pytest.mark.parametrize("width,n", [(32, 9_000), (1, 90_000), (16, 110_000), (37, 40_000), (64, 12_301), (300, 5_000)])
def test_cached_rows_come_back_in_every_way_of_the_refresh(width, n):
    # a group of lanes per key (the first); a wave per 64 keys, or, where most rows came back in the step before or the batch is of
    # medium size, per as many keys as its groups copy in one go: every shard caches everything, and what the others
    # push comes back in the next step; look-ups, where nothing does, behind those
    say("refresh", width, n)
    rng = np.random.default_rng(width)
    length = n
    root = rng.integers(0, 2, length).astype(np.uint8)
    everything = np.arange(length, dtype=np.int64)
    p = Pair(2, length, width, root, [everything, everything], init=("Uniform", -0.01, 0.01), lr=0.05)
    for step in range(6):
        k = [n - 3 * step, n - 7 * step]
        p.preprocess([rng.integers(0, length, m) for m in k], device_keys=True)
        train = 0 < step < 4
        out, ref = p.push_pull([rng.normal(0, 1e-3, size=(m, width)).astype(np.float32) if train else None for m in prev] if step else [None] * 2)
        for r in range(2):
            assert_close(out[r], ref[r], 1e-5, "dst step %d rank %d" % (step, r))
        prev = k
    p.compare_state(1e-5, "end")
    p.compare_ints([capi.VERSION, capi.UPDATES, capi.STATS], "end")
    p.close()


@pytest.mark.parametrize("bound", [0, 5])
def test_queries_built_beside_the_owners_and_behind_them(bound):
    # two shards that push n x 128 floats each: 56 Mi floats times shards are reached at 114,688 keys of each.  Steps on either side
    # of that take turns, with a third of the other shard's rows cached, so that the queries carry versions the pushes move
    say("queries beside the owners", bound)
    rng = np.random.default_rng(bound)
    length, width = 50_000, 128
    p, root = update_pair(2, length, width, bounds=(bound, bound), init=("Uniform", -0.01, 0.01), lr=0.05, cache="third", seed=3)
    prev = None
    for step, n in enumerate([114_688, 114_687, 120_000, 114_680, 114_688, 5_000, 300]):
        k = [n, n]
        p.preprocess([rng.integers(0, length, m) for m in k], device_keys=True)
        out, ref = p.push_pull([rng.normal(0, 1e-3, size=(m, width)).astype(np.float32) for m in prev] if prev else [None] * 2)
        for r in range(2):
            assert_close(out[r], ref[r], 1e-5, "dst step %d rank %d" % (step, r))
        prev = k
    p.compare_state(1e-5, "end")
    p.compare_ints([capi.VERSION, capi.UPDATES, capi.STATS], "end")
    p.close()
