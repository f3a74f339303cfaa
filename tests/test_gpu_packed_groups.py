"""Requests over several SCALAR tables of which some keep their cached keys packed and some do not: below the size from which keys are
packed, with neighbours too far apart, or recorded a moment ago. Against the CPU oracle, and by the time that the comparison takes."""
import numpy as np
import pytest

from conftest import announce
from helpers import assert_bits_equal, to_dev
from test_gpu_store import _check_dump

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def packs_a_million(monkeypatch):
    monkeypatch.setenv("PSKV_PACK_MIN_KEYS", str(1 << 20))


def keys_of(rng, n, wide=False):
    keys = np.cumsum(rng.integers(2, 1 << 30, n, dtype=np.uint64))
    if wide:
        keys[n // 3:] += np.uint64(1 << 48)
    return keys


@pytest.mark.parametrize("ahead", [False, True])
def test_some_tables_pack(capi, orc, dev, ahead):
    import torch
    announce("packed groups", ahead)
    rng = np.random.default_rng(11)
    sets = [keys_of(rng, (1 << 20) + 77), keys_of(rng, (1 << 20) + 5, True), keys_of(rng, 200_003)]
    S = len(sets)
    group = capi.Group(S, capi.MODE_SCALAR, initial_capacity=3 << 20)
    stores = [orc.Store(orc.MODE_SCALAR) for _ in range(S)]
    answers = []

    def check():
        group.sync()
        for out, want in answers:
            assert_bits_equal(out.cpu().numpy(), want)
        answers.clear()

    def step(parts):
        pos = np.concatenate([[0], np.cumsum([p.size for p in parts])]).astype(np.uint64)
        vals = rng.standard_normal(int(pos[-1])).astype(np.float32)
        keys = to_dev(np.concatenate(parts), dev)
        out = torch.empty(vals.size, dtype=torch.float32, device=dev)
        group.push(keys, pos, to_dev(vals, dev), pos)
        group.pull(keys, pos, out)
        for s, p in enumerate(parts):
            stores[s].push(p, vals[int(pos[s]):int(pos[s + 1])])
        answers.append((out, np.concatenate([stores[s].pull(p)[0] for s, p in enumerate(parts)])))
        if not ahead:
            check()

    for turn in range(S):
        for _ in range(5):  # (a record, a comparison that finds the keys equal, one that packs them, and two of the packed keys)
            step(sets)
        other = [p.copy() for p in sets]
        other[turn][[0, 255, other[turn].size - 1]] += np.uint64(1)  # one table's keys are others once: it is recorded again
        step(other)
    for _ in range(5):
        step(sets)
    check()
    for s in range(S):
        _check_dump(group.tables[s], stores[s], "table %d" % s)


def test_a_packed_neighbour_costs_nothing(capi, dev):
    """A table that is not packed is compared as fast beside a packed one as it is by itself: 16 B per key are read, not 30. (Limit: the
    time by itself, with the packed keys' bytes, and a quarter; at 30 B it takes 1.6 times as long.)"""
    import torch
    announce("packed neighbours")
    n, rng = 4_000_000, np.random.default_rng(4)

    def fastest(sets):
        group = capi.Group(len(sets), capi.MODE_SCALAR, initial_capacity=2 * max(p.size for p in sets))
        pos = np.concatenate([[0], np.cumsum([p.size for p in sets])]).astype(np.uint64)
        keys = to_dev(np.concatenate(sets), dev)
        vals, out = torch.ones(keys.numel(), device=dev), torch.empty(keys.numel(), device=dev)
        for rep in range(20):
            if rep == 8:
                for t in group.tables:
                    t.prof_enable()
            group.push(keys, pos, vals, pos)
            group.pull(keys, pos, out)
            group.sync()
        took = np.concatenate([t.prof_samples(capi.KERNEL_SAME_KEYS) for t in group.tables])
        group.close()
        assert took.size >= 12
        return took.min()

    packable = keys_of(rng, 1 << 20)
    some = [keys_of(rng, n, wide=True) for _ in range(8)]
    alone, beside = fastest(some), fastest([packable] + some)
    assert beside < alone * (n * 8 * 16 + packable.size * 14) / (n * 8 * 16) * 1.25, (alone, beside)


def test_keys_that_a_recorded_step_left(capi, orc, dev):
    """Steps that are recorded leave no room behind the cached keys for packed ones: requests that name them the ordinary way are compared
    with the keys themselves, until an ordinary request has left keys there."""
    import torch
    announce("packed behind a recording")
    rng = np.random.default_rng(21)
    n = (1 << 20) + 300
    group, store = capi.Group(1, capi.MODE_SCALAR, initial_capacity=2 * n), orc.Store(orc.MODE_SCALAR)
    keys, others = keys_of(rng, n), keys_of(rng, n)
    pos = np.array([0, n], np.uint64)
    dk, do, out = to_dev(keys, dev), to_dev(others, dev), torch.empty(n, dtype=torch.float32, device=dev)
    vals = torch.zeros(n, dtype=torch.float32, device=dev)

    def push(of, host, how):
        new = rng.standard_normal(n).astype(np.float32)
        vals.copy_(torch.from_numpy(new))
        how(of)
        store.push(host, new)
        group.sync()

    def ordinary(of):
        group.push(of, pos, vals, pos)
        group.pull(of, pos, out)

    recordings = []
    push(dk, keys, lambda of: recordings.append(group.record(capi.REPLAY_PUSH | capi.REPLAY_PULL, of, pos, vals, pos, out=out)))
    push(dk, keys, lambda of: recordings[0].run())
    for of, host in ((dk, keys), (do, others), (dk, keys)):
        for _ in range(5):
            push(of, host, ordinary)
            assert_bits_equal(out.cpu().numpy(), store.pull(host)[0])
    _check_dump(group.tables[0], store, "behind a recording")
    recordings[0].close()
    group.close()
