"""Pushes that stream through the slot array of a SCALAR table (csrc/stream_push.h), against the CPU oracle, bit for bit:
shapes around tiles, bins and images, growths by every factor, runs, the key that marks an empty slot, homes that
crowd one bin or wrap around the end of the array."""
import numpy as np
import pytest

from conftest import announce
from helpers import KMAX, assert_bits_equal, to_dev, unique_keys
from test_gpu_store import _check_dump

pytestmark = pytest.mark.gpu

M1, M2 = 0xFF51AFD7ED558CCD, 0xC4CEB9FE1A85EC53


def unmixed(h):
    """The keys whose hashes (the finaliser of murmur3) are h."""
    h = h.copy()
    for mul in (M2, M1):
        h ^= h >> np.uint64(33)
        h *= np.uint64(pow(mul, -1, 1 << 64))
    return h ^ (h >> np.uint64(33))


@pytest.fixture
def streaming(monkeypatch):
    monkeypatch.setenv("PSKV_STREAM", "1")


def push_both(t, o, dev, keys, vals, skip=0):
    """`skip`: the request starts that many elements behind the start of its buffers."""
    pad_k, pad_v = np.concatenate([keys[:skip], keys]), np.concatenate([vals[:skip], vals])
    t.push(to_dev(pad_k, dev)[skip:], to_dev(pad_v, dev)[skip:])
    o.push(keys, vals)


def streamed(t, capi, pushes):
    """Whether so many pushes streamed, three launches or more each (a growth on its own is two)."""
    return t.prof_read(capi.KERNEL_REHASH)[0] >= 3 * pushes


@pytest.mark.parametrize("capacity,n,load", [(8_000, 2_731, 0.5), (8_000, 3_968, 0.5), (16_000, 8_192, 0.5), (16_000, 8_193, 0.5),
                                             (40_000, 31_000, 0.85), (1_000, 20_000, 0.25), (100_000, 60_000, 0.5),
                                             (30_000, 250_001, 0.5), (700_000, 1_000_000, 0.5)])
def test_pushes_of_held_and_new_keys(capi, orc, dev, streaming, capacity, n, load):
    announce("streamed pushes", capacity, n, load)
    rng = np.random.default_rng(n)
    t = capi.Table(capi.MODE_SCALAR, initial_capacity=capacity, max_load=load)
    o = orc.Store(orc.MODE_SCALAR)
    t.prof_enable()
    universe = unique_keys(rng, 4 * n)
    for rep in range(5):
        m = n - rep * (n // 50)  # (sizes that repeat leave a record instead, once they are told to)
        keys = np.sort(rng.choice(universe, size=m, replace=False))
        vals = rng.standard_normal(m).astype(np.float32)
        vals[::7] = -0.0
        push_both(t, o, dev, keys, vals, skip=rep % 3)
        if rep % 2 == 0:
            _check_dump(t, o, "push %d" % rep)
    assert streamed(t, capi, 2)
    _check_dump(t, o, "all")


@pytest.mark.parametrize("n", [2_900, 8_192, 50_000])
def test_runs_and_the_empty_marker(capi, orc, dev, streaming, n):
    announce("streamed runs", n)
    rng = np.random.default_rng(n)
    t, o = capi.Table(capi.MODE_SCALAR, initial_capacity=n), orc.Store(orc.MODE_SCALAR)
    t.prof_enable()
    for rep, share in enumerate((0.0, 0.01, 0.5, 1.0)):
        base = unique_keys(rng, n)
        times = np.where(rng.random(n) < share, rng.integers(2, 5, n), 1)
        keys = np.repeat(base, times)[:n]
        if rep % 2:
            keys[-1 - rep:] = KMAX
        push_both(t, o, dev, np.sort(keys), rng.standard_normal(n).astype(np.float32))
        _check_dump(t, o, "runs %d" % rep)
    assert streamed(t, capi, 3)


@pytest.mark.parametrize("first,last", [(0.0, 1.0), (0.999, 1.0), (0.0, 0.01), (0.49, 0.51)])
def test_homes_that_crowd(capi, orc, dev, streaming, first, last):
    """More keys in one bin than a workgroup holds, probe chains from image to image and around the end; then the array grows
    by two, and the request that makes it do so names keys that those chains have displaced."""
    announce("streamed crowds", first, last)
    rng = np.random.default_rng(int(first * 1000))
    t, o = capi.Table(capi.MODE_SCALAR, initial_capacity=32_000, max_load=0.5), orc.Store(orc.MODE_SCALAR)  # 65,536 slots
    t.prof_enable()
    lo, hi = int(first * 2**64), min(int(last * 2**64), 2**64 - 1)
    crowd = np.unique(unmixed(rng.integers(lo, hi, size=12_000, dtype=np.uint64)))
    crowd = crowd[crowd != KMAX]
    push_both(t, o, dev, crowd, rng.standard_normal(crowd.size).astype(np.float32))
    _check_dump(t, o, "crowd")
    for size in (12_500, 30_000):  # (beside 12,000 keys held; the second makes the table grow)
        others = np.setdiff1d(unique_keys(rng, size - 6_000), crowd)
        keys = np.sort(np.concatenate([rng.choice(crowd, 6_000, replace=False), others]))
        push_both(t, o, dev, keys, rng.standard_normal(keys.size).astype(np.float32))
        _check_dump(t, o, "crowd and others")
    assert streamed(t, capi, 3)


def test_the_same_keys_again_and_again(capi, orc, dev, streaming):
    """A push that streams leaves no record; once the pushes are known to name the same keys they do, and are served from it."""
    announce("streamed repeats")
    n = 200_000
    rng = np.random.default_rng(5)
    t, o = capi.Table(capi.MODE_SCALAR, initial_capacity=n), orc.Store(orc.MODE_SCALAR)
    keys, others = unique_keys(rng, n), unique_keys(rng, n)
    t.prof_enable()
    for rep in range(8):
        push_both(t, o, dev, keys if rep != 5 else others, rng.standard_normal(n).astype(np.float32))
        if rep % 2:
            t.sync()
    assert t.prof_read(capi.KERNEL_SAME_KEYS)[0] >= 1
    _check_dump(t, o, "repeats")


@pytest.mark.parametrize("S", [2, 5])
def test_shares_of_a_request(capi, orc, dev, streaming, S):
    """Tables of a group, all of which stream, some of which grow."""
    announce("streamed shares", S)
    rng = np.random.default_rng(S)
    group, stores = capi.Group(S, capi.MODE_SCALAR, initial_capacity=20_000), [orc.Store(orc.MODE_SCALAR) for _ in range(S)]
    for t in group.tables:
        t.prof_enable()
    begin, end = capi.server_ranges(S)
    for rep in range(5):
        keys = unique_keys(rng, 40_000 + 9_000 * rep, S)
        if rep >= 2:  # an uneven request
            keys = keys[(keys < begin[1]) | (rng.random(keys.size) < 0.02)]
        vals = rng.standard_normal(keys.size).astype(np.float32)
        dk = to_dev(keys, dev)
        pos, val_pos, _ = capi.slice_keys(dk, begin, end, nvals=keys.size)
        group.push(dk, pos, to_dev(vals, dev), val_pos)
        for s in range(S):
            part = slice(int(pos[s]), int(pos[s + 1]))
            if keys[part].size:
                stores[s].push(keys[part], vals[part])
    for s in range(S):
        _check_dump(group.tables[s], stores[s], "table %d" % s)
    assert launches(group, capi.KERNEL_REHASH) >= 3 * 5 and launches(group, capi.KERNEL_PUSH_SCALAR) == 0


def launches(group, kernel):
    """By all tables of the group."""
    return sum(t.prof_read(kernel)[0] for t in group.tables)


def test_shares_that_stream_by_themselves(capi, orc, dev):
    """A request of which the rule lets one share stream, with the growth that it asks for, and the others not: both ways in one request."""
    announce("streamed shares by the rule")
    rng = np.random.default_rng(77)
    group, stores = capi.Group(3, capi.MODE_SCALAR, initial_capacity=1_000_000), [orc.Store(orc.MODE_SCALAR) for _ in range(3)]
    for t in group.tables:
        t.prof_enable()
    sizes = (10_000, 2_000_000, 0)
    parts = [unique_keys(rng, n) if n else np.zeros(0, np.uint64) for n in sizes]
    pos = np.concatenate([[0], np.cumsum(sizes)]).astype(np.uint64)
    vals = rng.standard_normal(int(pos[-1])).astype(np.float32)
    group.push(to_dev(np.concatenate(parts), dev), pos, to_dev(vals, dev), pos)
    # k_split, k_stream_push, k_regrow_rest and k_push_left; one k_scalar
    assert launches(group, capi.KERNEL_REHASH) == 4 and launches(group, capi.KERNEL_PUSH_SCALAR) == 1
    for s, keys in enumerate(parts):
        if keys.size:
            stores[s].push(keys, vals[int(pos[s]):int(pos[s + 1])])
        _check_dump(group.tables[s], stores[s], "table %d" % s)


@pytest.mark.parametrize("grows", [False, True])
def test_cached_values_that_are_ahead_of_the_slots(capi, orc, dev, streaming, monkeypatch, grows):
    """A push that streams reads the slots, which may lack what pushes of repeated keys have added to the key cache alone. Their values
    go back first; the room that the push needs, which takes the key cache's buffers out of use, comes before that."""
    announce("streamed behind repeats", grows)
    monkeypatch.setenv("PSKV_SCALAR_CACHE_MIN_KEYS", "1000")
    rng = np.random.default_rng(8)
    n = 20_000
    t, o = capi.Table(capi.MODE_SCALAR, initial_capacity=n if grows else 4 * n), orc.Store(orc.MODE_SCALAR)
    t.prof_enable()
    keys = np.concatenate([unique_keys(rng, n - 1), [np.uint64(KMAX)]])
    for rep in range(3):
        compared = t.prof_read(capi.KERNEL_SAME_KEYS)[0]
        for _ in range(8):
            push_both(t, o, dev, keys, rng.standard_normal(n).astype(np.float32))
            t.sync()
        assert t.prof_read(capi.KERNEL_SAME_KEYS)[0] > compared  # (the last ones have been served from the cache)
        before = t.prof_read(capi.KERNEL_REHASH)[0]
        others = np.unique(np.concatenate([rng.choice(keys, n // 2, replace=False), unique_keys(rng, n + 5_000 * rep)]))
        push_both(t, o, dev, others, rng.standard_normal(others.size).astype(np.float32))
        assert t.prof_read(capi.KERNEL_REHASH)[0] - before in ((3, 4) if grows else (3,))
        _check_dump(t, o, "ahead %d" % rep)


@pytest.mark.parametrize("capacity,images", [(30_000_000, 4), (60_000_000, 8), (120_000_000, 16)])
def test_bins_of_many_images(capi, orc, dev, streaming, capacity, images):
    """Arrays of 64M, 128M and 256M slots: the bins are as many as there may be, with four images each and more."""
    announce("streamed images", images)
    rng = np.random.default_rng(images)
    t, o = capi.Table(capi.MODE_SCALAR, initial_capacity=capacity), orc.Store(orc.MODE_SCALAR)
    t.prof_enable()
    assert t.counters()["slots"] == 4096 * 4096 * images
    universe = unique_keys(rng, 60_000)
    for rep in range(3):
        keys = np.sort(rng.choice(universe, 30_000 + rep, replace=False))
        push_both(t, o, dev, keys, rng.standard_normal(keys.size).astype(np.float32))
    assert t.prof_read(capi.KERNEL_REHASH)[0] == 9
    _check_dump(t, o, "images")


@pytest.mark.parametrize("first,last", [(0.0, 1.0), (0.999, 1.0), (0.49, 0.51)])
def test_values_that_are_no_numbers(capi, dev, monkeypatch, first, last):
    """Infinities and NaNs, each with a payload of its own: what a push leaves that streams, with and without a growth, is to the bit
    what one leaves that goes through the slots. (The sum of two NaNs is one of the two: which one depends on their order.)"""
    announce("streamed NaNs", first, last)
    rng = np.random.default_rng(int(first * 1000) + 7)
    tables = []
    for streams in ("0", "1"):
        monkeypatch.setenv("PSKV_STREAM", streams)
        tables.append(capi.Table(capi.MODE_SCALAR, initial_capacity=32_000, max_load=0.5))
        tables[-1].prof_enable()
    lo, hi = int(first * 2**64), min(int(last * 2**64), 2**64 - 1)
    crowd = np.unique(unmixed(rng.integers(lo, hi, size=12_000, dtype=np.uint64)))
    crowd = crowd[crowd != KMAX]

    def push(keys, number):
        bits = np.uint32(0x7FC00000 + number * 0x100000) + np.arange(keys.size, dtype=np.uint32)  # quiet, other ones every time
        vals = np.where(rng.random(keys.size) < 0.7, bits.view(np.float32),
                        rng.choice(np.array([np.inf, -np.inf, 1.5, -0.0], np.float32), keys.size))
        vals[rng.random(keys.size) < 0.2] *= np.float32(-1)
        for t in tables:
            t.push(to_dev(keys, dev), to_dev(vals, dev))
        a, b = (t.dump() for t in tables)
        assert np.array_equal(a[0], b[0])
        assert_bits_equal(b[2], a[2], "push %d" % number)

    push(crowd, 0)
    for number, size in ((1, 12_500), (2, 30_000)):  # (the second makes the tables grow)
        others = np.setdiff1d(unique_keys(rng, size - 6_000), crowd)
        runs = np.repeat(rng.choice(others, 50, replace=False), 2)
        push(np.sort(np.concatenate([rng.choice(crowd, 6_000, replace=False), others, runs, np.full(2, KMAX, np.uint64)])), number)
    assert streamed(tables[1], capi, 3)
    assert tables[0].prof_read(capi.KERNEL_REHASH)[0] == 2  # (the growth)
