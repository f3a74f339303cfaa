"""What requests leave allocated for a SCALAR table beside its slot array."""
import gc

import numpy as np
import pytest

from conftest import announce
from helpers import to_dev, unique_keys

pytestmark = pytest.mark.gpu


def held_by(capi, make):
    """Bytes of device memory that what `make` returns holds on to."""
    import torch
    gc.collect()  # (tables of earlier tests)
    torch.cuda.synchronize()
    capi.device_trim()
    before = torch.cuda.mem_get_info()[0]
    made = make()
    capi.device_trim()
    after = torch.cuda.mem_get_info()[0]
    made.close()
    return before - after


@pytest.mark.parametrize("n,per_key", [(900_000, 16), ((3 << 19) - 1, 16), (3 << 19, 22)])
def test_the_key_cache_and_its_packed_keys(capi, dev, monkeypatch, n, per_key):
    """8 B for a cached key, 4 for its value and 4 for its slot number, 6 more where keys are packed; an eighth to spare, and the steps that
    the arrays come in, an eighth of the next power of two: a quarter at most. Beside each table 2 MiB for what the system rounds up."""
    import torch
    announce("key cache memory", n)
    S = 4
    keys = [to_dev(unique_keys(np.random.default_rng(s), n), dev) for s in range(S)]
    all_keys, pos = torch.cat(keys), np.arange(S + 1, dtype=np.uint64) * n
    vals, out = (torch.zeros(S * n, device=dev) for _ in range(2))

    def steps():
        group = capi.Group(S, capi.MODE_SCALAR, initial_capacity=n)
        for _ in range(4):
            group.push(all_keys, pos, vals, pos)
            group.pull(all_keys, pos, out)
            group.sync()
        return group

    with_cache = held_by(capi, steps)
    monkeypatch.setenv("PSKV_SCALAR_CACHE_MIN_KEYS", "0")
    without = held_by(capi, steps)
    assert per_key * n * S <= with_cache - without <= S * (1.125 * 1.25 * per_key * n + (2 << 20)), (with_cache - without) / (n * S)


@pytest.mark.parametrize("then", ["nothing", "pull", "small push"])
def test_the_room_that_a_push_streams_through(capi, dev, monkeypatch, then):
    """12 B per key for keys and values by bin, 4 for the places of the keys that are left, not quite 1 for where each tile's bins start,
    an eighth to spare and the steps that arrays come in: 1.125 * 1.125 * 17 = 21.5 B per key. It goes back with the first request
    that does not stream."""
    import torch
    announce("streaming memory", then)
    n = 4_000_000
    some = unique_keys(np.random.default_rng(1), n)
    keys, some = to_dev(some, dev), some[:1000]
    vals, out = torch.zeros(n, device=dev), torch.zeros(n, device=dev)

    def filled():
        t = capi.Table(capi.MODE_SCALAR, initial_capacity=10_000_000)  # (no growth is near, nor an array for one)
        t.prof_enable()
        t.push(keys, vals)
        if then == "pull":
            t.pull(keys, out)
        elif then == "small push":
            t.push(some, np.zeros(1000, np.float32))  # (from host memory: it does not stream)
        t.sync()
        return t

    monkeypatch.setenv("PSKV_STREAM", "1")
    t = filled()
    assert t.prof_read(capi.KERNEL_REHASH)[0] == 3
    t.close()
    with_room = held_by(capi, filled)
    monkeypatch.setenv("PSKV_STREAM", "0")
    without = held_by(capi, filled)
    assert with_room - without <= (21.5 * n if then == "nothing" else 0) + (2 << 20), (with_room - without) / n
