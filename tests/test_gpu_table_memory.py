"""What requests leave allocated for a SCALAR table beside its slot array."""
import numpy as np
import pytest

from conftest import announce
from helpers import to_dev, unique_keys

pytestmark = pytest.mark.gpu


def held_by(capi, make):
    """Bytes of device memory that what `make` returns holds on to."""
    import torch
    torch.cuda.synchronize()
    capi.device_trim()
    before = torch.cuda.mem_get_info()[0]
    made = make()
    capi.device_trim()
    after = torch.cuda.mem_get_info()[0]
    made.close()
    return before - after


def test_the_key_cache_of_keys_that_are_never_packed(capi, dev, monkeypatch):
    """8 B for a cached key, 4 for its value and 4 for its slot number, an eighth to spare and the steps that the arrays come in (an
    eighth of a power of two): 1.125 * 1.125 * 16 = 20.3 B per key. Beside each table 2 MiB for what the system rounds up."""
    import torch
    announce("key cache memory")
    n, S = 900_000, 8
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
    assert 16 * n * S <= with_cache - without <= S * (20.3 * n + (2 << 20)), (with_cache - without) / (n * S)


@pytest.mark.parametrize("then", ["nothing", "pull", "small push"])
def test_the_room_that_a_push_streams_through(capi, dev, monkeypatch, then):
    """12 B per key for keys and values by bin, 4 for the places of the keys that are left, not quite 1 for where each tile's bins start,
    an eighth to spare and the steps that arrays come in: 1.125 * 1.125 * 17 = 21.5 B per key. It goes back with the first request
    that does not stream."""
    import torch
    announce("streaming memory", then)
    n = 4_000_000
    keys = to_dev(unique_keys(np.random.default_rng(1), n), dev)
    vals, out = torch.zeros(n, device=dev), torch.zeros(n, device=dev)

    def filled():
        t = capi.Table(capi.MODE_SCALAR, initial_capacity=n)
        t.prof_enable()
        t.push(keys, vals)
        t.size()  # (it is known then that the keys of the next request fit)
        if then == "pull":
            t.pull(keys[:n // 64], out)
        elif then == "small push":
            t.push(keys[:1000], vals[:1000])
        t.sync()
        return t

    t = filled()
    assert t.prof_read(capi.KERNEL_REHASH)[0] == 3  # (it streams: nobody asked for it)
    t.close()
    with_room = held_by(capi, filled)
    monkeypatch.setenv("PSKV_STREAM", "0")
    without = held_by(capi, filled)
    assert with_room - without <= (21.5 * n if then == "nothing" else 0) + (2 << 20), (with_room - without) / n
