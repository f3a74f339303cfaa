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
