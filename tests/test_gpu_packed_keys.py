"""Requests of many keys that repeat the cached one, whose keys a SCALAR table then keeps packed, 48 bits each next to
their neighbour: the same keys, keys that differ in single places, neighbours too far apart. Against the CPU oracle, bit for bit."""
import numpy as np
import pytest

from conftest import announce
from helpers import assert_bits_equal, to_dev
from test_gpu_store import _check_dump

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def packs_a_million(monkeypatch):
    monkeypatch.setenv("PSKV_PACK_MIN_KEYS", str(1 << 20))


@pytest.mark.parametrize("n,skip", [(1 << 20, 0), ((1 << 20) + 1, 1), ((1 << 20) + 255, 0), ((1 << 20) + 1023, 0)])
@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("ahead", [False, True])
def test_repeats_and_single_differences(capi, orc, dev, n, skip, wide, ahead):
    """`ahead`: requests that the host queues without waiting, so that it chooses their kernels before it is told of the ones before."""
    import torch
    announce("packed keys", n, skip, wide, ahead)
    rng = np.random.default_rng(n)
    keys = np.cumsum(rng.integers(2, 1 << 30, n, dtype=np.uint64))
    if wide:
        keys[n // 3:] += np.uint64(1 << 48)
    t, o = capi.Table(capi.MODE_SCALAR, initial_capacity=2 * n), orc.Store(orc.MODE_SCALAR)

    answers = []

    def check():
        t.sync()
        for out, want in answers:
            assert_bits_equal(out.cpu().numpy(), want)
        answers.clear()

    def request(ks):
        vals = rng.standard_normal(n).astype(np.float32)
        room = to_dev(np.concatenate([ks[:skip], ks]), dev)[skip:]
        out = torch.empty(n, dtype=torch.float32, device=dev)
        t.push(room, to_dev(vals, dev))
        t.pull(room, out)
        o.push(ks, vals)
        answers.append((out, o.pull(ks)[0]))
        if not ahead:
            check()

    # (a record, a comparison that finds the keys equal, one that packs them, and one of the packed keys)
    for places in ([], [], [], [], [], [0], [255, 256], [n - 1], [n // 2 + 3]):
        other = keys.copy()
        other[places] += np.uint64(1)  # (keys are two apart at least)
        request(other)
        if places:
            for _ in range(5):  # (comparisons that failed leave out a few)
                request(keys)
    check()
    _check_dump(t, o, "packed")
