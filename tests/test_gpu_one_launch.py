"""Requests of the row modes that are served by one launch (csrc/one_launch.h): the sizes where a workgroup's share ends
and where the request goes back to a lookup and a row kernel, refused requests, and workgroups that do not wait for
each other. Against the CPU oracle, bit for bit."""
import numpy as np
import pytest

from conftest import announce
from helpers import assert_bits_equal, to_dev, unique_keys

pytestmark = pytest.mark.gpu


def _share(k):
    return min(256, 1024 // ((k + 3) // 4))


def _shifted(a, dev, shift):
    import torch
    room = torch.zeros(a.size + shift, dtype=torch.float32, device=dev)
    room[shift:] = to_dev(a, dev)
    return room[shift:]


# floats per row, keys: one workgroup's share and a key more or less, the last share of a push and one beyond, rows
# that are a workgroup's all, and longer ones
FIXED = [(1, 1), (1, 256), (1, 257), (3, 511), (4, 513), (15, 256 * 512), (16, 256 * 512 + 1), (64, 63), (64, 65),
         (64, 64 * 512), (64, 64 * 512 + 1), (500, 9), (4093, 4), (4096, 3), (4097, 3)]


@pytest.mark.parametrize("looks", [None, "0"])
@pytest.mark.parametrize("k,n", FIXED)
def test_fixed_in_one_launch(capi, orc, dev, monkeypatch, k, n, looks):
    """New keys, held ones and a mix, pushed, pulled and both in one; with `looks` 0 no workgroup of a push waits for the
    verdict: every one reads all keys."""
    import torch
    announce("fixed in one launch", k, n, looks)
    if looks is not None:
        monkeypatch.setenv("PSKV_PUSH_LOOKS", looks)
    rng = np.random.default_rng(k * 7919 + n)
    t, o = capi.Table(capi.MODE_FIXED, row_len=k), orc.Store(orc.MODE_FIXED, k)
    keys = unique_keys(rng, 2 * n + 2)
    for turn in range(3):
        some = np.sort(rng.choice(keys, n, replace=False))
        vals = rng.standard_normal(n * k).astype(np.float32)
        out = _shifted(np.full(n * k, 7, np.float32), dev, turn)
        if turn == 2:
            t.pushpull(to_dev(some, dev), _shifted(vals, dev, 1), out)
            want = o.pushpull(some, vals)[0]
        else:
            t.push(to_dev(some, dev), _shifted(vals, dev, turn))
            o.push(some, vals)
            some = np.sort(rng.choice(keys, n, replace=False))
            t.pull(to_dev(some, dev), out)
            want = o.pull(some)[0]
        torch.cuda.synchronize()
        assert_bits_equal(out.cpu().numpy(), want, "turn %d" % turn)
    assert_bits_equal(t.dump()[2], o.dump()[2])


@pytest.mark.parametrize("looks", [None, "0"])
@pytest.mark.parametrize("k,n", [(5, 1), (5, 700), (64, 64 * 512 - 1)])
def test_a_push_that_repeats_a_key_changes_nothing(capi, orc, dev, monkeypatch, k, n, looks):
    """The repeat sits in the first, in the last or in any workgroup's share: no stored value changes, created rows are
    zero, the next sync says EINVAL, and the push behind it is served."""
    announce("fixed repeat", k, n, looks)
    if looks is not None:
        monkeypatch.setenv("PSKV_PUSH_LOOKS", looks)
    rng = np.random.default_rng(n)
    pool = unique_keys(rng, 2 * n)
    for at in sorted({0, n - 1, n // 2}):
        t, o = capi.Table(capi.MODE_FIXED, row_len=k), orc.Store(orc.MODE_FIXED, k)
        vals = rng.standard_normal(n * k).astype(np.float32)
        held = np.sort(rng.choice(pool, n, replace=False))
        t.push(to_dev(held, dev), to_dev(vals, dev))
        o.push(held, vals)
        bad = np.sort(rng.choice(pool, n, replace=False))
        bad = np.sort(np.append(bad, bad[at]))
        t.push(to_dev(bad, dev), to_dev(rng.standard_normal(bad.size * k).astype(np.float32), dev))
        with pytest.raises(capi.PskvError) as e:
            t.sync()
        assert e.value.code == capi.EINVAL
        o.pull(np.unique(bad))  # (the rows it created stay, as zero rows)
        some = np.unique(bad)
        more = rng.standard_normal(some.size * k).astype(np.float32)
        t.push(to_dev(some, dev), to_dev(more, dev))
        o.push(some, more)
        assert_bits_equal(t.dump()[2], o.dump()[2], "repeat at %d" % at)
        t.close()
