"""Device arrays and table state that one table leaves and the next one takes over."""
import os
import subprocess
import sys
import threading

import numpy as np
import pytest

from helpers import assert_bits_equal, to_dev, unique_keys
from conftest import REPO, announce

pytestmark = pytest.mark.gpu


def _fill_and_check(capi, orc, dev, rng, mode, n, rounds):
    """Tables that come and go: each starts small, grows into arrays that others have left, and holds exactly
    what was pushed (a stale array would show as a key that nobody pushed, or as a wrong sum)."""
    import torch
    for _ in range(rounds):
        t = capi.Table(mode, initial_capacity=int(rng.integers(1, 2000)))
        o = orc.Store(mode)
        k = 3 if mode == capi.MODE_FIXED else 1
        for _ in range(3):
            keys = unique_keys(rng, n)
            lens = rng.integers(1, 9, n).astype(np.int32) if mode == capi.MODE_VARLEN else None
            vals = rng.standard_normal(int(lens.sum()) if lens is not None else n * k).astype(np.float32)
            t.push(to_dev(keys, dev), to_dev(vals, dev), None if lens is None else to_dev(lens, dev))
            o.push(keys, vals, lens)
        torch.cuda.synchronize()
        dk, dl, dv = t.dump()
        ok, ol, ov = o.dump()
        assert np.array_equal(dk, ok) and np.array_equal(dl, ol)
        assert_bits_equal(dv, ov)
        t.close()


@pytest.mark.parametrize("mode", [0, 1, 2])
@pytest.mark.parametrize("n", [1, 700, 40_000])
def test_tables_take_over_what_others_left(capi, orc, dev, mode, n):
    announce("pool", mode, n)
    _fill_and_check(capi, orc, dev, np.random.default_rng(n + mode), mode, n, 4)
    capi.device_trim()
    _fill_and_check(capi, orc, dev, np.random.default_rng(n + mode + 1), mode, n, 2)


def test_tables_of_several_threads(capi, orc, dev):
    announce("pool threads")
    failed = []

    def work(seed):
        try:
            _fill_and_check(capi, orc, dev, np.random.default_rng(seed), seed % 3, 5000 + 100 * seed, 4)
        except BaseException as e:  # noqa: B036 (reported by the main thread)
            failed.append((seed, repr(e)))

    threads = [threading.Thread(target=work, args=(s,)) for s in range(6)]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    assert not failed, failed


def test_an_array_another_stream_is_still_using(capi, orc, dev):
    """A growth leaves its old array while kernels that read it are queued; a table on another stream takes it
    over at once and must wait for them."""
    import torch
    announce("pool streams")
    rng = np.random.default_rng(5)
    for _ in range(6):
        a, b = capi.Table(capi.MODE_SCALAR, initial_capacity=400_000), None
        oa, ob = orc.Store(capi.MODE_SCALAR), orc.Store(capi.MODE_SCALAR)
        ka, va = unique_keys(rng, 900_000), rng.standard_normal(900_000).astype(np.float32)
        kb, vb = unique_keys(rng, 300_000), rng.standard_normal(300_000).astype(np.float32)
        dka, dva, dkb, dvb = (to_dev(x, dev) for x in (ka, va, kb, vb))
        torch.cuda.synchronize()
        a.push(dka[:400_000].contiguous(), dva[:400_000].contiguous())
        a.push(dka, dva)  # grows: the old array is released with the move still queued
        b = capi.Table(capi.MODE_SCALAR, initial_capacity=400_000)
        b.push(dkb, dvb)
        oa.push(ka[:400_000], va[:400_000])
        oa.push(ka, va)
        ob.push(kb, vb)
        for t, o in ((a, oa), (b, ob)):
            dk, _, dv = t.dump()
            ok, _, ov = o.dump()
            assert np.array_equal(dk, ok)
            assert_bits_equal(dv, ov)
            t.close()


def test_tables_of_several_threads_on_one_stream(capi, orc, dev):
    """Two threads drive tables of their own on ONE stream of the caller's while a third creates tables on streams of
    their own, which take over what the others give up: the end of a table, which waits for the shared stream, says
    nothing about arrays that the other thread gives up after that wait."""
    import torch
    announce("pool shared stream")
    shared = torch.cuda.Stream(device=dev)
    failed = []

    def work(seed, stream):
        try:
            rng = np.random.default_rng(seed)
            for _ in range(8):
                n = 60_000 + 1000 * seed
                t, o = capi.Table(capi.MODE_SCALAR, initial_capacity=2000, stream=stream), orc.Store(orc.MODE_SCALAR)
                keep = []
                for _ in range(3):
                    keys, vals = unique_keys(rng, n), rng.standard_normal(n).astype(np.float32)
                    keep.append((to_dev(keys, dev), to_dev(vals, dev)))
                    torch.cuda.current_stream().synchronize()
                    t.push(*keep[-1])
                    o.push(keys, vals)
                dk, _, dv = t.dump()
                ok, _, ov = o.dump()
                assert np.array_equal(dk, ok)
                assert_bits_equal(dv, ov)
                t.close()
        except BaseException as e:  # noqa: B036 (reported by the main thread)
            failed.append((seed, repr(e)))

    threads = [threading.Thread(target=work, args=(s, stream)) for s, stream in
               enumerate([shared.cuda_stream, shared.cuda_stream, 0])]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    assert not failed, failed


_GIVES_BACK = """
import importlib, sys, time
sys.path.insert(0, %r)
import numpy as np, torch
capi = importlib.import_module("ps-lite_amd").capi
kept = sys.argv[1] == "kept"
x, g = torch.zeros(1000, device="cuda"), torch.cuda.CUDAGraph()
free = lambda: torch.cuda.mem_get_info()[0]
def table():
    t = capi.Table(capi.MODE_SCALAR, initial_capacity=1 << 26)  # 2 GiB of slots
    keys = np.arange(1, 100_000, dtype=np.uint64)
    t.push(keys, np.ones(keys.size, np.float32))
    t.sync()
    return t
table().close()
capi.device_trim()
torch.cuda.synchronize()
before = free()
t = table()
assert free() <= before - (2 << 30), "a table of 2 GiB takes 2 GiB"
t.close()
left = before - free()
assert (left >= (2 << 30)) == kept, left
if kept:  # in the middle of somebody's capture, which must not notice
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        x += 1
        torch.cuda.synchronize()
        g.capture_begin()
        x += 1
        time.sleep(3)
        g.capture_end()
    torch.cuda.synchronize()
    for _ in range(3):
        g.replay()
        torch.cuda.synchronize()
    assert (x == 4).all(), x[:4]
assert before - free() < (64 << 20), before - free()
t = table()  # and again
t.close()
print("ok", flush=True)
"""


@pytest.mark.parametrize("how", ["kept", "not kept"])
def test_the_last_table_gives_the_memory_back(capi, dev, how):
    """What tables have left goes back to the system some time after the last one has gone, also while another thread
    captures a stream; with PSKV_NO_ASYNC_ALLOC in the environment nothing is kept to begin with. (In a process of
    its own, where no other table is.)"""
    announce("gives back", how)
    env = dict(os.environ)
    env.pop("PSKV_NO_ASYNC_ALLOC", None)
    if how != "kept":
        env["PSKV_NO_ASYNC_ALLOC"] = "1"
    out = subprocess.run([sys.executable, "-c", _GIVES_BACK % REPO, how], stdout=subprocess.PIPE, stderr=subprocess.STDOUT,
                         text=True, timeout=90, env=env)
    assert out.returncode == 0 and out.stdout.strip().endswith("ok"), out.stdout
