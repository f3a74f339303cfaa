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
         (64, 64 * 512), (64, 64 * 512 + 1), (500, 9), (4093, 4), (4096, 3),
         # and those of several workgroups: a part of one quad, whole parts, one row, as many keys as go this way, too many floats
         (4097, 3), (4097, 256), (4097, 257), (8192, 2), (8195, 5), (100_003, 7), (1 << 22, 1), (16_384, 256), (16_385, 256)]


@pytest.mark.parametrize("looks", [None, "0"])
@pytest.mark.parametrize("k,n", FIXED)
def test_fixed_in_one_launch(capi, orc, dev, monkeypatch, k, n, looks):
    """New keys, held ones and a mix, pushed, pulled and both in one; with `looks` 0 no workgroup of a push waits for the
    verdict: the last one moves the rows of all."""
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
@pytest.mark.parametrize("k,n", [(5, 1), (5, 700), (64, 64 * 512 - 1), (4100, 1), (4100, 255), (9001, 3)])
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


@pytest.mark.parametrize("looks", [None, "0"])
@pytest.mark.parametrize("k,n", [(1, 256 * 65), (5, 700), (64, 64 * 511), (300, 20)])
def test_a_new_key_twice_in_a_request_that_is_not_sorted(capi, orc, dev, monkeypatch, k, n, looks):
    """Next to each other in no workgroup's eyes, but both of them one workgroup's, which therefore notices when it makes the
    row: the push is refused as a whole, whoever has waited for the verdict. In front of it and behind it pushes of keys in
    any order, new ones among them."""
    import torch
    announce("fixed, not sorted", k, n, looks)
    if looks is not None:
        monkeypatch.setenv("PSKV_PUSH_LOOKS", looks)
    rng = np.random.default_rng(n)
    t, o = capi.Table(capi.MODE_FIXED, row_len=k, initial_capacity=4 * n), orc.Store(orc.MODE_FIXED, k)
    pool = rng.permutation(unique_keys(rng, 2 * n + 1))

    def push(keys, both=False):
        vals = rng.standard_normal(keys.size * k).astype(np.float32)
        if not both:
            t.push(to_dev(keys, dev), _shifted(vals, dev, 1))
            return o.push(keys, vals)
        out = torch.full((keys.size * k,), 7.0, device=dev)
        t.pushpull(to_dev(keys, dev), to_dev(vals, dev), out)
        t.sync()
        assert_bits_equal(out.cpu().numpy(), o.pushpull(keys, vals)[0])

    push(pool[:n])
    push(pool[n // 2:n // 2 + n], both=True)
    # (three keys into the request, or two: a workgroup has at least that many)
    twice = pool[:n - 2]
    twice = np.concatenate([pool[-1:], twice[:1], pool[-1:], twice[1:]])
    t.push(to_dev(twice, dev), to_dev(rng.standard_normal(twice.size * k).astype(np.float32), dev))
    with pytest.raises(capi.PskvError) as e:
        t.sync()
    assert e.value.code == capi.EINVAL
    o.pull(pool[-1:])  # (the row it made stays, as a zero row)
    assert_bits_equal(t.dump()[2], o.dump()[2])
    push(rng.permutation(pool)[:n])
    push(rng.permutation(pool)[:n], both=True)
    assert_bits_equal(t.dump()[2], o.dump()[2])


@pytest.mark.parametrize("k", [4097, 20_000])
def test_long_rows_in_any_order(capi, orc, dev, k):
    """Keys that are not sorted, the key that marks an empty slot among them, rows made by pulls, many requests (whose counter
    records come from the same launch); a push that repeats a key it does not stand next to is refused, a pull served."""
    announce("long rows", k)
    rng = np.random.default_rng(k)
    pool = np.append(unique_keys(rng, 40), np.uint64(2**64 - 1))
    t, o = capi.Table(capi.MODE_FIXED, row_len=k, initial_capacity=8), orc.Store(orc.MODE_FIXED, k)

    def pull(keys):
        out = _shifted(np.full(keys.size * k, 7, np.float32), dev, 0)
        t.pull(to_dev(keys, dev), out)
        t.sync()
        return out.cpu().numpy()

    for turn in range(12):
        some = rng.permutation(pool)[:rng.integers(1, 17)]
        vals = rng.standard_normal(some.size * k).astype(np.float32)
        t.push(to_dev(some, dev), to_dev(vals, dev))
        o.push(some, vals)
        some = rng.permutation(pool)[:9]
        assert_bits_equal(pull(some), o.pull(some)[0], "turn %d" % turn)
    twice = np.append(pool[:5], pool[2])[::-1].copy()
    o.pull(pool[:5])
    with pytest.raises(capi.PskvError) as e:
        t.push(to_dev(twice, dev), to_dev(np.ones(twice.size * k, np.float32), dev))
        t.sync()
    assert e.value.code == capi.EINVAL
    assert_bits_equal(pull(twice), o.pull(twice)[0])
    assert_bits_equal(t.dump()[2], o.dump()[2])
    assert t.size() == o.size()


def _lens(rng, n, kind):
    if kind == "quads":
        return rng.choice(np.array([8, 16, 32, 64], np.int32), n)
    return rng.integers(0, 70, n).astype(np.int32)  # (rows without floats among them)


def _pull_async(t, dev, keys, out, out_lens=None):
    """A pull that does not wait for the size of its response."""
    import torch
    d_keys = to_dev(keys, dev)
    torch.cuda.synchronize()
    t.pull_raw(d_keys.data_ptr(), keys.size, out.data_ptr(), out.numel(), None if out_lens is None else out_lens.data_ptr())
    t.sync()


VAR = [("any", 1), ("any", 511), ("quads", 512), ("any", 513), ("any", 40_000), ("quads", 256 * 512), ("any", 256 * 512 + 1)]


@pytest.mark.parametrize("looks", [None, "0"])
@pytest.mark.parametrize("kind,n", VAR)
def test_varlen_started_by_one_launch(capi, orc, dev, monkeypatch, kind, n, looks):
    """Other keys in every request (some held, some new, some that a pull does not find), and a pull right behind the push of
    its keys; with `looks` 0 every workgroup goes through the request itself."""
    import torch
    announce("varlen in one launch", kind, n, looks)
    if looks is not None:
        monkeypatch.setenv("PSKV_PUSH_LOOKS", looks)
    rng = np.random.default_rng(n)
    t, o = capi.Table(capi.MODE_VARLEN), orc.Store(orc.MODE_VARLEN)
    keys = unique_keys(rng, 2 * n + 2)
    length = _lens(rng, keys.size, kind)
    length[0] = 3
    for turn in range(3):
        at = np.sort(rng.choice(keys.size, n, replace=False))
        lens = length[at]
        vals = rng.standard_normal(int(lens.sum())).astype(np.float32)
        t.push(to_dev(keys[at], dev), _shifted(vals, dev, turn), lens=to_dev(lens, dev))
        o.push(keys[at], vals, lens)
        for again in (True, False):
            if not again:
                at = np.sort(rng.choice(keys.size, n, replace=False))
            want, want_lens = o.pull(keys[at])[:2]
            out = _shifted(np.full(int(length[at].sum()) + 5, 7, np.float32), dev, turn)
            out_lens = torch.full((n,), 7, dtype=torch.int32, device=dev)
            _pull_async(t, dev, keys[at], out, out_lens)
            assert np.array_equal(out_lens.cpu().numpy(), want_lens), (turn, again)
            assert_bits_equal(out.cpu().numpy()[:want.size], want, "turn %d again %d" % (turn, again))
            assert (out.cpu().numpy()[want.size:] == 7).all()
    assert_bits_equal(t.dump()[2], o.dump()[2])


@pytest.mark.parametrize("looks", [None, "0"])
@pytest.mark.parametrize("n", [2, 700, 20_000])
def test_refused_varlen_requests(capi, orc, dev, monkeypatch, n, looks):
    """A repeated key, a length that is negative or too long, lens that do not add up: nothing is created or changed. A length
    that differs from the stored one: no stored value changes, rows it created are zero. A response without room:
    nothing is written. The request behind each is served."""
    import torch
    announce("varlen refused", n, looks)
    if looks is not None:
        monkeypatch.setenv("PSKV_PUSH_LOOKS", looks)
    rng = np.random.default_rng(n)
    t, o = capi.Table(capi.MODE_VARLEN), orc.Store(orc.MODE_VARLEN)
    keys = unique_keys(rng, 2 * n)
    length = rng.integers(1, 40, keys.size).astype(np.int32)
    held = np.arange(0, 2 * n, 2)

    def push(at, lens=None, ks=None):
        lens = length[at] if lens is None else lens
        ks = keys[at] if ks is None else ks
        vals = rng.standard_normal(int(length[at].sum())).astype(np.float32)
        t.push(to_dev(ks, dev), to_dev(vals, dev), lens=to_dev(lens, dev))
        return ks, vals, lens

    o.push(*push(held))
    t.sync()
    for what in ("repeat", "negative", "long", "sum"):
        at = np.sort(rng.choice(2 * n, n, replace=False))
        lens, ks, code = length[at].copy(), keys[at].copy(), capi.EINVAL
        j = int(rng.integers(1, n))
        if what == "repeat":
            ks[j] = ks[j - 1]
        elif what == "negative":
            lens[j] = -1
        elif what == "long":
            lens[j] = 1 << 28
        else:
            lens[j] += 1
            code = capi.ESIZE_MISMATCH
        push(at, lens, ks)
        with pytest.raises(capi.PskvError) as e:
            t.sync()
        assert e.value.code == code, what
        assert t.size() == (o.size()[0], o.size()[1]), what
        o.push(*push(held))
        t.sync()
    # a held row comes with another length, a new one with it
    at = np.array([held[0], held[0] + 1])
    lens = np.array([length[held[0]] + 1, 6], np.int32)
    t.push(to_dev(keys[at], dev), to_dev(np.ones(int(lens.sum()), np.float32), dev), lens=to_dev(lens, dev))
    with pytest.raises(capi.PskvError) as e:
        t.sync()
    assert e.value.code == capi.ELEN_CHANGED
    o.push(keys[at[1:]], np.zeros(6, np.float32), lens[1:])
    want = o.pull(keys)[0]
    out = torch.full((want.size,), 7.0, device=dev)
    with pytest.raises(capi.PskvError) as e:
        _pull_async(t, dev, keys, out[:want.size - 1])
    assert e.value.code == capi.ESIZE_MISMATCH and bool((out == 7).all())
    _pull_async(t, dev, keys, out)
    assert_bits_equal(out.cpu().numpy(), want)
    assert_bits_equal(t.dump()[2], o.dump()[2])


@pytest.mark.parametrize("S", [1, 5])
def test_varlen_requests_that_repeat(capi, orc, dev, S):
    """The same rows often enough to be expected, others of the same number, ragged ones and the first again: each starts with
    one launch or with two, as the rule has it, and finds what the others have left."""
    import torch
    announce("varlen repeats", S)
    rng = np.random.default_rng(S)
    n = 5000
    group, stores = capi.Group(S, capi.MODE_VARLEN), [orc.Store(orc.MODE_VARLEN) for _ in range(S)]
    begin, end = orc.server_ranges(S)
    pool = np.sort(rng.permutation(unique_keys(rng, 3 * n, S)))
    sets = []
    for i in range(3):
        lens = (rng.integers(1, 33, n) * (1 if i == 2 else 4)).astype(np.int32)
        sets.append((pool[i::3], lens))
    for which in (0, 0, 0, 0, 1, 0, 2, 2, 2, 1, 2, 0, 0, 0):
        keys, lens = sets[which]
        total = int(lens.sum())
        pos, val_pos, _ = orc.slice_keys(keys, begin, end, lens, total)
        vals = rng.standard_normal(total).astype(np.float32)
        out = torch.full((total,), 7.0, device=dev)
        out_lens = torch.zeros(n, dtype=torch.int32, device=dev)
        d_keys, d_lens = to_dev(keys, dev), to_dev(lens, dev)
        group.push(d_keys, pos, to_dev(vals, dev), val_pos, lens=d_lens)
        group.pull(d_keys, pos, out, out_pos=val_pos, out_lens=out_lens)
        group.sync()
        want = []
        for s in range(S):
            a, b, va, vb = int(pos[s]), int(pos[s + 1]), int(val_pos[s]), int(val_pos[s + 1])
            stores[s].push(keys[a:b], vals[va:vb], lens[a:b])
            want.append(stores[s].pull(keys[a:b])[0])
        assert_bits_equal(out.cpu().numpy(), np.concatenate(want))
        assert np.array_equal(out_lens.cpu().numpy(), lens)
    group.close()


@pytest.mark.parametrize("kind", ["push", "pull", "both"])
@pytest.mark.parametrize("n", [1, 4096, 4097, 2_500_001])
def test_cached_values_written_back_by_the_request_that_differs(capi, orc, dev, monkeypatch, kind, n):
    """The same keys often enough for the host to expect them, then others of the same number (2.5M: more workgroups than
    the GPU holds): the cached values reach the slots before the first of the others is looked up."""
    import torch
    announce("write back", kind, n)
    monkeypatch.setenv("PSKV_SCALAR_CACHE_MIN_KEYS", "1")
    rng = np.random.default_rng(n)
    t, o = capi.Table(capi.MODE_SCALAR), orc.Store(orc.MODE_SCALAR)
    pool = unique_keys(rng, n + n // 2 + 1)
    same = np.sort(rng.choice(pool, n, replace=False))
    if n > 1:
        same[-1] = 2**64 - 1  # (the key that lives in the side slot)
    other = np.sort(rng.choice(pool, n, replace=False))
    other[-1] = max(other[-1], same[-1])
    vals = [rng.standard_normal(n).astype(np.float32) for _ in range(2)]

    def request(keys, v):
        out = torch.zeros(n, device=dev)
        torch.cuda.synchronize()
        want = None
        if kind == "both":
            t.pushpull(to_dev(keys, dev), to_dev(v, dev), out)
            want = o.pushpull(keys, v)[0]
        else:
            if kind == "push" or keys is same:
                t.push(to_dev(keys, dev), to_dev(v, dev))
                o.push(keys, v)
            if kind == "pull":
                t.pull(to_dev(keys, dev), out)
                want = o.pull(keys)[0]
        t.sync()
        if want is not None:
            assert_bits_equal(out.cpu().numpy(), want)

    for _ in range(2):
        for turn in range(4):
            request(same, vals[turn & 1])
        request(other, vals[0])
    assert_bits_equal(t.dump()[2], o.dump()[2])


@pytest.mark.parametrize("kind", ["push", "pull", "both"])
@pytest.mark.parametrize("n", [2, 5, 1023, 1025, 70_001])
def test_cached_values_of_keys_that_stay_where_they_are(capi, orc, dev, monkeypatch, kind, n):
    """The slots lag behind the cache, and the request that differs names most keys at their cached positions, one or a few at
    others, or one of them twice, with the cached position in front or behind."""
    import torch
    announce("write back, some stay", kind, n)
    monkeypatch.setenv("PSKV_SCALAR_CACHE_MIN_KEYS", "1")
    rng = np.random.default_rng(n)
    pool = unique_keys(rng, 2 * n)
    pool[-1] = 2**64 - 1
    base = pool[::2].copy()
    base[-1] = pool[-1]
    others = []
    for j in sorted({0, n // 2, n - 1}):
        other = base.copy()
        other[j] = pool[2 * j] + np.uint64(1) if 2 * j + 1 < 2 * n and pool[2 * j] + np.uint64(1) < pool[2 * j + 1] else other[j]
        others.append(other)
        if j + 1 < n:
            for a, b in ((j, j + 1), (j + 1, j)):  # the key at b stands at both
                other = base.copy()
                other[a] = base[b]
                others.append(other)
            other = base.copy()  # everything behind j moves by one
            other[j + 1:] = base[j:-1]
            other[j] = base[j - 1] if j else base[0]
            others.append(np.sort(other))
    for turn, other in enumerate(others):
        t, o = capi.Table(capi.MODE_SCALAR), orc.Store(orc.MODE_SCALAR)
        for keys in (base, base, base, base, other):
            vals = rng.standard_normal(n).astype(np.float32)
            out = torch.zeros(n, device=dev)
            torch.cuda.synchronize()
            if kind == "both":
                t.pushpull(to_dev(keys, dev), to_dev(vals, dev), out)
                want = o.handle(True, True, keys, vals, out_cap=n)[1]
            elif kind == "push" or keys is base:
                t.push(to_dev(keys, dev), to_dev(vals, dev))
                o.push(keys, vals)
                continue
            else:
                t.pull(to_dev(keys, dev), out)
                want = o.pull(keys)[0]
            t.sync()
            assert_bits_equal(out.cpu().numpy(), want, "turn %d" % turn)
        t.sync()
        assert_bits_equal(t.dump()[2], o.dump()[2], "turn %d" % turn)


@pytest.mark.parametrize("S", [1, 3, 16, 31])
@pytest.mark.parametrize("n", [1, 2047, 2048, 2049, 30_001, 128 * 2048 + 1, 512 * 2048, 512 * 2048 + 1])
def test_slices_with_lens_of_few_keys(capi, orc, dev, n, S):
    """Boundaries and sums of lens by one scan (up to 1,048,576 keys): the edges of a workgroup's stretch, boundaries on a key,
    between keys, in front of all and behind all, several in one stretch; called twice, from either kind of memory."""
    announce("few slices", n, S)
    rng = np.random.default_rng(n * 31 + S)
    begin, end = orc.server_ranges(S)
    sets = [unique_keys(rng, n, S), np.arange(n, dtype=np.uint64) + begin[S // 2]]
    if S > 1:
        near = np.concatenate([np.arange(-3, 4).astype(np.int64).astype(np.uint64) + e for e in end[:-1]])
        sets.append(np.unique(np.concatenate([near, unique_keys(rng, max(1, n - near.size), S)])))
    for keys in sets:
        lens = rng.integers(0, 1000, keys.size).astype(np.int32)
        want = orc.slice_keys(keys, begin, end, lens, int(lens.sum()))
        for _ in range(2):
            got = capi.slice_keys(to_dev(keys, dev), begin, end, lens=to_dev(lens, dev), nvals=int(lens.sum()))
            for a, b in zip(got, want):
                assert np.array_equal(np.asarray(a), np.asarray(b))


@pytest.mark.parametrize("S", [1, 16, 31, 32])
@pytest.mark.parametrize("n", [1, 64, 65, 4096, 4097, 300_000])
def test_slices_without_lens(capi, orc, dev, n, S):
    """A wavefront for each boundary, up to 32 of them: where its search takes a round more, keys on the boundaries and beside
    them, and no key in most of the ranges."""
    announce("slices without lens", n, S)
    rng = np.random.default_rng(n * 37 + S)
    begin, end = orc.server_ranges(S)
    near = np.concatenate([np.arange(-3, 4).astype(np.int64).astype(np.uint64) + e for e in end[:-1]] or [end[:0]])
    for keys in (unique_keys(rng, n, S), np.arange(n, dtype=np.uint64) + begin[S // 2],
                 np.unique(np.concatenate([near, unique_keys(rng, n, S)]))):
        want = orc.slice_keys(keys, begin, end, None, 3 * keys.size)
        for _ in range(2):
            for a, b in zip(capi.slice_keys(to_dev(keys, dev), begin, end, nvals=3 * keys.size), want):
                assert np.array_equal(np.asarray(a), np.asarray(b))


@pytest.mark.parametrize("n", [2049, 70_000])
def test_slices_with_lens_of_any_size_and_order(capi, orc, dev, n):
    """Ranges without keys that end where they begin, lens whose sums need all the bits of a part's word and negative ones;
    and keys that are not sorted, which give no slices worth having but an answer, and leave the next call alone, which is one
    of the same keys in order. Refused is what the oracle refuses."""
    announce("few slices, lens of any size", n)
    rng = np.random.default_rng(n)
    keys = unique_keys(rng, n, 4)
    cut = [0, int(keys[n // 3]), int(keys[n // 3]), int(keys[2 * n // 3]) + 1, 2**64 - 1]
    begin, end = np.array(cut[:-1], np.uint64), np.array(cut[1:], np.uint64)
    d_keys, d_shuffled = to_dev(keys, dev), to_dev(rng.permutation(keys), dev)

    def sliced(slice_keys, error, *args, **more):
        try:
            return slice_keys(*args, **more)
        except error as e:
            return e.code

    largest, some = np.full(n, 2**31 - 1, np.int32), rng.integers(-300, 1000, n).astype(np.int32)
    for lens, short in ((largest, 0), (largest, 1), (some, 0), (rng.integers(-2**31, 2**31, n).astype(np.int32) | 1, 0)):
        nvals, d_lens = max(0, int(lens.astype(np.int64).sum()) - short), to_dev(lens, dev)
        want = sliced(orc.slice_keys, orc.OracleError, keys, begin, end, lens, nvals)
        refused = isinstance(want, int)
        assert refused or not short
        for k in (d_keys, d_shuffled, d_keys):
            got = sliced(capi.slice_keys, capi.PskvError, k, begin, end, lens=d_lens, nvals=nvals)
            if k is d_shuffled:
                continue
            if refused:
                assert got == want
                continue
            assert not isinstance(got, int), got
            for a, b in zip(got, want):
                assert np.array_equal(np.asarray(a), np.asarray(b))


@pytest.mark.parametrize("mode", ["scalar", "fixed", "varlen"])
def test_tables_of_a_group_grow_and_are_counted_together(capi, orc, dev, mode):
    """Eighteen tables of different sizes (two launches' worth) that one request makes grow, by two, four and eight and by
    more (which fills and scatters), or not at all; their sizes in one call."""
    announce("group growth", mode)
    rng = np.random.default_rng(7)
    S = 18
    code = {"scalar": capi.MODE_SCALAR, "fixed": capi.MODE_FIXED, "varlen": capi.MODE_VARLEN}[mode]
    k = 3 if mode == "fixed" else 0
    tables = []
    for s in range(S):
        stream = capi.load().pskv_table_stream(tables[0]._h) if tables else None
        tables.append(capi.Table(code, initial_capacity=1 << (4 + s), row_len=k, stream=stream))
    group = object.__new__(capi.Group)
    group.__dict__.update(tables=tables, S=S, mode=code, _lib=capi.load())
    import ctypes
    group._arr = (ctypes.c_void_p * S)(*[t._h for t in tables])
    group._at = ctypes.addressof(group._arr)
    stores = [orc.Store(code, k) for _ in range(S)]
    begin, end = orc.server_ranges(S)
    for turn, n in enumerate((2_000, 40_000, 60_000, 300_000)):
        keys = unique_keys(rng, n, S)
        lens = (keys % np.uint64(7)).astype(np.int32) if mode == "varlen" else None
        nvals = int(lens.sum()) if mode == "varlen" else n * max(k, 1)
        vals = rng.standard_normal(nvals).astype(np.float32)
        pos, val_pos, _ = orc.slice_keys(keys, begin, end, lens, nvals)
        group.push(to_dev(keys, dev), pos, to_dev(vals, dev), val_pos, lens=None if lens is None else to_dev(lens, dev))
        for s in range(S):
            a, b, va, vb = int(pos[s]), int(pos[s + 1]), int(val_pos[s]), int(val_pos[s + 1])
            stores[s].push(keys[a:b], vals[va:vb], None if lens is None else lens[a:b])
        sizes = [o.size() for o in stores]
        assert group.size() == (sum(x for x, _ in sizes), sum(y for _, y in sizes))
        assert [t.size() for t in tables] == [tuple(x) for x in sizes]
    for t, o in zip(tables, stores):
        got, want = t.dump(), o.dump()
        assert np.array_equal(got[0], want[0])
        assert_bits_equal(got[2], want[2])
    group.close()
