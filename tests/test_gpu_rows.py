"""Rows that do not fit 16-byte quads: every remainder of the row length, quads that hold two rows or more,
buffers on any float, pieces of a host-resident request that end inside a quad. Against the CPU oracle, bit
for bit."""
import numpy as np
import pytest

from helpers import assert_bits_equal, to_dev, unique_keys
from conftest import announce

pytestmark = pytest.mark.gpu


def _off_by(a, dev, shift):
    """The values on the device, `shift` floats behind a 16-byte boundary."""
    import torch
    room = torch.zeros(a.size + shift, dtype=torch.float32, device=dev)
    room[shift:] = to_dev(a, dev)
    return room[shift:]


@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("k", [1, 2, 3, 4, 5, 7, 31, 64, 66, 255, 1021, 1022, 1023, 1024, 1025, 1030])
def test_fixed_rows_of_any_length(capi, orc, dev, k, shift):
    announce("fixed rows", k, shift)
    import torch
    rng = np.random.default_rng(k)
    n = max(3, 60_000 // k) | 1
    t, o = capi.Table(capi.MODE_FIXED, row_len=k), orc.Store(orc.MODE_FIXED, k)
    keys = unique_keys(rng, 2 * n)
    for turn in range(4):
        some = np.sort(rng.choice(keys, n, replace=False))
        vals = rng.standard_normal(n * k).astype(np.float32)
        t.push(to_dev(some, dev), _off_by(vals, dev, shift))
        o.push(some, vals)
        if turn == 2:  # keys that the store has not seen are answered, and kept, as zero rows
            some = keys
        out = _off_by(np.full(some.size * k, 7, np.float32), dev, 3 * shift)
        t.pull(to_dev(some, dev), out)
        torch.cuda.synchronize()
        assert_bits_equal(out.cpu().numpy(), o.pull(some)[0], "k = %d" % k)
    assert_bits_equal(t.dump()[2], o.dump()[2])


LENGTHS = {"any": lambda rng, n: rng.integers(0, 101, n), "short": lambda rng, n: rng.integers(0, 4, n),
           "ones": lambda rng, n: np.ones(n, np.int64), "mixed": lambda rng, n: rng.choice([0, 1, 2, 3, 5, 258, 1025], n),
           "tail": lambda rng, n: np.where(np.arange(n) == n - 1, 3, 8)}


@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("n", [1, 130, 5000])
@pytest.mark.parametrize("which", sorted(LENGTHS))
def test_varlen_rows_of_any_length(capi, orc, dev, which, n, shift):
    announce("varlen rows", which, n, shift)
    import torch
    rng = np.random.default_rng(n)
    t, o = capi.Table(capi.MODE_VARLEN), orc.Store(orc.MODE_VARLEN)
    keys = unique_keys(rng, 2 * n)
    all_lens = LENGTHS[which](rng, 2 * n).astype(np.int32)
    for turn in range(4):
        pick = np.sort(rng.choice(2 * n, n, replace=False)) if turn != 1 else pick  # (turn 1: the same keys again)
        some, lens = keys[pick], all_lens[pick]
        vals = rng.standard_normal(int(lens.sum())).astype(np.float32)
        t.push(to_dev(some, dev), _off_by(vals, dev, shift), to_dev(lens, dev))
        o.push(some, vals, lens)
        if turn == 2:
            some = keys  # some of them absent: answered with length 0
        want, want_lens = o.pull(some)
        out = _off_by(np.full(want.size + 5, 7, np.float32), dev, 3 * shift)
        out_lens = torch.empty(some.size, dtype=torch.int32, device=dev)
        got = t.pull(to_dev(some, dev), out, out_lens)
        torch.cuda.synchronize()
        assert got == want.size and np.array_equal(out_lens.cpu().numpy(), want_lens)
        host = out.cpu().numpy()
        assert_bits_equal(host[:got], want, which)
        assert (host[got:] == 7).all()


@pytest.mark.parametrize("n,k", [(3, 1_500_001), (5, 1_048_579), (40_001, 131)])
def test_host_resident_rows_in_pieces(capi, orc, dev, n, k):
    """Several pieces of the ring per request; their edges fall inside rows and inside quads."""
    announce("host pieces", n, k)
    rng = np.random.default_rng(k)
    t, o = capi.Table(capi.MODE_FIXED, row_len=k), orc.Store(orc.MODE_FIXED, k)
    keys = unique_keys(rng, n)
    for _ in range(2):
        vals = rng.random(n * k, dtype=np.float32) - np.float32(0.5)
        t.push(keys, vals)
        o.push(keys, vals)
        out = np.zeros(n * k, np.float32)
        t.pull(keys, out)
        assert_bits_equal(out, o.pull(keys)[0])


@pytest.mark.parametrize("mode", ["fixed", "varlen"])
@pytest.mark.parametrize("n", [1, 255, 257, 1023, 1025, 140_001, (1 << 20) + 3])
def test_requests_that_partly_repeat(capi, orc, dev, mode, n):
    """The same keys several times (the kernels then expect them), then a few or all of them others, and a
    shorter request in between: references left at a position are used exactly where their key still is."""
    announce("partly repeat", mode, n)
    import torch
    rng = np.random.default_rng(n)
    m, k = (capi.MODE_FIXED, 5) if mode == "fixed" else (capi.MODE_VARLEN, 0)
    t, o = capi.Table(m, row_len=k), orc.Store(m, k)
    keys = unique_keys(rng, n + n // 2 + 2)
    all_lens = rng.integers(1, 6, keys.size).astype(np.int32)
    base = np.sort(rng.choice(keys.size, n, replace=False))
    near = base.copy()
    spare = np.setdiff1d(np.arange(keys.size), base)
    near[rng.integers(0, n, 3)] = spare[0]
    near = np.unique(near)
    other = np.sort(rng.choice(keys.size, n, replace=False))
    for pick in (base, base, base, near, base, base[: n // 2 + 1], base, base, other, base):
        some, lens = keys[pick], all_lens[pick]
        vals = rng.standard_normal(int(lens.sum()) if mode == "varlen" else some.size * k).astype(np.float32)
        args = (to_dev(lens, dev),) if mode == "varlen" else ()
        t.push(to_dev(some, dev), to_dev(vals, dev), *args)
        o.push(some, vals, lens if mode == "varlen" else None)
        want, want_lens = o.pull(some)
        out = torch.empty(want.size, dtype=torch.float32, device=dev)
        if mode == "varlen":
            out_lens = torch.empty(some.size, dtype=torch.int32, device=dev)
            t.pull(to_dev(some, dev), out, out_lens)
            torch.cuda.synchronize()
            assert np.array_equal(out_lens.cpu().numpy(), want_lens)
        else:
            t.pull(to_dev(some, dev), out)
            torch.cuda.synchronize()
        assert_bits_equal(out.cpu().numpy(), want)
    assert_bits_equal(t.dump()[2], o.dump()[2])


# mean lengths around the ones that lanes per row go by, a row sixteen times as long as the others, rows of nothing
RAGGED = {"seven": lambda rng, n: rng.integers(5, 10, n), "nine": lambda rng, n: rng.integers(1, 18, n),
          "with a long one": lambda rng, n: np.where(np.arange(n) == n // 2, 4099, rng.integers(0, 40, n)),
          "up to the longest": lambda rng, n: np.where(np.arange(n) % 500 == 3, 290, rng.integers(0, 37, n)),
          "hundreds": lambda rng, n: rng.integers(90, 165, n),
          # (three turns of 4, 8 and 16 lanes: means of 6, 12 and 24 quads; rows of two such rounds among them)
          "six quads": lambda rng, n: rng.integers(1, 47, n), "twelve quads": lambda rng, n: np.where(np.arange(n) % 97 == 5, 385, rng.integers(1, 88, n)),
          "twenty-four quads": lambda rng, n: rng.integers(1, 188, n)}


@pytest.mark.parametrize("n,S", [(700, 1), (30_001, 2), (140_003, 1)])
@pytest.mark.parametrize("which", sorted(RAGGED))
def test_ragged_pushes_row_by_row(capi, orc, dev, which, n, S):
    """Pushes behind one that has told the host of ragged rows: held and new rows, the same again, one that is refused."""
    announce("row by row", which, n, S)
    rng = np.random.default_rng(n)
    group, stores = capi.Group(S, capi.MODE_VARLEN), [orc.Store(orc.MODE_VARLEN) for _ in range(S)]
    begin, end = capi.server_ranges(S)
    keys = unique_keys(rng, 2 * n, S)
    all_lens = RAGGED[which](rng, 2 * n).astype(np.int32)
    all_lens[::13] += 1  # ragged in any case
    for turn in range(5):
        pick = np.sort(rng.choice(2 * n, n, replace=False)) if turn not in (2, 4) else pick
        some, lens = keys[pick], all_lens[pick].copy()
        if turn == 4:
            lens[n // 3] += 4  # not the stored length: nothing of this table's share is applied
        vals = rng.standard_normal(int(lens.sum())).astype(np.float32)
        dk, dl = to_dev(some, dev), to_dev(lens, dev)
        pos, val_pos, _ = capi.slice_keys(dk, begin, end, lens=dl, nvals=vals.size)
        group.push(dk, pos, _off_by(vals, dev, turn % 3), val_pos, lens=dl)
        if turn == 4:
            with pytest.raises(capi.PskvError):
                group.sync()
        else:
            group.sync()
        for s in range(S):
            part, floats = slice(int(pos[s]), int(pos[s + 1])), slice(int(val_pos[s]), int(val_pos[s + 1]))
            if turn < 4 or not part.start <= n // 3 < part.stop:
                stores[s].push(some[part], vals[floats], lens[part])
    for s in range(S):
        want_keys, want_lens, want = stores[s].dump()
        got_keys, got_lens, got = group.tables[s].dump()
        assert np.array_equal(got_keys, want_keys) and np.array_equal(got_lens, want_lens)
        assert_bits_equal(got, want, "%s table %d" % (which, s))


@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("k,n", [(1024, 2100), (1025, 8300), (1027, 2100), (4098, 1100), (1_500_001, 3)])
def test_rows_of_a_workgroup_or_more(capi, orc, dev, k, n, shift):
    """Requests beyond what one launch serves: new rows and held ones, pushed, pulled and both, and a push that is refused."""
    announce("wide rows", k, n, shift)
    import torch
    rng = np.random.default_rng(k)
    t, o = capi.Table(capi.MODE_FIXED, row_len=k), orc.Store(orc.MODE_FIXED, k)
    keys = unique_keys(rng, n + n // 2)
    for turn in range(4):
        some = np.sort(rng.choice(keys, n, replace=False))
        vals = rng.standard_normal(n * k).astype(np.float32)
        out = _off_by(np.full(n * k, 7, np.float32), dev, 3 * shift)
        if turn == 1:
            t.pull(to_dev(some, dev), out)
            want = o.pull(some)[0]
        elif turn == 2:
            t.pushpull(to_dev(some, dev), _off_by(vals, dev, shift), out)
            want = o.pushpull(some, vals)[0]
        else:
            if turn == 3:
                some[n // 2] = some[n // 2 - 1]
            t.push(to_dev(some, dev), _off_by(vals, dev, shift))
            if turn == 3:
                with pytest.raises(capi.PskvError):
                    t.sync()
                break
            o.push(some, vals)
            continue
        t.sync()
        assert_bits_equal(out.cpu().numpy(), want, "k = %d" % k)
    o.pull(some)  # (the rows that a refused push has made stay, as zero rows)
    for mine, theirs in zip(t.dump(), o.dump()):
        assert np.array_equal(mine, theirs) if mine.dtype != np.float32 else assert_bits_equal(mine, theirs) is None


@pytest.mark.parametrize("k", [1024, 1030])
def test_recorded_rows_of_a_workgroup_or_more(capi, orc, dev, k):
    announce("wide rows, recorded", k)
    import torch
    rng = np.random.default_rng(k)
    n, S = 41, 2
    keys, vals = unique_keys(rng, n, S), rng.standard_normal(n * k).astype(np.float32)
    group, o = capi.Group(S, capi.MODE_FIXED, row_len=k), orc.Store(orc.MODE_FIXED, k)
    dk, dv, out = to_dev(keys, dev), to_dev(vals, dev), torch.zeros(n * k, device=dev)
    pos, val_pos, _ = capi.slice_keys(dk, *capi.server_ranges(S), nvals=n * k)
    rec = group.record(capi.REPLAY_PUSH | capi.REPLAY_PULL, dk, pos, dv, val_pos, out=out)
    o.push(keys, vals)
    for _ in range(3):
        rec.run()
        group.sync()
        o.push(keys, vals)
        assert_bits_equal(out.cpu().numpy(), o.pull(keys)[0])


@pytest.mark.parametrize("mode,n", [("ragged", 3_000), ("ragged", 60_000), ("wide", 40)])
def test_rows_of_values_that_are_no_numbers(capi, orc, dev, mode, n):
    """Infinities, and NaNs that meet numbers only (their payload stays then, whichever way round they are added), through the row kernels
    that go by the rows and the wide ones; the ends of ragged rows, whose last quad is written whole, among them."""
    announce("rows of NaNs", mode, n)
    import torch
    rng = np.random.default_rng(n)
    keys = unique_keys(rng, n)
    ragged, k = mode == "ragged", 1030
    lens = rng.integers(1, 90, n).astype(np.int32) if ragged else None
    total = int(lens.sum()) if ragged else n * k
    t = capi.Table(capi.MODE_VARLEN) if ragged else capi.Table(capi.MODE_FIXED, row_len=k)
    o = orc.Store(orc.MODE_VARLEN, 0) if ragged else orc.Store(orc.MODE_FIXED, k)
    at = np.arange(total)
    for turn in range(5):
        vals = rng.standard_normal(total).astype(np.float32)
        vals[at % 11 == turn] = (np.uint32(0x7FC00000) + (at[at % 11 == turn] & 0xFFFF).astype(np.uint32)).view(np.float32)
        vals[at % 11 == 5] = np.inf
        vals[at % 11 == 6] = -np.inf
        vals[at % 11 == 7 + turn % 2] = -0.0
        t.push(to_dev(keys, dev), _off_by(vals, dev, turn % 3), None if lens is None else to_dev(lens, dev))
        o.push(keys, vals, lens)
        t.sync()
    out, out_lens = torch.empty(total, device=dev), torch.empty(n, dtype=torch.int32, device=dev)
    t.pull(to_dev(keys, dev), out, out_lens if ragged else None)
    t.sync()
    assert_bits_equal(out.cpu().numpy(), o.pull(keys)[0])
    for mine, theirs in zip(t.dump(), o.dump()):
        assert np.array_equal(mine, theirs) if mine.dtype != np.float32 else assert_bits_equal(mine, theirs) is None
