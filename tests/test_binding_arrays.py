"""Numpy arrays of every form as arguments of a slice (host memory: no GPU is asked): what the quick way of the binding takes as it
is, and what it leaves to the general way, which converts it."""
import numpy as np
import pytest


def _unaligned(a):
    room = np.zeros(a.nbytes + 1, np.uint8)
    room[1:] = np.frombuffer(a.tobytes(), np.uint8)
    return room[1:].view(a.dtype)


class _Sub(np.ndarray):
    pass


def _read_only(a):
    a = a.copy()
    a.setflags(write=False)
    return a


FORMS = {"plain": lambda a: a, "strided": lambda a: np.repeat(a, 2)[::2], "reversed": lambda a: a[::-1].copy()[::-1],
         "unaligned": _unaligned, "swapped": lambda a: a.astype(a.dtype.newbyteorder()), "subclass": lambda a: a.view(_Sub),
         "read-only": _read_only, "fortran": lambda a: np.asfortranarray(a), "long long": lambda a: a.astype("Q") if a.dtype == np.uint64 else a,
         "list": lambda a: a.tolist()}


@pytest.mark.parametrize("S", [0, 1, 3, 40])
@pytest.mark.parametrize("form", sorted(FORMS))
def test_slices_of_arrays_of_every_form(capi, form, S):
    n = 1000 if S else 0
    keys = np.sort(np.random.default_rng(S).integers(0, 1 << 63, n, dtype=np.uint64))
    lens = np.arange(n, dtype=np.int32) % 7
    begin, end = capi.server_ranges(S) if S else (np.zeros(0, np.uint64), np.zeros(0, np.uint64))
    give = FORMS[form]
    pos, val_pos, used = capi.slice_keys(give(keys), give(begin), give(end), lens=give(lens), nvals=int(lens.sum()))
    assert pos.dtype == val_pos.dtype == np.uint64 and used.dtype == np.uint8
    assert pos.shape == val_pos.shape == (S + 1,) and used.shape == (S,)
    want = np.concatenate([[0], np.searchsorted(keys, end)]).astype(np.uint64) if S else np.zeros(1, np.uint64)
    want_vals = np.concatenate([[0], np.cumsum(lens)])[want.astype(int)]
    assert np.array_equal(pos, want) and np.array_equal(val_pos, want_vals)
    assert np.array_equal(used != 0, np.diff(pos) != 0)
    if S > 1:  # (ranges that do not follow each other)
        with pytest.raises(capi.PskvError):
            capi.slice_keys(give(keys), give(begin), give(end[::-1].copy()), nvals=n)
