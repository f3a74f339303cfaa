"""Arrays of every form as the place that a pull's answer goes to: what the library writes itself, and what the binding takes
there from a copy."""
import array

import numpy as np
import pytest

from conftest import announce
from helpers import assert_bits_equal, unique_keys

pytestmark = pytest.mark.gpu


class _Sub(np.ndarray):
    pass


def _unaligned(a):
    return np.zeros(a.nbytes + 1, np.uint8)[1:].view(a.dtype)


# from an array of n values: another of the same number of them, in the form
FORMS = {"plain": lambda a: a, "strided": lambda a: np.repeat(a, 3)[::3], "reversed": lambda a: a[::-1], "unaligned": _unaligned,
         "swapped": lambda a: a.astype(a.dtype.newbyteorder()), "subclass": lambda a: a.view(_Sub),
         "wider": lambda a: a.astype(np.float64 if a.dtype == np.float32 else np.int64), "columns": lambda a: a.reshape(2, -1).T,
         "buffer": lambda a: memoryview(a.copy()), "wider buffer": lambda a: array.array("d" if a.dtype == np.float32 else "q", a.tolist())}


@pytest.mark.parametrize("call", ["pull", "pushpull"])
@pytest.mark.parametrize("mode", ["scalar", "varlen"])
@pytest.mark.parametrize("form", sorted(FORMS))
def test_answers_reach_arrays_of_every_form(capi, dev, form, mode, call):
    announce("answers", form, mode, call)
    rng = np.random.default_rng(3)
    n = 300
    keys, lens = unique_keys(rng, n), rng.integers(1, 9, n).astype(np.int32)
    varlen = mode == "varlen"
    total = int(lens.sum()) if varlen else n
    vals = rng.standard_normal(total).astype(np.float32)
    t = capi.Table(capi.MODE_VARLEN if varlen else capi.MODE_SCALAR)
    t.push(keys, vals, lens if varlen else None)
    room = total + total % 2 + 4
    out = FORMS[form](np.full(room, 0.1, np.float32))
    untouched = np.asarray(out).ravel()[total:].copy()
    out_lens = FORMS[form](np.full(n, -7, np.int32)) if varlen else None
    if call == "pull":
        want = vals
        got = t.pull(keys, out, out_lens)
    else:
        want = vals + vals
        got = t.pushpull(keys, vals, out, lens if varlen else None, out_lens)
    assert got == t.last_out_nvals == total
    answer = np.asarray(out).ravel()
    assert_bits_equal(answer[:total].astype(np.float32), want)
    assert np.array_equal(answer[total:], untouched)
    if varlen:
        assert np.array_equal(np.asarray(out_lens).ravel(), lens)


def test_places_that_no_answer_can_go_to(capi, dev):
    announce("answers refused")
    t = capi.Table(capi.MODE_SCALAR)
    keys, vals = np.arange(1, 5, dtype=np.uint64), np.ones(4, np.float32)
    t.push(keys, vals)
    wide = np.zeros(4)
    wide.setflags(write=False)
    for out, error in ((np.zeros(4, np.int64), TypeError), ([0.0] * 4, TypeError), (wide, ValueError)):
        with pytest.raises(error):
            t.pull(keys, out)
        with pytest.raises(error):
            t.pushpull(keys, vals, out)
    out = np.zeros(4, np.float32)
    t.pull(keys, out)
    assert_bits_equal(out, vals)  # (nothing has been pushed)
