"""pskv_match where its workgroups stop finding their stretches themselves (2,560 tiles of 1,024 keys, 4,096 of them where the
other set is small, or of 256 where it is twice as large): as many tiles and one more, and tiles whose keys all lie in front
of, behind or between those of the other set. Against numpy, bit for bit."""
import numpy as np
import pytest

from conftest import announce
from helpers import assert_bits_equal, from_dev, to_dev
from test_oracle_match import key_sets, numpy_model

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_src,n_dst", [(3_000_000, 4096 * 1024), (3_000_000, 4096 * 1024 + 1),
                                         (2_200_000, 4096 * 256), (2_200_000, 4096 * 256 + 1),
                                         (3_200_000, 2560 * 1024), (3_200_000, 2560 * 1024 + 1),
                                         ((29 << 18) - 5_250_000, 3_000_000), ((29 << 18) - 5_249_999, 3_000_000)])
@pytest.mark.parametrize("k", [1, 3])
def test_as_many_tiles_as_search_for_themselves(capi, dev, n_src, n_dst, k):
    announce("match own spans", n_src, n_dst, k)
    rng = np.random.default_rng(n_dst + k)
    sk, dk = key_sets(rng, n_src, n_dst, n_src // 2)
    sv = rng.integers(-50, 50, sk.size * k).astype(np.float32)
    dv = rng.integers(-50, 50, dk.size * k).astype(np.float32)
    want, want_n = numpy_model(sk, sv, dk, dv, k, 1)
    got = to_dev(dv, dev)
    assert capi.match(to_dev(sk, dev), to_dev(sv, dev), to_dev(dk, dev), got, k, capi.OP_PLUS) == want_n
    assert_bits_equal(from_dev(got), want)


@pytest.mark.parametrize("n_dst", [1, 256, 257, 600_000])
def test_tiles_outside_the_other_set(capi, dev, n_dst):
    announce("match outside", n_dst)
    dk = np.arange(n_dst, dtype=np.uint64) * np.uint64(16) + np.uint64(1 << 40)
    dv = np.ones(n_dst, np.float32)
    for sk in (np.arange(5000, dtype=np.uint64), np.arange(5000, dtype=np.uint64) + np.uint64(1 << 50), dk[:1] + np.uint64(1),
               dk[-1:], dk[n_dst // 2:n_dst // 2 + 1], np.concatenate([np.arange(300, dtype=np.uint64), dk[-1:]])):
        sv = np.full(sk.size, 2, np.float32)
        want, want_n = numpy_model(sk, sv, dk, dv, 1, 1)
        got = to_dev(dv, dev)
        assert capi.match(to_dev(sk, dev), to_dev(sv, dev), to_dev(dk, dev), got, 1, capi.OP_PLUS) == want_n
        assert_bits_equal(from_dev(got), want)


def _sets(kind, rng, n):
    if kind == "even":
        return np.arange(n, dtype=np.uint64) * np.uint64(3)
    if kind == "squares":
        return np.arange(n, dtype=np.uint64) ** np.uint64(2)
    if kind == "clusters":
        return np.unique((rng.integers(0, 1 << 40, 700, dtype=np.uint64) << np.uint64(20))[:, None]
                         + np.arange(n // 700 + 1, dtype=np.uint64)).ravel()
    if kind == "far away":  # all but a few of the keys
        return np.concatenate([np.arange(9, dtype=np.uint64), np.uint64(1 << 63) + np.arange(n, dtype=np.uint64)])
    return np.unique(rng.integers(0, 1 << 64, n, dtype=np.uint64))


@pytest.mark.parametrize("kind", ["even", "squares", "clusters", "far away", "any"])
@pytest.mark.parametrize("n_src,n_dst", [(2_000_000, 2560 * 1024), (2_700_000, 2561 * 1024 + 3), (1100, 2_700_000)])
def test_stretches_wherever_the_keys_lie(capi, dev, kind, n_src, n_dst):
    """Searches that guess from the keys around: keys spread evenly, by the square, in clusters, and with a gap."""
    announce("match guesses", kind, n_src, n_dst)
    rng = np.random.default_rng(n_dst)
    both = _sets(kind, rng, n_src + n_dst // 2)
    sk = np.sort(rng.choice(both, min(n_src, both.size), replace=False))
    dk = np.unique(np.concatenate([rng.choice(both, n_dst // 2, replace=False), both + np.uint64(1)]))[:n_dst]
    sv = rng.integers(-50, 50, sk.size).astype(np.float32)
    dv = rng.integers(-50, 50, dk.size).astype(np.float32)
    want, want_n = numpy_model(sk, sv, dk, dv, 1, 1)
    got = to_dev(dv, dev)
    assert capi.match(to_dev(sk, dev), to_dev(sv, dev), to_dev(dk, dev), got, 1, capi.OP_PLUS) == want_n
    assert_bits_equal(from_dev(got), want)
