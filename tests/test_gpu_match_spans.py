"""pskv_match where its workgroups stop finding their stretches themselves (4,096 tiles of 1,024 keys, or of 256 where the
other set is twice as large): one tile less and more, and tiles whose keys all lie in front of, behind or between those of
the other set. Against numpy, bit for bit."""
import numpy as np
import pytest

from conftest import announce
from helpers import assert_bits_equal, from_dev, to_dev
from test_oracle_match import key_sets, numpy_model

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_src,n_dst", [(3_000_000, 4096 * 1024), (3_000_000, 4096 * 1024 + 1),
                                         (2_200_000, 4096 * 256), (2_200_000, 4096 * 256 + 1)])
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
