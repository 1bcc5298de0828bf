"""from_monty of machine words against its definition (x / 2^32 mod p), every
class of word: below p, multiples of p and their neighbours, the largest."""
import numpy as np
import pytest

import pico_amd
from pico_amd.core import from_monty


@pytest.mark.parametrize("f", [pico_amd.KOALABEAR, pico_amd.BABYBEAR])
def test_from_monty_words(f):
    p = pico_amd.PRIMES[f]
    edge = [0, 1, p - 1, p, p + 1, 2 * p - 1, 2 * p, 2 * p + 1, 2 ** 31, 2 ** 32 - 1]
    words = np.concatenate([np.array(edge, np.uint64),
                            np.random.default_rng(1).integers(0, 2 ** 32, 6000, dtype=np.uint64)])
    rinv = pow(2 ** 32, p - 2, p)
    want = np.array([int(x) * rinv % p for x in words], np.uint32)
    small = words.astype(np.uint32)
    for a in (words, small, small.reshape(10, -1)[:, ::3], small[:0], small[3], list(map(int, words[:9]))):
        got = from_monty(f, a)
        assert got.dtype == np.uint32 and got.shape == np.shape(a)
        if a is words or a is small:
            assert np.array_equal(got, want)
    assert np.array_equal(from_monty(f, small.reshape(10, -1)[:, ::3]), want.reshape(10, -1)[:, ::3])
    assert int(from_monty(f, small[3])) == int(want[3])
