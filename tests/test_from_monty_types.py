"""from_monty gives back the kind of value it is given: numpy scalars for scalars
(they hash and work as dictionary keys), arrays for arrays; what numpy cannot
hold as unsigned words is refused."""
import numpy as np
import pytest

import pico_amd
from pico_amd.core import from_monty, to_monty

FIELDS = [pico_amd.KOALABEAR, pico_amd.BABYBEAR]


@pytest.mark.parametrize("f", FIELDS)
@pytest.mark.parametrize("make", [int, np.uint32, np.uint64, np.int64, lambda x: np.array(x, np.uint32),
                                  lambda x: np.array([x], np.uint32)[0]],
                         ids=["int", "uint32", "uint64", "int64", "0-d array", "element"])
def test_scalars(f, make):
    for x in (0, 1, 5, pico_amd.PRIMES[f] - 1):
        got = from_monty(f, make(int(to_monty(f, x))))
        assert type(got) is np.uint32 and got == x and hash(got) == hash(x)
        assert {x: "found"}[got] == "found"


@pytest.mark.parametrize("f", FIELDS)
def test_arrays(f):
    words = np.arange(12, dtype=np.uint32)
    want = from_monty(f, words.tolist())
    for a in (words, words.reshape(3, 4), words.reshape(3, 4).T, words.reshape(1, 12, 1), words[:1], words[:0],
              words.astype(">u4"), words.astype(np.uint16)):
        got = from_monty(f, a)
        assert type(got) is np.ndarray and got.dtype == np.uint32 and got.shape == a.shape
        assert np.array_equal(got, want[np.asarray(a, np.int64)])


@pytest.mark.parametrize("f", FIELDS)
def test_refused(f):
    for a in (-1, [-1, 2], [2 ** 64], [None]):
        with pytest.raises((OverflowError, TypeError)):
            from_monty(f, a)
    assert np.array_equal(from_monty(f, [2 ** 63, 1]), from_monty(f, np.array([2 ** 63, 1], np.uint64)))
