"""Which kernel a program gets (no GPU needed): programs on either side of every
limit of the resident form and of the rule between the two."""
import pytest

import pico_amd
from pico_amd import KOALABEAR, air, workloads
from pico_amd.air import RESIDENT, WINDOWED


def wide(columns, constants=0):
    """One constraint per column: three products, a difference."""
    b = air.AirBuilder(KOALABEAR)
    for c in range(columns):
        x, y, z = b.main(c), b.main((c + 1) % columns), b.main((c + 2) % columns)
        x = x * y * z - b.main(c, next=True)
        b.when_transition().assert_zero(x + (2 + c) if c < constants else x)
    return b


def shared(rounds, columns=20):
    b = air.AirBuilder(KOALABEAR)
    s = [b.main(c) for c in range(columns)]
    for _ in range(rounds):
        s = [s[i] * s[(i + 1) % columns] + s[(i + 5) % columns] for i in range(columns)]
    for x in s:
        b.assert_zero(x)
    return b


FEW = 1 << 10
MANY = 1 << 21


@pytest.mark.parametrize("builder,few,many", [
    (lambda: wide(1), WINDOWED, WINDOWED),         # a short program is a short chain
    (lambda: wide(4), RESIDENT, WINDOWED),         # staging costs more than the program over many rows
    (lambda: wide(12), RESIDENT, RESIDENT),
    (lambda: wide(40), RESIDENT, RESIDENT),
    (lambda: wide(256), RESIDENT, RESIDENT),       # 512 column slots
    (lambda: wide(305), RESIDENT, RESIDENT),       # 610 slots
    (lambda: wide(320), WINDOWED, WINDOWED),       # 640: more than LDS holds
    (lambda: wide(40, 40), RESIDENT, RESIDENT),
    (lambda: wide(256, 256), WINDOWED, WINDOWED),  # the constants no longer fit
    (lambda: shared(1), RESIDENT, RESIDENT),
    (lambda: shared(8), WINDOWED, WINDOWED),       # each slice would repeat most of the work
    (lambda: workloads.lookup_air(90, 24, 2)[0], RESIDENT, RESIDENT),
    (lambda: workloads.lookup_air(300, 100, 2)[0], WINDOWED, WINDOWED),
], ids=["1 column", "4 columns", "12 columns", "40 columns", "256 columns", "305 columns", "320 columns", "constants", "many constants",
        "little shared", "much shared", "24 lookups", "100 lookups"])
def test_form(builder, few, many):
    p = builder().compile()
    assert (p.form(FEW), p.form(MANY)) == (few, many)


def test_fixed_form():
    p, q = wide(40).compile(), shared(8).compile()
    p.debug_form(WINDOWED)
    assert p.form(MANY) == WINDOWED
    p.debug_form(None)
    assert p.form(MANY) == RESIDENT
    with pytest.raises(pico_amd.PgError):
        q.debug_form(RESIDENT)
    with pytest.raises(pico_amd.PgError):
        p.debug_form(7)
    assert q.form(FEW) == WINDOWED and p.form(3) == 0 and p.form(0) == 0
