"""The proof-of-work search with every number of pending inputs (the smallest
witness, against the oracle's challenger), and the reduced openings of heights on
both sides of the line between one and four waves per 64 rows."""
import numpy as np
import pytest

import pico_amd
from pico_amd import BABYBEAR, KOALABEAR

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("f", [KOALABEAR, BABYBEAR])
@pytest.mark.parametrize("pending", range(8))
def test_grind_finds_the_smallest_witness(ctx, oracle, f, pending):
    for bits in (0, 1, 6, 12):
        ch, och = pico_amd.DuplexChallenger(f), oracle.Challenger(f)
        seen = list(range(3, 3 + 8 + pending))  # one permutation, `pending` inputs left
        for c in (ch, och):
            c.observe(seen)
        print(f"grind field {f} pending {pending} bits {bits}", flush=True)
        w = pico_amd.fri_grind(ctx, f, ch, bits)
        assert not any(och.clone().check_witness(bits, c) for c in range(w))
        assert och.check_witness(bits, w)


@pytest.mark.parametrize("f", [KOALABEAR, BABYBEAR])
@pytest.mark.parametrize("log_h", [0, 3, 6, 14, 15])
@pytest.mark.parametrize("nmats", [1, 3, 6])
def test_reduced_rows_match_oracle(ctx, oracle, f, log_h, nmats):
    p = pico_amd.PRIMES[f]
    widths = [1, 33, 4, 64, 7, 32][:nmats]
    hosts = [oracle.random_matrix(f, 40 + i, 1 << log_h, w) for i, w in enumerate(widths)]
    pcs = pico_amd.TwoAdicFriPcs(ctx, f, 1)
    dom = pcs.natural_domain_for_degree(1 << log_h)
    _, data = pcs.commit([(dom, ctx.upload(a, field=f)) for a in hosts])
    rng = np.random.default_rng(13 + nmats)
    pts = rng.integers(0, p, (2, 4)).astype(np.uint32)
    alpha = rng.integers(0, p, 4).astype(np.uint32)
    print(f"reduce field {f} 2^{log_h} x {nmats} matrices", flush=True)
    vals = [pcs.open_values(data, k, pts) for k in range(nmats)]
    ro = pcs.reduce_openings([(data, [pts] * nmats)], [vals], alpha)
    ldes = [oracle.coset_lde(f, a, 1, pico_amd.GENERATORS[f]) for a in hosts]
    ref = oracle.pcs_reduce(f, ldes, [2] * nmats, np.concatenate([pts] * nmats),
                            [v[q] for v in vals for q in range(2)], alpha)
    assert list(ro) == [log_h + 1]
    assert np.array_equal(ro[log_h + 1].to_host(f), ref[log_h + 1])
    data.free()
