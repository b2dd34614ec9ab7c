"""Lattices of boxes whose single sweeps go one colour a launch, against the oracle
on the GPU: the state from one kind of call to the other."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("case", [
    # app, lattice, shape, Q, launches of a single sweep
    ("ising", "sq/4n", (362, 5944, 1), 2, 2),
    ("potts", "sq/4n", (210, 150, 1), 30, 2),
    ("potts", "sq/8n", (1400, 1402, 1), 100, 4),
    ("potts", "sc/6n", (40, 42, 44), 300, 2),
], ids=lambda c: "%s-%s-%s" % (c[0], c[1], "x".join(map(str, c[2]))))
def test_single_sweeps_equal_oracle(orc, case):
    import spparks_amd as S
    app, lat, shape, q, launches = case
    print("single sweeps", case, flush=True)
    d = orc.make_desc(app, lat, *shape, q, 0.7)
    spin, seeds = orc.script_init(d, 17, 1, q)
    with S.Lattice(app, lat, *shape, nspins=q, temperature=0.7) as L:
        L.upload(spin, seeds)
        for n in (1, 2, 1, 3):
            nacc, eng = orc.sweeps(d, spin, seeds, n)
            _, gn, ge = L.sweeps(n)
            assert np.array_equal(gn, nacc) and np.array_equal(ge, eng), n
            assert n > 1 or L.last_timing()[1] == launches
        s, k = L.download()
        assert np.array_equal(s, spin) and np.array_equal(k, seeds)
