"""Lattices that sweep in boxes (k_sweep_tile) against the oracle on the GPU:
calls of one sweep (split between two launches), of a launch, of several with
a remainder, and the state handed to and from the other kernels."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [
    # app, lattice, shape, Q, kT, seed
    ("ising", "sq/4n", (306, 250, 1), 2, 2.269, 1),        # ragged rows, clipped boxes
    ("ising", "sq/4n", (2046, 130, 1), 2, 2.0, 2),
    ("ising/single", "sq/4n", (300, 202, 1), 2, 2.269, 3),
    ("potts", "sq/4n", (210, 150, 1), 30, 0.7, 4),
    ("potts", "sq/8n", (128, 128, 1), 100, 0.5, 5),        # would fit one workgroup
    ("potts", "sq/8n", (330, 274, 1), 300, 0.6, 6),
    ("potts", "sc/6n", (40, 40, 40), 9, 0.9, 7),
    ("potts", "sc/26n", (50, 36, 30), 70000, 0.5, 8),
    ("potts", "sc/26n", (32, 32, 32), 255, 0.0, 9),
    ("potts/neigh", "sc/26n", (34, 32, 30), 300, 0.5, 10),
    ("potts/neighonly", "sq/8n", (202, 150, 1), 70000, 0.7, 11),
]
COLOURS = {"sq/4n": 2, "sq/8n": 4, "sc/6n": 2, "sc/26n": 8}
CALLS = [1, 2, 5, 1, 9, 33]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "%s-%s-%s" % (c[0], c[1], "x".join(map(str, c[2]))))
def test_boxes_equal_oracle(orc, case):
    import spparks_amd as S
    app, lat, shape, q, kt, seed = case
    print("boxes", case, flush=True)
    d = orc.make_desc(app, lat, *shape, q, kt)
    spin, seeds = orc.script_init(d, seed, 1, q)
    with S.Lattice(app, lat, *shape, nspins=q, temperature=kt) as L:
        L.upload(spin, seeds)
        for k, n in enumerate(CALLS):
            nacc, eng = orc.sweeps(d, spin, seeds, n)
            if k % 2:
                L.prepare(n)
            if k == 3:
                L.set_graph(0)      # launches from the host, from here on
            tot, gn, ge = L.sweeps(n)
            assert np.array_equal(gn, nacc) and np.array_equal(ge, eng) and tot == nacc[-1], n
            if n > 1:
                launches = L.last_timing()[1]
                assert launches < COLOURS[lat] * n and launches % 2 == 0, "not in boxes"
        s, k = L.download()
        assert np.array_equal(s, spin) and np.array_equal(k, seeds)
        # a chosen workgroup size keeps the per-colour kernels; the state carries over
        L.set_launch(256)
        nacc, eng = orc.sweeps(d, spin, seeds, 3)
        _, gn, ge = L.sweeps(3)
        assert np.array_equal(gn, nacc) and np.array_equal(ge, eng)
        s, k = L.download()
        assert np.array_equal(s, spin) and np.array_equal(k, seeds)
