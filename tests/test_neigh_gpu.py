"""The packed potts/neigh and potts/neighonly kernel (k_sweep_neigh) against
the oracle on the GPU: both sides of the sizes and values it takes, both
storage types, rows of every length mod 4, random and coarse states, T = 0."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [
    # app, lattice, shape, Q, kT, seed, sweeps
    ("potts/neigh", "sc/26n", (94, 90, 92), 200, 0.5, 51, 3),
    ("potts/neighonly", "sc/26n", (96, 94, 90), 32767, 0.6, 52, 3),
    ("potts/neighonly", "sc/26n", (96, 94, 90), 32768, 0.6, 53, 2),   # one value more: the one-site kernel
    ("potts/neigh", "sc/26n", (98, 92, 88), 3, 0.9, 54, 4),
    ("potts/neighonly", "sc/26n", (100, 88, 90), 2, 1.5, 55, 4),
    ("potts/neigh", "sc/26n", (2, 2, 2), 5, 0.7, 56, 5),
    ("potts/neigh", "sq/8n", (1030, 1024, 1), 255, 0.4, 57, 4),       # just above the line
    ("potts/neighonly", "sq/8n", (1036, 1020, 1), 20000, 0.0, 58, 6),
    ("potts/neigh", "sq/8n", (1024, 1024, 1), 256, 0.5, 59, 3),       # on it: the one-site kernel
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "%s-%s-%s-q%d" % (c[0], c[1], "x".join(map(str, c[2])), c[3]))
def test_packed_neigh_equals_oracle(orc, case):
    import spparks_amd as S
    app, lat, shape, q, kt, seed, n = case
    print("neigh", case, flush=True)
    d = orc.make_desc(app, lat, *shape, q, kt)
    spin, seeds = orc.script_init(d, seed, 1, q)
    with S.Lattice(app, lat, *shape, nspins=q, temperature=kt) as L:
        L.upload(spin, seeds)
        for block in (0, 64, 1024):   # 0: the default; a chosen one keeps the per-colour kernels
            if block:
                L.set_launch(block)
            nacc, eng = orc.sweeps(d, spin, seeds, n)
            tot, gn, ge = L.sweeps(n)
            assert np.array_equal(gn, nacc) and np.array_equal(ge, eng) and tot == nacc[-1], block
        s, k = L.download()
        assert np.array_equal(s, spin) and np.array_equal(k, seeds)
