"""Two sweeps per launch in every band and stage (k_sweep_bits_pair) against
the oracle on the GPU, on lattices that the library sends there."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [
    # app, shape, kT, seed: band and stage as the rows and their number give
    ("ising", (1022, 1000, 1), 2.269, 1),           # 4, 64
    ("ising/single", (1024, 2000, 1), 2.269, 2),    # 8, 64
    ("ising", (900, 3070, 1), 1.7, 3),              # 12, 64
    ("ising", (1500, 1002, 1), 2.269, 4),           # 4, 128
    ("ising", (2048, 2046, 1), 0.0, 5),             # 8, 128
    ("ising/single", (1300, 2500, 1), 2.4, 6),      # 12, 128
    ("ising", (2000, 3100, 1), 2.269, 7),           # 16, 128
    ("ising", (3000, 1020, 1), 2.269, 8),           # 4, 256
    ("ising/single", (3000, 2006, 1), 2.269, 9),    # 8, 256
    ("ising", (2600, 3002, 1), 2.269, 10),          # 12, 256
    ("ising", (4096, 1024, 1), 2.269, 11),          # 4, whole rows
    ("ising/single", (4096, 1500, 1), 2.269, 12),   # 8, whole rows
    ("potts", (4096, 2600, 1), 0.9, 13),            # 12, whole rows
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "%s-%dx%d" % (c[0], c[1][0], c[1][1]))
def test_two_sweeps_a_launch_equal_oracle(orc, case):
    import spparks_amd as S
    app, shape, kt, seed = case
    print("pairs", case, flush=True)
    d = orc.make_desc(app, "sq/4n", *shape, 2, kt)
    spin, seeds = orc.script_init(d, seed, 1, 2)
    with S.Lattice(app, "sq/4n", *shape, nspins=2, temperature=kt) as L:
        L.upload(spin, seeds)
        for n in (8, 5):
            nacc, eng = orc.sweeps(d, spin, seeds, n)
            _, gn, ge = L.sweeps(n)
            assert np.array_equal(gn, nacc) and np.array_equal(ge, eng), n
            assert L.last_timing()[1] == 2 * (n // 4) + 2 * (n % 4), "not two sweeps a launch"
        s, k = L.download()
    assert np.array_equal(s, spin) and np.array_equal(k, seeds)
