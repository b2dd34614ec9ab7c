"""Lattices that sweep on bit planes of the spins (k_sweep_slice) against the
oracle on the GPU: words of 32 sites and of fewer, one to five plane groups,
rows of one word to sixteen, idle lanes, T = 0, two states; the state handed
to and from the other layouts."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [
    # app, shape, Q, kT, seed
    ("potts", (128, 128, 128), 10000, 0.5, 1),
    ("potts", (128, 120, 130), 16, 0.9, 2),         # one plane group
    ("potts", (190, 100, 90), 200, 0.6, 3),         # three words of 32, 32, 31: idle quads
    ("potts", (1022, 50, 42), 3000, 0.5, 4),        # 16 words a row
    ("potts", (134, 126, 124), 1000000, 0.3, 5),    # three words of 23, 23, 21; five plane groups
    ("potts", (160, 120, 110), 65536, 0.0, 6),      # T = 0
    ("ising", (192, 110, 100), 2, 3.0, 7),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "%s-%s-q%d" % (c[0], "x".join(map(str, c[1])), c[2]))
def test_sliced_sweeps_equal_oracle(orc, case):
    import spparks_amd as S
    app, shape, q, kt, seed = case
    print("sliced", case, flush=True)
    d = orc.make_desc(app, "sc/26n", *shape, q, kt)
    spin, seeds = orc.script_init(d, seed, 1, q)
    with S.Lattice(app, "sc/26n", *shape, nspins=q, temperature=kt) as L:
        L.upload(spin, seeds)

        def run(n, launches):
            nacc, eng = orc.sweeps(d, spin, seeds, n)
            tot, gn, ge = L.sweeps(n)
            assert np.array_equal(gn, nacc) and np.array_equal(ge, eng) and tot == nacc[-1], n
            assert L.last_timing()[1] == launches * n

        run(1, 4)
        L.prepare(2)
        run(2, 4)
        s, k = L.download()
        assert np.array_equal(s, spin) and np.array_equal(k, seeds)
        L.set_graph(0)
        run(1, 4)
        assert L.energy() == orc.energy(d, spin)
        # a chosen workgroup size keeps the per-colour kernels; the state carries over
        L.set_launch(256)
        run(1, 8)
        s, k = L.download()
        assert np.array_equal(s, spin) and np.array_equal(k, seeds)


def test_state_carries_from_planes_to_sweeps_without_allocation(orc):
    import spparks_amd as S
    from test_zz_no_alloc import DeviceRows
    d = orc.make_desc("potts", "sc/26n", 128, 128, 128, 500, 0.6)
    spin, seeds = orc.script_init(d, 9, 1, 500)
    orc.sweeps(d, spin, seeds, 3)
    with S.Lattice("potts", "sc/26n", 128, 128, 128, nspins=500, temperature=0.6) as L:
        s0, rseed = S.strict_init_params(9)
        L.set_range(s0, 1, 500)
        L.init_seeds(rseed)
        L.sweeps(1)
        rows = DeviceRows(2)
        L.sweeps_noalloc(1, rows.ptr.value)
        L.sync()
        rows.free()
        L.sweeps(1)
        s, k = L.download()
    assert np.array_equal(s, spin) and np.array_equal(k, seeds)
