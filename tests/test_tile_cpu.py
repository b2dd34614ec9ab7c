"""The tile kernel's own steps (spk_tile.h: load a box with its halo, run
several colour passes on it, store what it owns), run on the host by
tests/emul/spk_emul_tile under AddressSanitizer, against the oracle: boxes
that cut every dimension, that span some, that are clipped at the lattice's
end, that with their halo are wider than the lattice; launches that start
and end inside a sweep."""
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
EMUL = os.path.join(HERE, "emul", "spk_emul_tile")
COLOURS = {"sq/4n": 2, "sq/8n": 4, "sc/6n": 2, "sc/26n": 8}

CASES = [
    # app, lattice, shape, Q, kT, seed, storage, box, passes of each launch
    ("ising", "sq/4n", (64, 48, 1), 2, 2.269, 1, 0, (16, 12, 1), [8, 8]),
    ("ising", "sq/4n", (50, 38, 1), 2, 2.0, 2, 0, (24, 10, 1), [4, 6]),      # ragged rows, clipped boxes
    ("ising", "sq/4n", (18, 6, 1), 2, 2.0, 3, 0, (8, 4, 1), [16, 32]),       # halo wider than the lattice
    ("ising", "sq/4n", (34, 64, 1), 2, 1.8, 4, 0, (34, 8, 1), [1, 1, 2]),    # whole ragged rows; a sweep in two launches
    ("ising", "sq/4n", (40, 20, 1), 2, 0.0, 5, 0, (8, 20, 1), [4, 4]),       # T = 0; whole columns
    ("potts", "sq/4n", (44, 26, 1), 5, 1.1, 6, 0, (16, 8, 1), [4, 4]),
    ("potts", "sq/4n", (30, 26, 1), 70000, 0.4, 7, 2, (8, 6, 1), [2, 6]),
    ("potts", "sq/8n", (64, 64, 1), 100, 0.5, 8, 0, (16, 8, 1), [16, 16]),
    ("potts", "sq/8n", (54, 42, 1), 9, 0.9, 9, 0, (24, 10, 1), [2, 2, 4]),
    ("potts", "sq/8n", (38, 50, 1), 300, 0.7, 10, 1, (38, 6, 1), [8, 12]),
    ("ising", "sq/8n", (26, 22, 1), 2, 1.5, 11, 0, (8, 2, 1), [32]),
    ("potts", "sc/6n", (30, 14, 10), 9, 0.9, 12, 0, (16, 6, 4), [4, 4]),
    ("ising", "sc/6n", (22, 12, 10), 2, 1.7, 13, 0, (22, 4, 6), [3, 3]),
    ("potts", "sc/26n", (32, 16, 12), 10000, 0.5, 14, 1, (32, 4, 4), [8, 8]),
    ("potts", "sc/26n", (22, 14, 10), 255, 0.6, 15, 0, (8, 6, 4), [4, 4, 16]),
    ("potts", "sc/26n", (18, 10, 6), 70000, 0.4, 16, 2, (16, 10, 2), [4, 12]),
    ("potts", "sc/26n", (10, 6, 2), 4, 0.6, 17, 0, (8, 2, 2), [16, 8]),
    ("ising", "sc/26n", (12, 10, 8), 2, 3.0, 18, 0, (12, 10, 2), [24]),
    ("potts/neigh", "sq/4n", (20, 14, 1), 5, 0.8, 19, 0, (8, 6, 1), [4, 4]),
    ("potts/neigh", "sc/26n", (18, 8, 6), 300, 0.5, 20, 1, (8, 4, 4), [8, 8]),
    ("potts/neigh", "sc/6n", (12, 8, 6), 7, 0.0, 21, 0, (8, 8, 2), [2, 4]),
    ("potts/neighonly", "sq/8n", (26, 14, 1), 70000, 0.7, 22, 2, (8, 4, 1), [8, 4]),
    ("potts/neighonly", "sc/26n", (10, 6, 4), 9, 0.6, 23, 0, (10, 2, 2), [4, 4]),
    ("ising/single", "sq/4n", (42, 30, 1), 2, 2.269, 24, 0, (16, 8, 1), [8, 4]),
    ("ising/single", "sc/6n", (14, 10, 6), 2, 1.7, 25, 0, (8, 4, 4), [4]),
]


@pytest.mark.parametrize("vec", [4, 1])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "%s-%s-%s-%s" % (c[0], c[1], "x".join(map(str, c[2])),
                                                                       "x".join(map(str, c[7]))))
def test_boxes_give_the_oracles_sweeps(orc, tmp_path, case, vec):
    app, lat, shape, q, kt, seed, stype, box, cuts = case
    if vec == 4 and app not in ("potts", "ising"):
        pytest.skip("the proposal variants run one site per thread")
    n = sum(cuts) // COLOURS[lat]
    d = orc.make_desc(app, lat, *shape, q, kt)
    spin, seeds = orc.script_init(d, seed, 1, q)
    e0 = orc.energy(d, spin)
    fin, fout = str(tmp_path / "in.bin"), str(tmp_path / "out.bin")
    np.concatenate([spin, seeds]).astype(np.int32).tofile(fin)
    nacc, eng = orc.sweeps(d, spin, seeds, n)
    apps = {"potts": 0, "ising": 1, "potts/neigh": 2, "potts/neighonly": 3, "ising/single": 4}
    lats = {"sq/4n": 0, "sq/8n": 1, "sc/6n": 2, "sc/26n": 3}
    subprocess.run([EMUL, str(apps[app]), str(lats[lat]), *map(str, shape), str(q), repr(kt), str(stype), str(vec),
                    *map(str, box), ",".join(map(str, cuts)), fin, fout], check=True, timeout=120)
    N = spin.size
    raw = open(fout, "rb").read()
    got = np.frombuffer(raw[:8 * N], np.int32)
    rows = np.frombuffer(raw[8 * N:], np.int64).reshape(n, 2)
    assert np.array_equal(got[:N], spin) and np.array_equal(got[N:], seeds)
    assert np.array_equal(np.cumsum(rows[:, 0]), nacc)
    assert np.array_equal(e0 + 2 * np.cumsum(rows[:, 1]), eng)
