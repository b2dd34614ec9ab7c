"""The packed potts/neigh and potts/neighonly pass (spk_neigh.h), run on the
host by tests/emul/spk_emul_neigh under AddressSanitizer, against the oracle:
both lattices and storage types, rows of every length mod 4, edge-2 boxes
(duplicate neighbours), random and coarse states, T = 0, the largest Q."""
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
EMUL = os.path.join(HERE, "emul", "spk_emul_neigh")

CASES = [
    # app, lattice, shape, Q, kT, seed, sweeps
    ("potts/neigh", "sc/26n", (16, 8, 6), 200, 0.5, 31, 4),
    ("potts/neighonly", "sc/26n", (10, 6, 8), 32767, 0.6, 32, 4),
    ("potts/neigh", "sc/26n", (12, 4, 6), 3, 0.9, 33, 6),       # few values: most are repeats
    ("potts/neighonly", "sc/26n", (14, 6, 4), 2, 1.5, 34, 6),
    ("potts/neigh", "sc/26n", (2, 2, 2), 5, 0.7, 35, 6),
    ("potts/neighonly", "sc/26n", (2, 4, 6), 4, 0.0, 36, 6),
    ("potts/neigh", "sc/26n", (18, 4, 2), 1, 0.5, 37, 3),       # no unlike neighbour at all
    ("potts/neighonly", "sc/26n", (18, 4, 2), 1, 0.5, 38, 3),   # and no draw
    ("potts/neigh", "sq/8n", (22, 6, 1), 255, 0.4, 39, 6),
    ("potts/neighonly", "sq/8n", (16, 14, 1), 20000, 0.0, 40, 12),
    ("potts/neigh", "sq/8n", (2, 2, 1), 3, 0.8, 41, 6),
    ("potts/neighonly", "sq/8n", (34, 4, 1), 9, 0.3, 42, 12),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "%s-%s-%s-q%d" % (c[0], c[1], "x".join(map(str, c[2])), c[3]))
def test_packed_neigh_passes_give_the_oracles_sweeps(orc, tmp_path, case):
    app, lat, shape, q, kt, seed, n = case
    d = orc.make_desc(app, lat, *shape, q, kt)
    spin0, seeds0 = orc.script_init(d, seed, 1, q)
    spin, seeds = spin0.copy(), seeds0.copy()
    e0 = orc.energy(d, spin)
    nacc, eng = orc.sweeps(d, spin, seeds, n)
    fin, fout = str(tmp_path / "in.bin"), str(tmp_path / "out.bin")
    np.concatenate([spin0, seeds0]).astype(np.int32).tofile(fin)
    apps, lats = {"potts/neigh": 2, "potts/neighonly": 3}, {"sq/8n": 1, "sc/26n": 3}
    for stype in (0, 1) if q < 256 else (1,):
        subprocess.run([EMUL, str(apps[app]), str(lats[lat]), *map(str, shape), str(q), repr(kt), str(n), str(stype),
                        fin, fout], check=True, timeout=120)
        N = spin.size
        raw = open(fout, "rb").read()
        got = np.frombuffer(raw[:8 * N], np.int32)
        rows = np.frombuffer(raw[8 * N:], np.int64).reshape(n, 2)
        assert np.array_equal(got[:N], spin) and np.array_equal(got[N:], seeds), stype
        assert np.array_equal(np.cumsum(rows[:, 0]), nacc)
        assert np.array_equal(e0 + 2 * np.cumsum(rows[:, 1]), eng)
