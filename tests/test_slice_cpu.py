"""The bit-sliced passes' own steps (spk_slice.h), run on the host by
tests/emul/spk_emul_slice under AddressSanitizer, against the oracle: words
of 32 sites and of fewer, rows of one word and of several, idle lanes, plane
counts on both sides of a byte, edge-2 boxes, T = 0, two states."""
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
EMUL = os.path.join(HERE, "emul", "spk_emul_slice")

CASES = [
    # app, lattice, shape, Q, kT, seed, sweeps
    ("potts", "sc/26n", (64, 8, 8), 10000, 0.5, 11, 3),
    ("potts", "sc/26n", (128, 6, 4), 65536, 0.5, 12, 3),
    ("potts", "sc/26n", (20, 14, 10), 255, 0.6, 13, 4),
    ("potts", "sc/26n", (70, 6, 6), 1048576, 0.3, 14, 3),   # 20 planes
    ("potts", "sc/26n", (2, 2, 2), 4, 0.6, 15, 5),
    ("potts", "sc/26n", (2, 4, 6), 5, 1.4, 16, 4),
    ("potts", "sc/26n", (36, 2, 6), 300, 0.0, 17, 4),       # T = 0
    ("potts", "sc/26n", (102, 4, 4), 2, 1.2, 18, 4),
    ("ising", "sc/26n", (64, 6, 4), 2, 3.0, 19, 4),
    ("potts", "sc/26n", (128, 10, 2), 128, 0.7, 20, 3),     # 5 rows: the last wavefront partly idle
    ("potts", "sc/26n", (78, 6, 4), 129, 0.9, 21, 3),       # 39 sites: words of 20 and 19
    ("potts", "sc/26n", (66, 4, 4), 256, 0.6, 22, 3),       # 33 sites: 17 and 16
    ("potts", "sc/26n", (134, 4, 2), 257, 0.8, 23, 3),      # 67 sites: three words of 23, 23, 21
    ("potts", "sc/26n", (1024, 2, 2), 50, 0.6, 24, 2),      # 16 words a row
    ("potts", "sc/26n", (720, 2, 2), 50, 0.6, 25, 2),       # 12 words a row, four idle quads
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "%s-%s-%s-q%d" % (c[0], c[1], "x".join(map(str, c[2])), c[3]))
def test_sliced_passes_give_the_oracles_sweeps(orc, tmp_path, case):
    app, lat, shape, q, kt, seed, n = case
    d = orc.make_desc(app, lat, *shape, q, kt)
    spin, seeds = orc.script_init(d, seed, 1, q)
    e0 = orc.energy(d, spin)
    fin, fout = str(tmp_path / "in.bin"), str(tmp_path / "out.bin")
    np.concatenate([spin, seeds]).astype(np.int32).tofile(fin)
    nacc, eng = orc.sweeps(d, spin, seeds, n)
    apps, lats = {"potts": 0, "ising": 1}, {"sq/8n": 1, "sc/26n": 3}
    subprocess.run([EMUL, str(apps[app]), str(lats[lat]), *map(str, shape), str(q), repr(kt), str(n), fin, fout],
                   check=True, timeout=120)
    N = spin.size
    raw = open(fout, "rb").read()
    got = np.frombuffer(raw[:8 * N], np.int32)
    rows = np.frombuffer(raw[8 * N:], np.int64).reshape(n, 2)
    assert np.array_equal(got[:N], spin) and np.array_equal(got[N:], seeds)
    assert np.array_equal(np.cumsum(rows[:, 0]), nacc)
    assert np.array_equal(e0 + 2 * np.cumsum(rows[:, 1]), eng)
