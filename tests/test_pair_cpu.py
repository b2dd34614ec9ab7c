"""The two-sweep bit-plane kernel's steps in every band and stage (spk_bits.h),
run on the host by tests/emul/spk_emul_pair under AddressSanitizer, against the
oracle: whole and ragged last words, rows that fill a stage and that do not,
bands that end past the lattice, T = 0."""
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
EMUL = os.path.join(HERE, "emul", "spk_emul_pair")

# stage, nx: one word a row, ragged, and rows that fill the stage
ROWS = [(64, 64), (64, 150), (64, 1024), (64, 1022), (128, 1026), (128, 2048), (256, 2050), (256, 4096), (256, 4090)]


@pytest.mark.parametrize("band,ny", [(4, 66), (8, 66), (12, 64), (16, 70)])
@pytest.mark.parametrize("stage,nx", ROWS)
@pytest.mark.parametrize("app,kt", [("ising", 2.269), ("ising/single", 1.9)])
def test_bands_give_the_oracles_sweeps(orc, tmp_path, app, kt, stage, nx, band, ny):
    if nx > 2048 and app == "ising/single" and band != 8:
        pytest.skip("covered by the smaller rows")
    kt = 0.0 if nx == 150 and band == 8 else kt
    d = orc.make_desc(app, "sq/4n", nx, ny, 1, 2, kt)
    spin, seeds = orc.script_init(d, nx + ny + band, 1, 2)
    e0 = orc.energy(d, spin)
    fin, fout = str(tmp_path / "in.bin"), str(tmp_path / "out.bin")
    np.concatenate([spin, seeds]).astype(np.int32).tofile(fin)
    nacc, eng = orc.sweeps(d, spin, seeds, 4)
    subprocess.run([EMUL, {"ising": "1", "ising/single": "4"}[app], str(nx), str(ny), repr(kt), str(band), str(stage),
                    "2", fin, fout], check=True, timeout=120)
    N = spin.size
    raw = open(fout, "rb").read()
    got = np.frombuffer(raw[:8 * N], np.int32)
    rows = np.frombuffer(raw[8 * N:], np.int64).reshape(4, 2)
    assert np.array_equal(got[:N], spin) and np.array_equal(got[N:], seeds)
    assert np.array_equal(np.cumsum(rows[:, 0]), nacc)
    assert np.array_equal(e0 + 2 * np.cumsum(rows[:, 1]), eng)
