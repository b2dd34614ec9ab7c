"""sc/26n lattices of narrow rows against the oracle on the GPU, on each side of
the line between bit planes (4 launches a sweep) and the packed kernel (8)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,q,launches", [
    ((32, 512, 512), 100, 4),      # words half full
    ((32, 512, 512), 60000, 8),
    ((16, 700, 700), 100, 8),      # a quarter
], ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_narrow_rows_equal_oracle(orc, shape, q, launches):
    import spparks_amd as S
    print("narrow", shape, q, flush=True)
    d = orc.make_desc("potts", "sc/26n", *shape, q, 0.5)
    spin, seeds = orc.script_init(d, 91, 1, q)
    with S.Lattice("potts", "sc/26n", *shape, nspins=q, temperature=0.5) as L:
        s0, rseed = S.strict_init_params(91)
        L.set_range(s0, 1, q)
        L.init_seeds(rseed)
        nacc, eng = orc.sweeps(d, spin, seeds, 2)
        _, gn, ge = L.sweeps(2)
        assert L.last_timing()[1] == 2 * launches
        assert np.array_equal(gn, nacc) and np.array_equal(ge, eng)
        s, k = L.download()
        assert np.array_equal(s, spin) and np.array_equal(k, seeds)
