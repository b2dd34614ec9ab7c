"""The per-colour kernels of potts/neigh, potts/neighonly and ising/single
against the oracle on the GPU.  By default lattices as small as these sweep in
boxes; a chosen workgroup keeps them on the kernels that larger ones take, and
the launch count says so."""
import numpy as np
import pytest

from test_gpu_parity import VARIANT_CASES, gpu_init, oracle_run, say

pytestmark = pytest.mark.gpu

COLOURS = {"sq/4n": 2, "sq/8n": 4, "sc/6n": 2, "sc/26n": 8}
MORE = [
    # several workgroups, a last one partly idle, each storage type
    ("potts/neigh", "sq/4n", (150, 66, 1), 300, 0.8, 84, 4),
    ("potts/neighonly", "sc/6n", (26, 18, 10), 70000, 0.5, 85, 4),
    ("potts/neigh", "sq/8n", (106, 94, 1), 200, 0.6, 86, 4),
    ("ising/single", "sq/4n", (130, 98, 1), 2, 2.0, 87, 6),
    ("potts/neigh", "sc/26n", (20, 18, 22), 200, 0.5, 88, 3),       # the packed kernel, as it runs by default
    ("potts/neighonly", "sc/26n", (22, 20, 18), 32768, 0.6, 89, 3),  # one value more than it takes
]


@pytest.mark.parametrize("block", [64, 256, 512])
@pytest.mark.parametrize("case", VARIANT_CASES + MORE, ids=lambda c: "%s-%s-%s" % (c[0], c[1], "x".join(map(str, c[2]))))
def test_variant_kernels_bit_exact(orc, case, block):
    import spparks_amd as S
    app, lat, shape, q, kt, seed, n = case
    say("variant kernel", case, "block", block)
    _, _, spin, seeds, nacc, eng = oracle_run(orc, app, lat, shape, q, kt, seed, n)
    with gpu_init(S, app, lat, shape, q, kt, seed) as L:
        L.set_launch(block)
        L.set_bitplanes(0)
        tot, gn, ge = L.sweeps(n)
        assert L.last_timing()[1] == COLOURS[lat] * n
        s, k = L.download()
    assert np.array_equal(s, spin) and np.array_equal(k, seeds)
    assert np.array_equal(gn, nacc) and np.array_equal(ge, eng) and tot == nacc[-1]
