"""Batched replicas that sweep on bit planes (k_batch_slice) against the
oracle on the GPU, beside replicas on packed spins: one to five plane groups,
words of 32 sites and of fewer, rows of one word and of several, wavefronts
partly idle, T = 0, two states; eager, graph and tuned blocks, replicas that end
in different blocks, uploads of one array, and an extent used again."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MIX = [
    # app, lattice, shape, Q, kT, seed, sweeps
    ("potts", "sc/26n", (64, 8, 8), 10000, 0.5, 201, 7),
    ("potts", "sc/26n", (32, 16, 8), 16, 0.9, 202, 5),       # one plane group, half of each word
    ("potts", "sc/26n", (78, 10, 6), 200, 0.6, 203, 6),      # words of 20 and 19, 15 rows of 8 a wavefront
    ("potts", "sc/26n", (190, 6, 6), 1000000, 0.3, 204, 4),  # three words of 32, 32, 31: idle quads; five groups
    ("potts", "sc/26n", (1022, 2, 4), 3000, 0.5, 205, 3),    # 16 words a row
    ("potts", "sc/26n", (40, 40, 40), 65536, 0.0, 206, 5),   # T = 0; 25 wavefronts a pass
    ("ising", "sc/26n", (64, 16, 4), 2, 3.0, 207, 4),
    ("potts", "sc/26n", (10, 6, 4), 3000, 0.5, 208, 4),      # on packed spins from here on
    ("potts", "sq/8n", (22, 6, 1), 9, 0.9, 209, 5),
    ("ising", "sq/4n", (64, 48, 1), 2, 2.269, 210, 9),
]


def start(orc, case):
    app, lat, shape, q, kt, seed, _ = case
    d = orc.make_desc(app, lat, *shape, q, kt)
    return (d, *orc.script_init(d, seed, 1, q))


def add(B, case):
    from spparks_amd import batch as bmod
    app, lat, shape, q, kt, seed, n = case
    return B.add(bmod.replica_desc(app, lat, *shape, nspins=q, temperature=kt, seed=seed, nsweeps=n))


@pytest.mark.parametrize("mode", ["eager", "graph", "autotune"])
def test_batch_with_sliced_replicas_equals_oracle(orc, mode):
    from spparks_amd import batch as bmod, hip
    print("sliced batch", mode, flush=True)
    with bmod.Batch(16 << 20, 16) as B:
        ids = [add(B, c) for c in MIX]
        if mode != "autotune":
            B.set_launch(64, 16)
        for k in range(4):
            B.run(3, graph=mode == "graph")
            if k == 0:   # 4 passes a sweep on planes; sc/26n 8, sq/8n 4, sq/4n 2 on packed spins
                assert B.last_timing()["launches"] == 3 * (4 + 8 + 4 + 2)
            if k == 1:
                B.download(ids[2])
        for rid, case in zip(ids, MIX):
            d, spin, seeds = start(orc, case)
            e0 = orc.energy(d, spin)
            nacc, eng = orc.sweeps(d, spin, seeds, case[6])
            gn, ge = B.trace(rid, case[6])
            assert np.array_equal(gn, nacc) and np.array_equal(ge, eng), (case, e0)
            assert B.checksum(rid) == hip.checksum(spin, seeds), case
            gs, gk = B.download(rid)
            assert np.array_equal(gs, spin) and np.array_equal(gk, seeds), case


def test_sliced_replica_takes_uploads_and_an_extent_again(orc):
    from spparks_amd import batch as bmod, hip
    case = MIX[2][:6] + (20,)
    with bmod.Batch(bmod.replica_bytes("potts", "sc/26n", 78, 10, 6, 200), 2) as B:
        other = add(B, case[:5] + (99, 3))
        B.set_launch(128, 8)
        B.run(3)
        B.remove(other)
        rid = add(B, case)
        d, spin, seeds = start(orc, case)
        B.run(2)
        orc.sweeps(d, spin, seeds, 2)
        _, fresh, _ = start(orc, case[:5] + (5, 1))
        B.upload(rid, spin=fresh)        # the seeds go on
        spin = fresh.copy()
        B.run(2)
        orc.sweeps(d, spin, seeds, 2)
        assert B.checksum(rid) == hip.checksum(spin, seeds)
        _, _, seeds = start(orc, case[:5] + (6, 1))
        B.upload(rid, seed=seeds)        # the spins go on
        B.run(3)
        orc.sweeps(d, spin, seeds, 3)
        s, k = B.download(rid)
        assert np.array_equal(s, spin) and np.array_equal(k, seeds)
        assert B.status(rid)[3] == orc.energy(d, spin)


def test_queue_takes_no_more_than_its_solves_and_refuses_what_the_device_lacks():
    import spparks_amd as S
    from spparks_amd import batch as bmod
    reqs = [{"app": a, "lattice": l, "shape": s, "nspins": q, "kT": k, "seed": sd, "sweeps": n, "arrive": 0.0}
            for a, l, s, q, k, sd, n in MIX[:4]]
    small, _ = bmod.serve(reqs, pool_bytes=sum(bmod.replica_bytes(c[0], c[1], *c[2], c[3]) for c in MIX[:4]), max_live=4)
    large, st = bmod.serve(reqs, pool_bytes=1 << 30, max_live=4)
    assert st["max_live"] == 4
    for a, b in zip(small, large):
        assert a["status"] == b["status"] == 0 and a["checksum"] == b["checksum"] and a["energy"] == b["energy"]
    with pytest.raises(S.HipError, match="not available"):
        bmod.serve(reqs, pool_bytes=1 << 44, max_live=4)
