"""The library's host side on the CPU: its own sources, built as host code
against a stand-in for the HIP runtime (tests/emul/spk_host.hip) in which
kernels do nothing and every launch and allocation is counted.  What a call
launches, allocates and gives back, and what it does when an allocation
fails."""
import ctypes as C
import os

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
LIB = os.path.join(HERE, "emul", "libspk_host.so")


class Runtime:
    """The stand-in's own calls."""

    def __init__(self, L):
        self.L = L
        for name in ("device_bytes", "device_calls", "pinned_calls", "execs", "captures"):
            f = getattr(L, "spk_host_" + name)
            f.restype = C.c_long
            setattr(self, name, f)
        L.spk_host_log.restype = C.c_char_p
        for name in ("limit", "free_memory"):
            getattr(L, "spk_host_" + name).argtypes = [C.c_size_t]

    def limit(self, more):
        """Device allocations fail beyond `more` bytes from now."""
        self.L.spk_host_limit(self.device_bytes() + more if more is not None else 0)

    def fail_pinned(self, n):
        self.L.spk_host_fail_pinned(n)

    def fail_info(self, n):
        self.L.spk_host_fail_info(n)

    def free_memory(self, n):
        self.L.spk_host_free_memory(n)

    def log(self):
        """(kernel, workgroups, threads) of the launches since the last call."""
        return [(a, int(b), int(c)) for a, b, c in
                (line.rsplit(" ", 2) for line in self.L.spk_host_log().decode().splitlines())]

    def sweeps(self):
        """Names of the sweep kernels launched since the last call."""
        return [n.split("<")[0] for n, _, _ in self.log() if n.startswith(("k_sweep", "k_batch"))]


@pytest.fixture
def host(monkeypatch):
    from spparks_amd import batch, build, hip
    if not os.path.exists(LIB):
        build.build_host_library()
    L = hip.load_library(LIB)
    monkeypatch.setattr(hip, "_lib", L)
    monkeypatch.setattr(batch, "_bound", False)
    r = Runtime(L)
    L.spk_host_reset()
    yield r
    L.spk_host_reset()


def lattice(app="potts", style="sq/8n", shape=(64, 64, 1), q=100, kt=0.5):
    import spparks_amd as S
    return S.Lattice(app, style, *shape, nspins=q, temperature=kt)


@pytest.mark.parametrize("shape", [(64, 64, 1), (256, 256, 1)])
def test_download_without_pinned_memory_takes_the_staging_path(host, shape):
    with lattice(shape=shape) as L:
        host.fail_pinned(1)
        spin, seed = L.download()
        assert spin.size == seed.size == L.n
        L.download()


def state_bytes(L):
    """Bytes of a two-state sq/4n lattice's planes and of their seeds."""
    nx, ny, _ = L.shape
    pw = (nx // 2 + 31) // 32
    return 2 * ny * pw * 4, 2 * ny * pw * 32 * 4


@pytest.mark.parametrize("second", [0.0, 0.5, 1.2])
def test_two_state_lattice_without_second_planes_sweeps_one_colour_a_launch(host, second):
    """Room for the planes and their seeds, and for none, some, or the planes
    and part of the seeds of the second ones."""
    with lattice("ising", "sq/4n", (1000, 1000, 1), 2, 2.269) as L:
        planes, seeds = state_bytes(L)
        host.limit(int(planes * (1 + second) + seeds))
        host.log()
        L.prepare(5)
        L.sweeps(5)
        assert host.sweeps() == ["k_sweep_bits"] * 10 and L.last_timing()[1] == 10
        host.limit(None)
        L.sweeps(4)
        assert host.sweeps() == ["k_sweep_bits"] * 8
    with lattice("ising", "sq/4n", (1000, 1000, 1), 2, 2.269) as L:
        L.sweeps(4)
        assert host.sweeps() == ["k_sweep_bits_pair"] * 2


def test_sliced_lattice_without_its_seeds_keeps_no_planes(host):
    with lattice("potts", "sc/26n", (128, 128, 128), 10000) as L:
        before = host.device_bytes()
        host.limit(128**3 * 5)   # planes of 2 bytes a site fit, 4 of seeds beside them do not
        host.log()
        L.sweeps(2)
        assert host.sweeps() == ["k_sweep_color"] * 16
        assert host.device_bytes() == before


@pytest.mark.parametrize("shape,q,sliced", [
    ((16, 700, 700), 100, False),      # words a quarter full
    ((16, 1000, 1000), 10000, False),
    ((32, 512, 512), 60000, False),    # half full
    ((32, 700, 700), 3000, False),
    ((32, 512, 512), 5, True),
    ((32, 700, 700), 1000000, True),
    ((48, 500, 500), 60000, True),     # three quarters
    ((224, 224, 200), 10000, True),
])
def test_narrow_rows_sweep_on_planes_only_where_that_is_faster(host, shape, q, sliced):
    """A row of up to 16 sites a colour leaves half of its plane words or more
    empty: large lattices of them sweep packed (one launch a colour)."""
    with lattice("potts", "sc/26n", shape, q) as L:
        host.log()
        L.sweeps(1)
        assert host.sweeps() == (["k_sweep_slice"] * 4 if sliced else ["k_sweep_color"] * 8)


@pytest.mark.parametrize("case", [("potts", "sq/8n", (128, 128, 1), 100), ("ising", "sq/4n", (100, 100, 1), 2)],
                         ids=lambda c: "x".join(map(str, c[2])))
def test_boxes_capture_no_graph(host, case):
    """Lattices of one workgroup's size have no graph to capture for each number of
    sweeps and each temperature, as in one workgroup."""
    with lattice(*case) as L:
        captures = host.captures()
        for n in range(2, 40, 7):
            L.set_temperature(0.1 * n)
            L.prepare(n)
            host.log()
            L.sweeps(n)
            assert set(host.sweeps()) == {"k_sweep_tile"}
        assert host.captures() == captures


def test_boxes_take_long_calls_in_pieces(host):
    with lattice("potts", "sq/8n", (600, 500, 1)) as L:
        L.prepare(2)
        L.energy()
        before = host.device_bytes()
        host.log()
        L.sweeps(2500)
        log = [n.split("<")[0] for n, _, _ in host.log()]
        assert log.count("k_zero_u64") == log.count("k_fold_rows") == 3
        assert host.device_bytes() == before
        assert log.count("k_sweep_tile") == L.last_timing()[1] < 2500 and log.count("k_sweep_tile") % 2 == 0


def mixed_queue(n, seed=6):
    rng = np.random.default_rng(seed)
    reqs = []
    for i in range(n):
        e = 2 * int(rng.integers(8, 33))
        style, shape, q = [("sc/26n", (e, e, e), 3000), ("sq/8n", (4 * e, 4 * e, 1), 100),
                           ("sc/26n", (2 * e, e, e), 100)][int(rng.integers(0, 3))]
        reqs.append({"app": "potts", "lattice": style, "shape": shape, "nspins": q, "kT": 0.5, "seed": i + 1,
                     "sweeps": int(rng.integers(3, 60)), "arrive": 0.0})
    return reqs


def test_queue_of_mixed_solves_records_few_graphs(host):
    """A queue whose replicas come and go changes its tile counts, and the sweeps
    each kind has left, with nearly every block: the blocks share graphs."""
    from spparks_amd import batch
    start = host.captures()
    res, st = batch.serve(mixed_queue(300), pool_bytes=4 << 30, max_live=16, block_sweeps=5, block=256, grid=2048)
    assert all(r["status"] == 0 for r in res) and st["blocks"] > 100
    # sweeps of a block are 5 until the queue runs out; of the kinds present (4:
    # planes and packed rows of u8 and u16) the two with most replicas always are, and the
    # grid has four sizes an octave
    assert host.captures() - start <= 40
    assert host.execs() == 0


def test_batch_holds_a_bounded_number_of_graphs(host):
    from spparks_amd import batch
    with batch.Batch(16 << 20, 2) as B:
        B.set_launch(256, 1024)
        B.add(batch.replica_desc("potts", "sq/8n", 64, 64, nspins=100, temperature=0.5, nsweeps=10**6))
        for n in (100, *range(1, 101)):      # (the longest first: its tables serve the others)
            B.run(n)
        assert host.execs() == 64
        start = host.captures()
        for n in range(37, 101):
            B.run(n)
        assert host.captures() == start      # the 64 used last are held
        B.run(36)
        assert host.captures() == start + 1 and host.execs() == 64
    assert host.execs() == 0


def test_batch_takes_replicas_where_free_memory_is_not_known(host):
    from spparks_amd import batch
    with batch.Batch(64 << 20, 2) as B:
        B.set_launch(256, 1024)
        host.fail_info(1)
        assert B.add(batch.replica_desc("potts", "sc/26n", 64, 64, 64, nspins=100, temperature=0.5, nsweeps=3)) == 0
        host.log()
        B.run(3)
        assert "k_batch_slice" not in host.sweeps()
    host.fail_info(2)   # the queue's pool, and the planes of its first solve
    res, _ = batch.serve(mixed_queue(4), pool_bytes=1 << 30, max_live=4, block=256, grid=1024)
    assert all(r["status"] == 0 for r in res)


def test_batch_gives_back_the_memory_of_planes(host):
    """All but one of its chunks of 64 MiB (the first replica that comes again
    finds its planes there), and that one with the batch."""
    from spparks_amd import batch
    base = host.device_bytes()
    desc = batch.replica_desc("potts", "sc/26n", 128, 128, 128, nspins=1000, temperature=0.5, nsweeps=1)
    with batch.Batch(256 << 20, 20) as B:
        B.set_launch(256, 1024)
        empty = host.device_bytes()
        ids = [B.add(desc) for _ in range(16)]      # 12 MiB of planes and seeds each: 5 a chunk
        B.run(1)
        held = host.device_bytes()
        assert held - empty >= 4 * (64 << 20)
        for rid in ids[::2] + ids[1::2]:
            B.remove(rid)
        assert held - host.device_bytes() == 3 * (64 << 20)
        calls = host.device_calls()
        host.log()
        B.add(desc)
        B.run(1)
        assert "k_batch_slice" in host.sweeps() and host.device_calls() == calls
    assert host.device_bytes() == base


def shapes_tried(host):
    """Launch shapes of the batched kernel of packed spins since the last log."""
    return len({(g, b) for n, g, b in host.log() if n.startswith("k_batch_step")})


def test_launch_shape_is_tuned_on_packed_spins(host):
    """A block of replicas on planes only has no shape to choose: the next one with
    packed spins does, in a batch and in a queue."""
    from spparks_amd import batch
    planes = batch.replica_desc("potts", "sc/26n", 64, 64, 64, nspins=100, temperature=0.5, nsweeps=60)
    packed = batch.replica_desc("potts", "sq/8n", 64, 64, nspins=100, temperature=0.5, nsweeps=60)
    with batch.Batch(64 << 20, 4) as B:
        B.run(5)
        assert B.last_timing()["block"] == 0
        B.add(planes)
        host.log()
        B.run(5)
        assert shapes_tried(host) == 0 and B.last_timing()["block"] > 0
        B.add(packed)
        B.run(20)
        assert shapes_tried(host) == 9
        B.run(20)
        assert shapes_tried(host) == 1
        B.set_launch(0, 0)
        B.run(20)
        assert shapes_tried(host) == 9
    reqs = [{"app": "potts", "lattice": l, "shape": s, "nspins": 100, "kT": 0.5, "seed": 1, "sweeps": 100, "arrive": t}
            for l, s, t in (("sc/26n", (64, 64, 64), 0.0), ("sq/8n", (64, 64, 1), 0.0))]
    res, _ = batch.serve(reqs, pool_bytes=batch.replica_bytes("potts", "sc/26n", 64, 64, 64, 100), max_live=4,
                         block_sweeps=20)      # one after the other
    assert all(r["status"] == 0 for r in res) and shapes_tried(host) == 9


@pytest.mark.parametrize("case,single", [
    (("ising", "sq/4n", (692, 580, 1), 2), True),
    (("ising", "sq/4n", (362, 5944, 1), 2), True),
    (("potts", "sc/6n", (16, 128, 196), 255), True),
    (("potts", "sq/8n", (600, 500, 1), 100), False),
    (("potts", "sq/8n", (1174, 4090, 1), 100), True),
    (("potts", "sc/26n", (64, 64, 64), 1000), False),
], ids=lambda v: v[1] + "-" + "x".join(map(str, v[2])) if isinstance(v, tuple) else None)
def test_single_sweep_of_boxes_goes_one_colour_a_launch_where_that_is_faster(host, case, single):
    with lattice(*case) as L:
        k = {"sq/4n": 2, "sc/6n": 2, "sq/8n": 4, "sc/26n": 8}[case[1]]
        L.energy()
        captures = host.captures()
        for n in (1, 2, 3, 1):
            L.prepare(n)
            host.log()
            L.sweeps(n)
            if n == 1 and single:
                assert host.sweeps() == ["k_sweep_color"] * (k * n) and L.last_timing()[1] == k * n
            else:
                assert set(host.sweeps()) == {"k_sweep_tile"}
        assert host.captures() == captures


@pytest.mark.parametrize("app,shape,pairs", [
    ("ising/single", (44, 4748, 1), False),     # bands in rounds on the compute units
    ("ising/single", (834, 8680, 1), False),
    ("ising/single", (558, 9782, 1), False),
    ("ising/single", (1580, 5552, 1), True),
    ("ising", (1404, 7722, 1), True),
    ("ising", (4096, 4096, 1), True),
])
def test_two_sweeps_a_launch_where_that_is_faster(host, app, shape, pairs):
    with lattice(app, "sq/4n", shape, 2, 2.269) as L:
        host.log()
        L.sweeps(4)
        names = set(host.sweeps())
        assert pairs == ("k_sweep_bits_pair" in names), names


@pytest.mark.parametrize("case,boxes", [
    # sites a thread against packs, and boxes against one colour a launch
    (("ising", "sc/6n", (178, 18, 128), 2), False),
    (("potts", "sc/6n", (138, 16, 132), 100), False),
    (("ising/single", "sq/4n", (6776, 346, 1), 2), False),
    (("ising", "sc/6n", (16, 104, 154), 2), True),
    (("potts", "sq/8n", (128, 128, 1), 100), True),
    (("potts", "sc/26n", (64, 64, 64), 100000), True),
], ids=lambda v: v[1] + "-" + "x".join(map(str, v[2])) if isinstance(v, tuple) else None)
def test_boxes_where_they_are_faster(host, case, boxes):
    with lattice(*case) as L:
        host.log()
        L.sweeps(24)
        assert boxes == ("k_sweep_tile" in host.sweeps())


def test_calls_of_two_launches_capture_no_graph(host):
    with lattice("potts", "sc/6n", (150, 130, 110), 50) as L:
        captures = host.captures()
        for _ in range(3):
            L.prepare(1)
            host.log()
            L.sweeps(1)
            assert host.sweeps() == ["k_sweep_color"] * 2
        assert host.captures() == captures
        L.sweeps(2)
        assert host.captures() == captures + 1


def test_long_calls_of_first_appearance_boxes_are_replayed(host):
    with lattice("potts/neighonly", "sc/26n", (92, 32, 44), 656669) as L:
        captures = host.captures()
        L.sweeps(3)
        L.set_temperature(0.4)
        L.sweeps(3)
        assert host.captures() == captures and "k_sweep_tile" in host.sweeps()
        L.prepare(24)
        assert host.captures() == captures + 1
        host.log()
        L.sweeps(24)
        assert host.captures() == captures + 1
        assert host.sweeps() == ["k_sweep_tile"] * L.last_timing()[1]


def test_few_replicas_on_planes_take_no_more_workgroups_than_they_need(host):
    """An ensemble of constant shape; the grid grows in steps only once it has
    changed."""
    from spparks_amd import batch
    with batch.Batch(64 << 20, 4) as B:
        B.set_launch(256, 1024)
        B.add(batch.replica_desc("potts", "sc/26n", 64, 64, 64, nspins=100, temperature=0.5, nsweeps=60))
        host.log()
        B.run(10)
        grids = {g for n, g, _ in host.log() if n.startswith("k_batch_slice")}
        assert len(grids) == 1 and 16 <= grids.pop() <= 24      # 1024 rows, 16 a wavefront, 4 wavefronts


def test_kind_of_few_sweeps_takes_few_steps(host):
    """Beside a replica of another kind with many."""
    from spparks_amd import batch
    with batch.Batch(64 << 20, 4) as B:
        B.set_launch(256, 1024)
        B.add(batch.replica_desc("potts", "sc/26n", 64, 64, 64, nspins=100, temperature=0.5, nsweeps=10))
        B.add(batch.replica_desc("ising", "sq/4n", 64, 64, nsweeps=100, temperature=2.0))
        host.log()
        B.run(100)
        names = host.sweeps()
        assert names.count("k_batch_step") == 2 * 100 and names.count("k_batch_slice") <= 4 * 20
