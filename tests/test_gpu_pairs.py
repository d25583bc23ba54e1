"""Paths whose form depends on sizes, through the C ABI.

The contact pass of k_con_dis where its work lists can go wrong, bit for bit
against the oracle: no candidates at all, one round (at most 192
pairs per cell), several rounds, nodes whose candidates straddle a round or a
64-lane word, and lists near the 40-entry limit; and the bonds and angles at the
edges of the short arithmetic (rest shape, crushed, stretched, bonds at and below
its range); the division phase's flag test; reads of device memory; batches past one
scan of the live list; grids smaller than their tissue; the search with the contact
pass or in its own launch."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _run(oracle_mesh, X, Y, Z, n, skin, steps, seed, grow=0.0):
    from cellsim3d_amd import abi as A
    from cellsim3d_amd import configs, engine
    from oracle import oracle as O
    p = configs.base_params(seed)
    p.growth_rate = grow
    p.division_vol = 1e30
    p.pair_skin = skin
    p.voxel_capacity = 64
    rng = np.random.default_rng(seed)
    V = [np.zeros((n, 192), np.float32) for _ in range(3)]
    for v in V:
        v[:, :180] = rng.normal(0, 0.3, (n, 180)).astype(np.float32)
    V = [v.reshape(-1) for v in V]
    sim = O.Sim(p, oracle_mesh, X, Y, Z, n, max_cells=n, budget=1 << 14)
    for f, v in zip((A.F_VX, A.F_VY, A.F_VZ), V):
        sim.set(f, v)
    sim.init()
    with engine.Context(oracle_mesh, capacity_cells=n, voxel_budget=1 << 21) as ctx:
        s = ctx.add_system(p, X, Y, Z, n, max_cells=n, voxels=1 << 14, V=V)
        counts = s.get(A.F_CANDCOUNT).reshape(n, 192)
        assert not counts[:, 180:].any()
        fields = [A.F_FCX, A.F_FCY, A.F_FCZ, A.F_FDX, A.F_FDY, A.F_FDZ, A.F_X, A.F_Y, A.F_Z, A.F_VX, A.F_VY, A.F_VZ]
        for k in range(2):
            for f in fields:
                a, b = s.get(f)[:n * 192], sim.get(f)[:n * 192]
                assert np.array_equal(a, b, equal_nan=True), (k, f, int((a != b).sum()))
            if k == 0:
                # the partner lists: ascending keys of nodes within attraction_range
                pc = s.get(A.F_PAIRCOUNT).reshape(n, 192)
                keys = s.get(A.F_PAIRS).reshape(n, 40, 192)
                P = np.stack([a.reshape(-1) for a in (X, Y, Z)]).astype(np.float64)
                for c in range(n):
                    for i in np.flatnonzero(pc[c]):
                        g = keys[c, :pc[c, i], i]
                        assert np.all(np.diff(g) > 0)
                        d = np.sqrt(((P[:, g] - P[:, c * 192 + i][:, None]) ** 2).sum(0))
                        assert np.all(d < p.attraction_range + 1e-5)
                sim.step(steps)
                s.step(steps)
                ctx.sync()
        status = s.info()[2]
    return counts, status


# spacing in x, cells, skin -> rounds of 192 pairs in the fullest cell
@pytest.mark.parametrize("spacing,n,skin,rounds", [(4.0, 3, 0.05, (0, 0)), (2.1, 2, 0.05, (1, 1)), (1.9, 5, 0.15, (2, 4)),
                                                   (1.8, 7, 0.2, (4, 9)), (1.75, 9, 0.22, (6, 38))])
def test_pair_rounds_match_oracle(oracle_mesh, spacing, n, skin, rounds):
    from cellsim3d_amd import abi as A
    from cellsim3d_amd import configs
    print("pairs: spacing %g, %d cells, skin %g" % (spacing, n, skin), flush=True)
    centres = [(spacing * (i % 3), spacing * (i // 3), 0.3 * (i % 2)) for i in range(n)]
    X, Y, Z = configs.place(configs.unit_mesh(), centres, 0.02, np.random.default_rng(n))
    counts, status = _run(oracle_mesh, X, Y, Z, n, skin, 4, 3 + n)
    assert not status & A.SYS_FATAL_MASK
    full = -(-int(counts.sum(1).max()) // 192)
    assert rounds[0] <= full <= rounds[1], full


# a cell scaled per axis, then some nodes drawn to their first neighbour, to the given
# distance (0: the shape as it is).  (Scaling a whole cell far down would put its 180
# nodes into one search bin of 32 entries, which the engine refuses.)
@pytest.mark.parametrize("scale,bond", [((1.0, 1.0, 1.0), 0.0), ((1.0, 1.0, 0.02), 0.0), ((1.0, 0.3, 3.0), 0.0),
                                        ((1.0, 1.0, 1.0), 2e-3), ((1.0, 1.0, 1.0), 1e-4), ((1.0, 1.0, 1.0), 1e-6)])
def test_deformed_cells_match_oracle(oracle_mesh, scale, bond):
    from cellsim3d_amd import configs, mesh as M
    print("bonds and angles: scale %s, bond %g" % (scale, bond), flush=True)
    m = configs.unit_mesh()
    base = M.centred(m).astype(np.float32)
    A = [np.zeros((2, 192), np.float32) for _ in range(3)]
    for k in range(3):
        A[k][0, :180] = base[:, k] * np.float32(scale[k])
        A[k][1, :180] = base[:, k] + np.float32(5.0 if k == 0 else 0.0)
        if bond:
            for i in range(0, 180, 20):
                A[k][0, i] = A[k][0, m["nn"][i, 0]] + np.float32(bond)
    # one step: the strongly deformed ones move far, and both sides with them
    _run(oracle_mesh, A[0].reshape(-1), A[1].reshape(-1), A[2].reshape(-1), 2, 0.05, 1, 7)


# the flag test of the division phase reads 16 flags at a time between 16-byte
# boundaries: rooms that start at any of them, counts around them, and flag values
# other than 1, which are no event (d_cell_div, GPUbounce.cu:2489-2500)
@pytest.mark.parametrize("offset", [0, 1, 7, 15])
@pytest.mark.parametrize("n", [1, 15, 16, 17, 33, 70])
def test_every_flagged_cell_divides(oracle_mesh, n, offset):
    from cellsim3d_amd import abi as A
    from cellsim3d_amd import configs, engine
    print("flags: %d cells from slot %d" % (n, offset), flush=True)
    _, X, Y, Z, _ = configs.lattice_tissue(n, 0.2, seed=n)
    p = configs.base_params(2)
    p.voxel_capacity = 64
    with engine.Context(oracle_mesh, capacity_cells=offset + 2 * n, voxel_budget=1 << 21, bin_budget=1 << 23) as ctx:
        if offset:
            ctx.add_system_raw(p, 0, max_cells=offset, voxels=1)
        for cells in ([], [0], [n - 1], [n // 2], sorted({0, n // 3, n - 1})):
            s = ctx.add_system(p, X, Y, Z, n, max_cells=2 * n, voxels=1 << 12)
            flags = np.zeros(2 * n, np.int8)
            flags[:n:2] = 2
            flags[1:n:2] = -1
            flags[n:] = 1  # past the live cells
            for c in cells:
                flags[c] = 1
            s.set(A.F_DIVFLAG, flags)
            assert s.k_divide() == len(cells)
            assert s.info()[0] == n + len(cells)
            moved = np.flatnonzero((s.get(A.F_X)[:n * 192].reshape(n, 192) != X.reshape(n, 192)).any(1))
            assert moved.tolist() == cells
            s.remove()


# reads below, between and above the sizes where the way back changes (one piece of
# 16 KB and 1 MB, 64 KB together, the 2 MB slots and the ring of four), odd lengths
# among them
@pytest.mark.parametrize("n", [1, 3, 13, 14, 21, 22, 70, 73, 76, 700, 1400, 3001])
def test_reads_return_what_was_written(oracle_mesh, n):
    from cellsim3d_amd import abi as A
    from cellsim3d_amd import configs, engine
    print("reads of %d cells" % n, flush=True)
    L = engine.lib()
    p = configs.base_params(2)
    rng = np.random.default_rng(n)
    with engine.Context(oracle_mesh, capacity_cells=n + 3, voxel_budget=1 << 20, bin_budget=1 << 23) as ctx:
        ctx.add_system_raw(p, 0, max_cells=2, voxels=1)
        s = ctx.add_system_raw(p, n, max_cells=n + 1, voxels=16)
        want = {}
        for f in (A.F_X, A.F_Y, A.F_Z, A.F_VX, A.F_VY, A.F_VZ):
            want[f] = rng.random((n + 1) * 192).astype(np.float32)
            s.set(f, want[f])
        for f in (A.F_PRESSURE, A.F_CMX, A.F_CMY, A.F_CMZ, A.F_VOLUME):
            want[f] = rng.random(n + 1).astype(np.float32)
            s.set(f, want[f])
        flags = rng.integers(-3, 3, n + 1).astype(np.int8)
        s.set(A.F_DIVFLAG, flags)
        for f, w in want.items():
            assert np.array_equal(s.get(f), w), f
        assert np.array_equal(s.get(A.F_DIVFLAG), flags)
        for nb in (1, 4, 7, 4 * (n * 96 + 1)):  # parts of a field
            part = np.full(4 * (n + 1) * 192, 77, np.uint8)
            engine.check(L.cs3d_get(ctx.h, s.id, A.F_Y, part.ctypes.data, nb), "cs3d_get")
            assert np.array_equal(part[:nb], want[A.F_Y].view(np.uint8)[:nb]) and np.all(part[nb:] == 77)
        st = s.get_state()
        assert st["n"] == n and st["status"] == 0
        for k, f in enumerate((A.F_X, A.F_Y, A.F_Z)):
            assert np.array_equal(st["xyz"][k], want[f][:n * 192])
        for k, f in enumerate((A.F_VX, A.F_VY, A.F_VZ)):
            assert np.array_equal(st["v"][k], want[f][:n * 192])
        for k, f in enumerate((A.F_CMX, A.F_CMY, A.F_CMZ)):
            assert np.array_equal(st["CM"][k], want[f][:n])
        assert np.array_equal(st["P"], want[A.F_PRESSURE][:n]) and np.array_equal(st["V"], want[A.F_VOLUME][:n])
        # without some of the outputs
        P = np.zeros(n, np.float32)
        engine.check(L.cs3d_get_state(ctx.h, s.id, None, None, P.ctypes.data, None, None, None, None), "cs3d_get_state")
        assert np.array_equal(P, want[A.F_PRESSURE][:n])


def test_more_systems_than_one_scan_of_the_live_list(oracle_mesh):
    """1030 systems in one batch (the live list scans 1024 at a time) of 0 to 3 cells, some
    stopped at a horizon and some removed: each ends where it ends alone."""
    from cellsim3d_amd import abi as A
    from cellsim3d_amd import configs, engine
    print("1030 systems", flush=True)
    kinds = []
    for n in range(4):
        p = configs.base_params(3 + n)
        p.grid_interval = 2
        p.division_vol = 1e30  # (the default is the reference mesh's, below this mesh's rest volume)
        X, Y, Z = configs.place(configs.unit_mesh(), [(2.1 * i, 0.1 * i, 0) for i in range(n)], 0.02,
                                np.random.default_rng(n)) if n else (np.zeros(0, np.float32),) * 3
        kinds.append((p, X, Y, Z, n))
    nsys = 1030
    with engine.Context(oracle_mesh, capacity_cells=4 * nsys, voxel_budget=nsys * 33 * 64,
                        bin_budget=nsys * (16384 * A.BIN_WORDS + 16)) as ctx:
        alone = {}
        for n, k in enumerate(kinds):
            for steps in (3, 12):
                s = ctx.add_system(*k, max_cells=max(n, 1), voxels=32)
                s.step(steps)
                ctx.sync()
                alone[n, steps] = [s.get(f)[:n * 192] for f in (A.F_X, A.F_VZ, A.F_FDY)]
                s.remove()
        systems = []
        for i in range(nsys):
            n = (i * 7 + i // 5) % 4
            s = ctx.add_system(*kinds[n], max_cells=max(n, 1), voxels=32)
            if i % 11 == 3:
                s.set_horizon(3)
            systems.append((i, n, s))
        for i, n, s in systems:
            if i % 50 == 7:
                s.remove()
        ctx.step(12)  # a captured ten and two eager steps
        ctx.sync()
        cells, steps, status = ctx.poll(0, nsys)
        for i, n, s in systems:
            if i % 50 == 7:
                assert cells[s.id] == -1
                continue
            k = 3 if i % 11 == 3 else 12
            assert (cells[s.id], steps[s.id], status[s.id]) == (n, k, 0), i
            if i < 40 or i > 1015 or i % 37 == 0:
                for f, want in zip((A.F_X, A.F_VZ, A.F_FDY), alone[n, k]):
                    assert np.array_equal(s.get(f)[:n * 192], want), (i, f)


# cells, workgroups per CU that the caller allows (0: no call), systems stepped together
@pytest.mark.parametrize("n,cap,both", [(1, 0, False), (9, 0, False), (70, 0, False), (70, 0, True), (150, 0, True), (300, 1, True)])
def test_grids_smaller_than_the_tissue(oracle_mesh, n, cap, both):
    """Every cell divides in the first step, while the host still knows of half of them:
    the grids of the following steps cover a part and stride, and the graph captured
    with them gives way to a wider one at 300.  As with a host that looks after each step."""
    from cellsim3d_amd import abi as A
    from cellsim3d_amd import configs, engine
    print("grids: %d cells, cap %d, both %d" % (n, cap, both), flush=True)
    _, X, Y, Z, _ = configs.lattice_tissue(n, 0.2, seed=n)
    p = configs.base_params(2)
    p.voxel_capacity = 64
    p.division_vol = 0.8 * configs.mesh_volume(configs.unit_mesh())  # the cells are above it, their daughters below
    p.div_time_steps = 100
    fields = (A.F_X, A.F_VY, A.F_FCZ, A.F_FDX, A.F_VOLUME, A.F_CANDCOUNT)
    got = []
    for look in (True, False):
        with engine.Context(oracle_mesh, capacity_cells=6 * n + 2, voxel_budget=1 << 21, bin_budget=1 << 26) as ctx:
            if cap:
                ctx.set_launch(cap)
            systems = [ctx.add_system(p, X, Y, Z, n, max_cells=2 * n + 1, voxels=1 << 12) for _ in range(2 if both else 1)]
            for _ in range(24 if look else 2):
                (ctx if both else systems[0]).step(1 if look else 12)
                for s in systems:
                    s.info()
            ctx.sync()
            assert all(s.info()[0] == 2 * n for s in systems)
            got.append([[s.get(f) for f in fields] for s in systems])
    for a, b in zip(*got):
        for f, u, v in zip(fields, a, b):
            k = 2 * n * (1 if f == A.F_VOLUME else 192)
            assert np.array_equal(u[:k], v[:k], equal_nan=True), f


@pytest.mark.parametrize("both", [False, True])
def test_search_in_its_own_launch_or_with_the_contacts(oracle_mesh, both):
    """1060 cells take more workgroups than a search with the contact pass is allowed, a cap
    of 4 per CU fewer: the same states, through full and partial searches and divisions."""
    from cellsim3d_amd import abi as A
    from cellsim3d_amd import configs, engine
    n = 1060
    print("search place, both %d" % both, flush=True)
    _, X, Y, Z, info = configs.lattice_tissue(n, 0.5, seed=9)
    rng = np.random.default_rng(9)
    V = [rng.normal(0, 1.0, n * 192).astype(np.float32) for _ in range(3)]
    p = configs.base_params(2)
    p.voxel_capacity = 64
    p.pair_skin = 0.02
    p.division_vol = np.float32(1.0005 * info["v0"])
    p.div_time_steps = 1000
    fields = (A.F_X, A.F_VY, A.F_FCZ, A.F_FDX, A.F_CANDCOUNT)
    got = []
    for cap in (0, 4):
        with engine.Context(oracle_mesh, capacity_cells=5 * n, voxel_budget=1 << 22, bin_budget=1 << 29) as ctx:
            if cap:
                ctx.set_launch(cap)
            systems = [ctx.add_system(p, X, Y, Z, n, max_cells=2 * n, voxels=1 << 14, V=V) for _ in range(2 if both else 1)]
            for _ in range(4):
                (ctx if both else systems[0]).step(13)
                ctx.sync()
                got.append([(s.info()[0], s.info()[2], [s.get(f) for f in fields]) for s in systems])
    assert got[3][0][0] > n
    for a, b in zip(got[:4], got[4:]):
        for (na, sa, fa), (nb, sb, fb) in zip(a, b):
            assert (na, sa) == (nb, sb)
            for f, u, v in zip(fields, fa, fb):
                assert np.array_equal(u[:na * 192], v[:na * 192], equal_nan=True), f
