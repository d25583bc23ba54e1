"""Captured steps of a tissue that outgrows the grids that it was captured with."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _dividing(A, configs, n, steps):
    """A tissue whose cells all divide in its first step, and their volumes' limit."""
    _, X, Y, Z, info = configs.lattice_tissue(n, 0.2, seed=n)
    p = configs.base_params(2)
    p.voxel_capacity = 64
    p.division_vol = 0.8 * info["v0"]
    p.div_time_steps = steps
    return p, X, Y, Z


@pytest.mark.parametrize("prepared", [False, True])
def test_step_returns_while_the_stream_is_busy(oracle_mesh, prepared):
    """cs3d_step of a tissue that needs wider grids than it was captured with enqueues
    and returns: it waits neither for the steps before it nor for its own."""
    from cellsim3d_amd import abi as A
    from cellsim3d_amd import configs, engine
    print("busy stream, prepared %d" % prepared, flush=True)
    n, big = 150, 8000
    p, X, Y, Z = _dividing(A, configs, n, 1)
    q = configs.single_tissue(big)
    q["params"].voxel_capacity = 64
    with engine.Context(oracle_mesh, capacity_cells=big + 4 * n, voxel_budget=1 << 24, bin_budget=1 << 30) as ctx:
        a = ctx.add_system(q["params"], q["X"], q["Y"], q["Z"], big, max_cells=big, voxels=1 << 14)
        b = ctx.add_system(p, X, Y, Z, n, max_cells=4 * n, voxels=1 << 12)
        a.step(20)
        if prepared:
            ctx.prepare_graph(b)
        b.step(10)  # captured for 150 cells (256 workgroups); 300 after it
        assert b.info()[0] == 2 * n
        a.step(1500)
        t0 = time.perf_counter()
        b.step(20)
        t1 = time.perf_counter()
        ctx.sync()
        t2 = time.perf_counter()
        print("step returned after %.1f ms, the stream was busy for %.1f ms" % (1e3 * (t1 - t0), 1e3 * (t2 - t0)), flush=True)
        assert t2 - t0 > 0.1  # 1500 steps of 8000 cells
        assert t1 - t0 < 0.25 * (t2 - t0)
        assert a.info() == (big, 1520, 0) and b.info() == (2 * n, 30, 0)


# cells at the start; workgroups per CU allowed (0: no call); systems stepped together
@pytest.mark.parametrize("n,cap,both", [(150, 0, False), (403, 0, False), (150, 0, True), (403, 1, True)])
@pytest.mark.parametrize("prepared", [False, True])
def test_growth_past_the_captured_grids(oracle_mesh, n, cap, both, prepared):
    """Every cell divides in the first step, while the host still knows of half of them:
    the grids captured for those stride (one system without a cap), and wider ones take
    over when the host knows.  As without graphs and with a host that looks after each step."""
    from cellsim3d_amd import abi as A
    from cellsim3d_amd import configs, engine
    print("growth: %d cells, cap %d, both %d, prepared %d" % (n, cap, both, prepared), flush=True)
    p, X, Y, Z = _dividing(A, configs, n, 100)
    fields = (A.F_X, A.F_VY, A.F_FCZ, A.F_FDX, A.F_CANDCOUNT)
    got = []
    for eager in (True, False):
        with engine.Context(oracle_mesh, capacity_cells=6 * n, voxel_budget=1 << 22, bin_budget=1 << 28) as ctx:
            if cap:
                ctx.set_launch(cap)
            if eager:
                ctx.set_graph(False)
            systems = [ctx.add_system(p, X, Y, Z, n, max_cells=2 * n + 1, voxels=1 << 13) for _ in range(2 if both else 1)]
            if prepared:
                ctx.prepare_graph(*([] if both else systems))
            for _ in range(40 if eager else 2):
                (ctx if both else systems[0]).step(1 if eager else 20)
                if eager:
                    ctx.sync()
                    for s in systems:
                        s.info()
            ctx.sync()
            assert all(s.info() == (2 * n, 40, 0) for s in systems)
            got.append([[s.get(f)[:2 * n * 192] for f in fields] for s in systems])
    for a, b in zip(*got):
        for f, u, v in zip(fields, a, b):
            assert np.array_equal(u, v), f


def test_eager_steps_widen_their_grids(oracle_mesh):
    """One long call without graphs: its first step doubles the tissue, past the grids of
    its start, and the later ones take grids for what they find.  2000 steps take less than
    1.25 times those of a host that has looked (1.5 times on the grids of the start, 1.1
    with the first of them enqueued before the division is seen), and give the same state."""
    from cellsim3d_amd import abi as A
    from cellsim3d_amd import configs, engine
    print("eager grids", flush=True)
    n, steps = 204, 2000
    p, X, Y, Z = _dividing(A, configs, n, 1)
    p.grid_interval = 10
    took, state = {True: [], False: []}, []
    with engine.Context(oracle_mesh, capacity_cells=8 * n, voxel_budget=1 << 22, bin_budget=1 << 28) as ctx:
        ctx.set_graph(False)
        for rep in range(3):
            for looked in (True, False):
                s = ctx.add_system(p, X, Y, Z, n, max_cells=8 * n, voxels=1 << 14)
                if looked:
                    s.step(1)
                ctx.sync()
                s.info()
                t = time.perf_counter()
                s.step(steps - looked)
                ctx.sync()
                took[looked].append((time.perf_counter() - t) / (steps - looked))
                assert s.info() == (2 * n, steps, 0)
                if rep == 0:
                    state.append([s.get(f) for f in (A.F_X, A.F_VY, A.F_FDZ)])
                s.remove()
    print({k: [round(1e6 * x, 1) for x in v] for k, v in took.items()}, flush=True)
    for a, b in zip(*state):
        assert np.array_equal(a, b)
    assert min(took[False]) < 1.25 * min(took[True])
