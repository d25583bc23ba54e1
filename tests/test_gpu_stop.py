"""A step that a candidate overflow ends, through the C ABI: it ends with the search, for
every cell of the system alike, wherever the search runs."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

STACK = 6  # cells drawn together: 43 candidates of some node within 0.4 (a list holds 40),
           # at most 26 nodes in a search bin (which holds 32)


def _stack(A, configs, s, X, Y, Z):
    """The first cells of system s put into one place beside the tissue, 0.04 apart."""
    from cellsim3d_amd import mesh as M
    base = M.centred(configs.unit_mesh()).astype(np.float32)
    for f, a, step in ((A.F_X, X, 0.03), (A.F_Y, Y, 0.02), (A.F_Z, Z, 0.01)):
        k = (A.F_X, A.F_Y, A.F_Z).index(f)
        v = s.get(f)
        lo = a.min() - 6.0
        for c in range(STACK):
            v[c * 192:c * 192 + 180] = base[:, k] + np.float32(lo + step * c)
        s.set(f, v)


# cells; workgroups per CU allowed (0: no call; 1060 cells take more workgroups than a
# search with the contact pass is allowed, with 4 per CU fewer); a second, sound tissue
@pytest.mark.parametrize("n,both", [(7, False), (12, True), (301, True), (1060, False), (1060, True)])
def test_a_candidate_overflow_ends_the_step_at_its_search(oracle_mesh, n, both):
    from cellsim3d_amd import abi as A
    from cellsim3d_amd import configs, engine
    print("overflow: %d cells, both %d" % (n, both), flush=True)
    _, X, Y, Z, _ = configs.lattice_tissue(n, 0.4, seed=n)
    rng = np.random.default_rng(n)
    V = [rng.normal(0, 0.5, n * 192).astype(np.float32) for _ in range(3)]
    p = configs.base_params(2)
    p.voxel_capacity = 64
    p.pair_skin = 0.1
    p.division_vol = 1e30
    p.add_rands = 1
    kept = (A.F_VX, A.F_VY, A.F_VZ, A.F_FCX, A.F_FCY, A.F_FCZ, A.F_FDX, A.F_FDY, A.F_FDZ, A.F_FRX, A.F_FRY, A.F_FRZ,
            A.F_CMX, A.F_VOLUME)
    ended = []
    for cap in (0, 4):
        with engine.Context(oracle_mesh, capacity_cells=2 * n, voxel_budget=1 << 22, bin_budget=1 << 28) as ctx:
            if cap:
                ctx.set_launch(cap)
            s = ctx.add_system(p, X, Y, Z, n, max_cells=n, voxels=1 << 14, V=V)
            t = ctx.add_system(p, X, Y, Z, n, max_cells=n, voxels=1 << 14, V=V) if both else None
            target = ctx if both else s
            target.step(2)
            ctx.sync()
            assert s.info()[2] == 0
            _stack(A, configs, s, X, Y, Z)
            before = {f: s.get(f) for f in kept}
            x0 = s.get(A.F_X)
            target.step(13)  # a captured ten and three eager steps
            ctx.sync()
            assert s.info() == (n, 2, A.SYS_CAND_OVERFLOW)
            for f in kept:
                assert np.array_equal(s.get(f), before[f]), f
            x1 = s.get(A.F_X)
            moved = (x1 != x0).reshape(n, 192)[:, :180]
            assert moved.any(1).all()  # every cell was moved by the step that ended
            ended.append((x1, s.get(A.F_CANDCOUNT)))
            if both:
                assert t.info() == (n, 15, 0)
                got = [t.get(f) for f in kept]
                s.remove()
                t.remove()
                u = ctx.add_system(p, X, Y, Z, n, max_cells=n, voxels=1 << 14, V=V)
                u.step(15)
                ctx.sync()
                for f, v in zip(kept, got):
                    assert np.array_equal(u.get(f), v), f
    for a, b in zip(*ended):
        assert np.array_equal(a, b)
