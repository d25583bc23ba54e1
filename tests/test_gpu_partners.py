"""The partner lists (CS3D_F_PAIRS, CS3D_F_PAIRCOUNT), which are made when they are read:
equal, entry for entry, to the reference's rule evaluated on the host, wherever the
contact pass that they belong to came from, and whatever happened to the candidates
since."""
import numpy as np
import pytest
from scipy.spatial import cKDTree

pytestmark = pytest.mark.gpu


def _rule(p, X, box, grid, n):
    """(node, key) of every accepted pair, sorted: distance, voxel list and bbox tests of
    propagate.cu:360-421 and the voxel range of propagatebound.cu:224-245 in float32."""
    f = np.float32
    P = [a.reshape(-1, 192)[:n, :180].reshape(-1).astype(f) for a in X]
    own = np.repeat(np.arange(n), 180)
    ar = f(p.attraction_range)
    q = cKDTree(np.stack(P, 1).astype(np.float64)).query_pairs(float(ar) * 1.001, output_type="ndarray")
    q = np.concatenate([q, q[:, ::-1]])
    i, j = q[own[q[:, 0]] != own[q[:, 1]]].T
    d = [a[i] - a[j] for a in P]
    ok = ~(d[0] * d[0] + d[1] * d[1] + d[2] * d[2] > ar * ar)
    g, dims, DL = grid[:3].view(f), grid[3:6], f(p.grid_dl)
    box = box.reshape(-1, 6)[:n].astype(f)
    far = np.zeros(i.size, f)
    for a in range(3):
        v = np.clip(((P[a] - g[a]) / DL).astype(np.int32), 0, dims[a] - 1)
        lo = np.maximum(((box[:, 2 * a] - ar - g[a]) / DL).astype(np.int32), 0)
        hi = np.minimum(((box[:, 2 * a + 1] + ar - g[a]) / DL).astype(np.int32), dims[a] - 1)
        b = own[j]
        ok &= (lo[b] <= v[i]) & (v[i] <= hi[b])
        x, b0, b1 = P[a][i], box[b, 2 * a], box[b, 2 * a + 1]
        t = (x - b1 > 0).astype(f) * (x - b1)
        t = t + (b0 - x > 0).astype(f) * (b0 - x)
        far = far + t * t
    ok &= ~(far > ar * ar)
    i, j = i[ok], j[ok]
    node, key = own[i] * 192 + i % 180, own[j] * 192 + j % 180
    o = np.lexsort((key, node))
    return np.stack([node[o], key[o]], 1)


def _lists(A, s, n):
    """(node, key) of the system's lists, in their own order."""
    pc = s.get(A.F_PAIRCOUNT).reshape(-1, 192)[:n]
    keys = s.get(A.F_PAIRS).reshape(-1, 40, 192)[:n]
    assert not pc[:, 180:].any() and pc.min() >= 0 and pc.max() <= 40
    c, i = np.nonzero(pc)
    return np.array([(a * 192 + b, k) for a, b in zip(c, i) for k in keys[a, :pc[a, b], b]], np.int64).reshape(-1, 2)


def _rules_state(A, s):
    return s.get(A.F_BBOX), s.get(A.F_GRID).view(np.int32)  # completes a pending grid, as the next step does


def _xyz(A, s):
    return [s.get(f) for f in (A.F_X, A.F_Y, A.F_Z)]


def _tissue(A, configs, engine, oracle_mesh, n, skin=0.05, cap=0, speed=0.5, large=(), **over):
    _, X, Y, Z, info = configs.lattice_tissue(n, 0.5, seed=n)
    for x in (X, Y, Z):
        for c in large:  # 1.16 times the volume
            v = x[c * 192:c * 192 + 180]
            v[:] = v.mean() + np.float32(1.05) * (v - v.mean())
    rng = np.random.default_rng(n)
    V = [rng.normal(0, speed, n * 192).astype(np.float32) for _ in range(3)]
    p = configs.base_params(2)
    p.voxel_capacity = 64
    p.pair_skin = skin
    p.division_vol = 1e30
    for k, v in over.items():
        setattr(p, k, v(info) if callable(v) else v)
    ctx = engine.Context(oracle_mesh, capacity_cells=6 * n, voxel_budget=1 << 24, bin_budget=1 << 29)
    if cap:
        ctx.set_launch(cap)
    return ctx, ctx.add_system(p, X, Y, Z, n, max_cells=2 * n, voxels=1 << 14, V=V), p


# 1060 cells: the search in its own launch, with 4 workgroups per CU with the contacts
@pytest.mark.parametrize("n,cap,grid", [(2, 0, 1), (13, 0, 1), (64, 0, 10), (301, 0, 1), (1060, 0, 10), (1060, 4, 10)])
def test_lists_follow_the_latest_contact_pass(oracle_mesh, n, cap, grid):
    from cellsim3d_amd import abi as A
    from cellsim3d_amd import configs, engine
    print("partners: %d cells, cap %d" % (n, cap), flush=True)
    ctx, s, p = _tissue(A, configs, engine, oracle_mesh, n, cap=cap, grid_interval=grid, speed=2.0)
    with ctx:
        want = _rule(p, _xyz(A, s), *_rules_state(A, s), n)
        assert want.shape[0] > 0
        assert np.array_equal(_lists(A, s, n), want)
        for steps in (1, 1, 11, 4):
            s.step(steps)
            ctx.sync()
            rules = _rules_state(A, s)
            s.step(1)
            ctx.sync()
            want = _rule(p, _xyz(A, s), *rules, n)
            assert np.array_equal(_lists(A, s, n), want), steps
            assert np.array_equal(_lists(A, s, n), want)  # read again
        # a search for its own sake replaces the candidates, not the lists
        s.time_kernel(2, 2)
        assert np.array_equal(_lists(A, s, n), want)
        # a larger room
        s.grow(3 * n)
        assert np.array_equal(_lists(A, s, n), want)
        # a given state: positions written by the caller, friction alone, then all forces
        rules = _rules_state(A, s)
        moved = [x + np.float32(0.02) * np.random.default_rng(5 + k).standard_normal(x.size).astype(np.float32)
                 for k, x in enumerate(_xyz(A, s))]
        for f, x in zip((A.F_X, A.F_Y, A.F_Z), moved):
            s.set(f, x)
        assert np.array_equal(_lists(A, s, n), want)
        s.k_dis_force(0)
        want = _rule(p, moved, *rules, n)
        assert np.array_equal(_lists(A, s, n), want)
        s.set(A.F_X, moved[0] + np.float32(0.01) * np.sin(np.arange(moved[0].size)).astype(np.float32))
        s.k_con_force()
        assert np.array_equal(_lists(A, s, n), _rule(p, _xyz(A, s), *rules, n))
        assert s.info()[2] == 0


@pytest.mark.parametrize("n,cap", [(24, 0), (700, 0), (1060, 0), (1060, 4)])
def test_lists_after_divisions(oracle_mesh, n, cap):
    """Three cells divide in the first step; the second searches near them only."""
    from cellsim3d_amd import abi as A
    from cellsim3d_amd import configs, engine
    print("partners after divisions: %d cells, cap %d" % (n, cap), flush=True)
    ctx, s, p = _tissue(A, configs, engine, oracle_mesh, n, cap=cap, speed=0.0, large=(1, n // 2, n - 1),
                        division_vol=lambda info: np.float32(1.08 * info["v0"]), div_time_steps=1)
    with ctx:
        s.step(1)
        ctx.sync()
        m = n + 3
        assert s.info()[0] == m
        for _ in range(3):
            rules = _rules_state(A, s)
            s.step(1)
            ctx.sync()
            want = _rule(p, _xyz(A, s), *rules, m)
            assert np.array_equal(_lists(A, s, m), want)
        assert s.info() == (m, 4, 0) and (want[:, 0] >= n * 192).any()


# read before the step that ends at its search, or only after it
@pytest.mark.parametrize("n,cap,before", [(12, 0, True), (12, 0, False), (1060, 0, False), (1060, 4, False)])
def test_lists_outlive_a_search_that_overflows(oracle_mesh, n, cap, before):
    from cellsim3d_amd import abi as A
    from cellsim3d_amd import configs, engine, mesh as M
    print("partners, overflow: %d cells, cap %d" % (n, cap), flush=True)
    ctx, s, p = _tissue(A, configs, engine, oracle_mesh, n, skin=0.1, cap=cap)
    base = M.centred(configs.unit_mesh()).astype(np.float32)
    with ctx:
        s.step(1)
        ctx.sync()
        rules = _rules_state(A, s)
        s.step(1)
        ctx.sync()
        want = _rule(p, _xyz(A, s), *rules, n)
        assert want.shape[0] > 0
        if before:
            assert np.array_equal(_lists(A, s, n), want)
        for k, x in enumerate(_xyz(A, s)):  # six cells in one place: 43 candidates of some node
            at = x.min() - np.float32(6.0)
            for c in range(6):
                x[c * 192:c * 192 + 180] = base[:, k] + (at + np.float32((0.03, 0.02, 0.01)[k] * c))
            s.set((A.F_X, A.F_Y, A.F_Z)[k], x)
        s.step(3)
        ctx.sync()
        assert s.info() == (n, 2, A.SYS_CAND_OVERFLOW)
        assert np.array_equal(_lists(A, s, n), want)
