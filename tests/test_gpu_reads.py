"""Reads of device memory: what the first one of a context costs."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_first_read_costs_what_the_next_one_does(oracle_mesh):
    """The pinned memory of small reads comes with the context, not with its first read
    (16 us where the next takes 14; allocated in it, 42)."""
    from cellsim3d_amd import configs, engine
    print("first reads", flush=True)
    p = configs.base_params(2)
    first, later = [], []
    for _ in range(9):
        with engine.Context(oracle_mesh, capacity_cells=8, voxel_budget=1 << 16, bin_budget=1 << 22) as ctx:
            s = ctx.add_system_raw(p, 8, max_cells=8, voxels=16)
            ctx.sync()
            for into in (first, later):
                t = time.perf_counter()
                s.info()
                into.append(time.perf_counter() - t)
    print("first %.1f us, next %.1f us" % (1e6 * np.median(first), 1e6 * np.median(later)), flush=True)
    assert np.median(first) < 2.0 * np.median(later)
