"""One context read from several threads: its grid taken and batches made of it
while another thread builds."""
import threading

import numpy as np
import pytest

from proteindf_amd import calc_grid, engine, guess, molecules

pytestmark = pytest.mark.gpu


def test_grid_and_batches_while_another_thread_builds():
    mol = molecules.water_cluster(2, 6)
    info = calc_grid.orbital_info(mol)
    rng = np.random.default_rng(1)
    P = guess.pack_lower(0.5 * guess.density_guess(mol, info, seed=6, eps=0.05))
    grid = np.concatenate([mol.xyz[rng.integers(0, mol.n_atoms, 40000)] + rng.normal(0.0, 1.0, (40000, 3)),
                           rng.uniform(0.0, 1.0, (40000, 1))], 1)
    ctx = engine.XcContext(info)
    ctx.set_grid(grid)
    E = ctx.build_rks(P)[0]
    print("[gpu-case] a context shared by threads", flush=True)
    builds, grids, batches = [], [], []
    work = [lambda: builds.extend(ctx.build_rks(P)[0] for _ in range(20)),
            lambda: grids.extend(ctx.get_grid() for _ in range(20)),
            lambda: batches.append(engine.XcBatch([ctx])),
            lambda: batches.append(engine.XcBatch([ctx]))]
    threads = [threading.Thread(target=w) for w in work]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert builds == [E] * 20
    assert len(grids) == 20 and all(np.array_equal(g, grid) for g in grids)
    assert [float(b.build_rks([P])[0][0]) for b in batches] == [E] * 2
    for b in batches:
        b.close()
    ctx.close()
