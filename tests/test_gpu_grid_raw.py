"""Generated grids with Stratmann-Scuseria weights at the edges of the wave's
atom loops (1, 63, 64 and 66 atoms, dummies among them), against the oracle:
points in its order, weights to 1e-12 (1e-13 of 1, where 1 - g cancels)."""
import numpy as np
import pytest

from oracle import oracle
from proteindf_amd import calc_grid, engine, molecules

pytestmark = pytest.mark.gpu


def _case(waters, dummies):
    if waters == 0:
        return np.array([8], dtype=np.int32), np.zeros((1, 3))
    mol = molecules.water_cluster(waters, seed=waters)
    rng = np.random.default_rng(waters)
    Z = np.append(mol.Z, np.zeros(dummies, dtype=mol.Z.dtype))
    return Z, np.vstack([mol.xyz, mol.xyz.mean(0) + rng.normal(0.0, 2.0, (dummies, 3))])


@pytest.mark.parametrize("waters,dummies", [(0, 0), (1, 0), (21, 0), (21, 1), (22, 0), (43, 2)])
def test_ss_grid_matches_oracle(waters, dummies):
    Z, xyz = _case(waters, dummies)
    kw = dict(n_rad=17, n_ang=50, pruning=1, partitioning=1)
    print(f"[gpu-case] SS grid of {len(Z)} atoms", flush=True)
    o = oracle.grid_opts(**kw)
    ctx = engine.XcContext(calc_grid.orbital_info(molecules.water_cluster(1, seed=0)))
    ctx.generate_grid_ex(Z, xyz, engine.GridOpts(**{f: getattr(o, f) for f, _ in engine.GridOpts._fields_}))
    g = ctx.get_grid()
    ctx.close()
    ref = oracle.generate_grid_ex(Z, xyz, o)[0]
    # a point at the weight screen may be kept by one side alone
    big, ref_big = g[np.abs(g[:, 3]) > 1e-13], ref[np.abs(ref[:, 3]) > 1e-13]
    assert len(big) == len(ref_big) and abs(len(g) - len(ref)) <= 1e-3 * len(ref)
    np.testing.assert_allclose(big[:, :3], ref_big[:, :3], rtol=0, atol=1e-11)
    np.testing.assert_allclose(big[:, 3], ref_big[:, 3], rtol=1e-12, atol=1e-13)
