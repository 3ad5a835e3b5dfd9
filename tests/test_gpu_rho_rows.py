"""rho and the grid come back in the caller's order also past the 2^22 points
that cross the bus at a time."""
import numpy as np
import pytest

from proteindf_amd import calc_grid, engine, guess, molecules

pytestmark = pytest.mark.gpu


def test_rows_of_more_points_than_cross_at_a_time():
    n = (1 << 22) + 5003
    mol = molecules.water_cluster(1, 4)
    info = calc_grid.orbital_info(mol)
    rng = np.random.default_rng(0)
    xyz = mol.xyz[rng.integers(0, 3, n)] + rng.normal(0.0, 1.5, (n, 3))
    grid = np.concatenate([xyz, rng.uniform(0.0, 1e-3, (n, 1))], 1)
    P = guess.pack_lower(0.5 * guess.density_guess(mol, info, seed=4, eps=0.05))
    print(f"[gpu-case] rho of {n} points", flush=True)
    ctx = engine.XcContext(info)
    ctx.set_grid(grid)
    np.testing.assert_array_equal(ctx.get_grid(), grid)
    rho = ctx.build_uks(P, 0.5 * P, want_rho=True)[3]
    want, grad = ctx.density_at_points(P, xyz, want_grad=True)
    ctx.close()
    scale = np.abs(want).max()
    np.testing.assert_allclose(rho[:, 0], want, rtol=0, atol=1e-12 * scale)
    np.testing.assert_allclose(rho[:, 1:4], grad, rtol=0, atol=1e-12 * np.abs(grad).max())
    np.testing.assert_allclose(rho[:, 4], 0.5 * want, rtol=0, atol=1e-12 * scale)
