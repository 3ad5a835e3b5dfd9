"""Host entry points: packed P in, packed K out, and the integrated densities
summed by the build, against the same sums over the returned rho."""
import numpy as np
import pytest

from proteindf_amd import calc_grid, engine, guess, molecules

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 129, 256, 3001])
@pytest.mark.parametrize("uks", [False, True])
def test_whole_density_is_the_weighted_sum_of_rho(n, uks):
    mol = molecules.water_cluster(1, 8)
    info = calc_grid.orbital_info(mol)
    rng = np.random.default_rng(n)
    grid = np.concatenate([mol.xyz[rng.integers(0, 3, n)] + rng.normal(0.0, 1.0, (n, 3)),
                           rng.uniform(0.0, 1.0, (n, 1))], 1)
    P = guess.pack_lower(0.5 * guess.density_guess(mol, info, seed=8, eps=0.05))
    print(f"[gpu-case] whole density, {n} points, uks {uks}", flush=True)
    ctx = engine.XcContext(info)
    ctx.set_grid(grid)
    if uks:
        rho = ctx.build_uks(P, 0.7 * P, want_rho=True)[3]
        got, want = ctx.whole_density(2), (grid[:, 3:4] * rho[:, [0, 4]]).sum(0)
    else:
        K0 = rng.normal(size=P.shape)
        rho = ctx.build_rks(P, want_rho=True)[2]
        K = ctx.build_rks(P)[1]
        K1 = ctx.build_rks(P, K0.copy())[1]  # accumulates, in packed order
        np.testing.assert_allclose(K1, K0 + K, rtol=0, atol=1e-13 * np.abs(K).max() + 1e-15)
        ctx.build_rks_update(P)  # doubles the stored density
        got, want = ctx.whole_density(), 2.0 * (grid[:, 3] * rho[:, 0]).sum()
    ctx.close()
    np.testing.assert_allclose(got, want, rtol=1e-13)
