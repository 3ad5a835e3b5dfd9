"""pdfxc_whole_density holds the integrals of the context's last host build and
nothing older: zero after HF, zero beta after RKS, refused before a build, after
a new grid and after a build that failed."""
import numpy as np
import pytest

from proteindf_amd import calc_grid, engine, guess, molecules

pytestmark = pytest.mark.gpu


def test_values_are_those_of_the_last_build():
    mol = molecules.water_cluster(1, 8)
    info = calc_grid.orbital_info(mol)
    rng = np.random.default_rng(2)
    grid = np.concatenate([mol.xyz[rng.integers(0, 3, 500)] + rng.normal(0.0, 1.0, (500, 3)),
                           rng.uniform(0.0, 1.0, (500, 1))], 1)
    P = guess.pack_lower(0.5 * guess.density_guess(mol, info, seed=8, eps=0.05))
    print("[gpu-case] whole density over builds", flush=True)
    ctx = engine.XcContext(info)

    def refused():
        with pytest.raises(engine.PdfxcError) as e:
            ctx.whole_density()
        assert e.value.code == engine.ERROR_CODES["ARGUMENT"]

    refused()
    ctx.set_grid(grid)
    refused()
    rho = ctx.build_uks(P, 0.7 * P, want_rho=True)[3]
    ab = (grid[:, 3:4] * rho[:, [0, 4]]).sum(0)
    np.testing.assert_allclose(ctx.whole_density(2), ab, rtol=1e-13)
    ctx.build_rks(P)
    np.testing.assert_allclose(ctx.whole_density(2), [ab[0], 0.0], rtol=1e-13)
    ctx.build_uks(P, 0.7 * P)
    ctx.build_uks(P, P, functional=engine.PDFXC_HF)
    assert ctx.whole_density(2) == (0.0, 0.0)
    ctx.build_rks(P)
    ctx.build_rks(P, functional=engine.PDFXC_HF)
    assert ctx.whole_density() == 0.0
    ctx.build_rks(P)
    ctx.set_tuning(k_tiles=24)  # the same grid and build
    np.testing.assert_allclose(ctx.whole_density(), ab[0], rtol=1e-13)
    ctx.set_grid(grid[:300])
    refused()
    ctx.build_rks(P)
    bad = grid.copy()
    bad[7, 0] = np.nan
    with pytest.raises(engine.PdfxcError):
        ctx.set_grid(bad)
    refused()
    with pytest.raises(engine.PdfxcError):
        ctx.build_rks(P)
    refused()
    ctx.close()
