"""A batch of molecules whose shells have 3 and 6 primitives at most: the records
of all of them take the longer stride, in LDS too."""
import numpy as np
import pytest

from proteindf_amd import calc_grid, engine, guess, molecules

pytestmark = pytest.mark.gpu


def _chain(n):
    rng = np.random.default_rng(n)
    xyz = np.stack([1.7 * np.cos(0.9 * np.arange(n)), 1.7 * np.sin(0.9 * np.arange(n)), 0.35 * np.arange(n)], 1)
    return molecules.Molecule(["H"] * n, xyz + rng.uniform(-0.1, 0.1, xyz.shape), f"H{n}")


@pytest.mark.parametrize("prec", ["fp64", "bf16x3", "bf16x3k", "bfp", "f16k"])
def test_batch_of_short_and_long_contractions(prec):
    made = []
    for mol in (_chain(60), molecules.water_cluster(1, 2), _chain(16), molecules.water_cluster(3, 4)):
        info = calc_grid.orbital_info(mol)
        ctx = engine.XcContext(info, engine.default_opts(precision=engine.PRECISIONS[prec]))
        rng = np.random.default_rng(mol.n_atoms)
        n = 3000
        ctx.set_grid(np.concatenate([mol.xyz[rng.integers(0, mol.n_atoms, n)] + rng.normal(0.0, 1.0, (n, 3)),
                                     rng.uniform(0.0, 1.0, (n, 1))], 1))
        P = guess.pack_lower(np.diag(np.full(info.n_aos, 0.2)))
        made.append((ctx, P, *ctx.build_rks(P)[:2]))
    print("[gpu-case] a batch of two record lengths", prec, flush=True)
    batch = engine.XcBatch([m[0] for m in made])
    for _ in range(2):
        E, Ks = batch.build_rks([m[1] for m in made])
        for k, (_, _, e, K) in enumerate(made):
            assert E[k] == e
            np.testing.assert_allclose(Ks[k], K, rtol=0, atol=1e-12 * np.abs(K).max())
    batch.close()
    for m in made:
        m[0].close()
