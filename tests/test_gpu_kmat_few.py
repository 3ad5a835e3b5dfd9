"""FP64 K pass of few blocks: shapes joined into the widest, items cut to fill
the CUs, every patch exactly once; a batch of such contexts, whose items are its
own; against the oracle and, for the batch, against each context."""
import numpy as np
import pytest

from oracle import oracle
from proteindf_amd import calc_grid, engine, guess, molecules

pytestmark = pytest.mark.gpu


def _grid(mol, n, seed):
    rng = np.random.default_rng(seed)
    return np.concatenate([mol.xyz[rng.integers(0, mol.n_atoms, n)] + rng.normal(0.0, 0.7, (n, 3)),
                           rng.uniform(0.0, 1.0, (n, 1))], 1)


# 18 to 456 AOs without screening: narrow blocks alone, both narrow shapes with wide ones, wide ones cut
@pytest.mark.parametrize("waters,n_pts", [(1, 1000), (7, 1000), (10, 2000), (13, 1500), (19, 900), (24, 700)])
def test_few_blocks_of_every_width(waters, n_pts):
    mol = molecules.water_cluster(waters, waters)
    info = calc_grid.orbital_info(mol)
    PA = 0.5 * guess.density_guess(mol, info, seed=waters, eps=0.05)
    grid = _grid(mol, n_pts, waters)
    print(f"[gpu-case] K of few blocks, {info.n_aos} AOs, {n_pts} points", flush=True)
    ctx = engine.XcContext(info)
    ctx.set_grid(grid)
    E, K, _ = ctx.build_rks(guess.pack_lower(PA))
    KA, KB = ctx.build_uks(guess.pack_lower(PA), guess.pack_lower(PA))[1:3]
    ctx.close()
    e_ref, K_ref, _ = oracle.calc_xc_rks(oracle.AoTable.from_basis(info), grid, PA)
    assert abs(E - e_ref) <= 1e-10
    for got in (K, KA, KB):
        np.testing.assert_allclose(guess.unpack_lower(got, info.n_aos), K_ref, rtol=0, atol=1e-10)


def test_a_batch_sizes_its_own_items():
    made = []
    for waters, n in ((1, 40000), (7, 30000), (13, 20000), (20, 1000), (3, 1), (10, 60000)):
        mol = molecules.water_cluster(waters, waters)
        info = calc_grid.orbital_info(mol)
        ctx = engine.XcContext(info)
        ctx.set_grid(_grid(mol, n, n))
        P = guess.pack_lower(0.5 * guess.density_guess(mol, info, seed=waters, eps=0.05))
        made.append((ctx, P, *ctx.build_rks(P)[:2]))
    print("[gpu-case] a batch of few blocks each", flush=True)
    batch = engine.XcBatch([m[0] for m in made])
    for _ in range(2):
        E, Ks = batch.build_rks([m[1] for m in made])
        for k, (_, _, e, K) in enumerate(made):
            assert E[k] == e
            np.testing.assert_allclose(Ks[k], K, rtol=0, atol=1e-12 * np.abs(K).max())
    batch.close()
    for m in made:
        m[0].close()
