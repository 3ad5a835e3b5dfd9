"""FP64 K pass at the edges of its workgroup shapes: odd and even tile counts,
the widest block of every shape, blocks cut into several items, partial slabs.
K sums of a few hundred points agree with the oracle to the 1e-10 of every
FP64 build; one grid in another order or other items changes the summation
order alone."""
import numpy as np
import pytest
import torch

from oracle import oracle
from proteindf_amd import calc_grid, engine, guess, molecules

pytestmark = pytest.mark.gpu


def _points(mol, n, seed):
    rng = np.random.default_rng(seed)
    return np.concatenate([mol.xyz[rng.integers(0, mol.n_atoms, n)] + rng.normal(0.0, 1.0, (n, 3)),
                           rng.uniform(0.0, 1.0, (n, 1))], 1)


# 13 AOs a water without screening: 1, 2, 8, 9, 10, 11, 16, 17 and 22 tiles a side
@pytest.mark.parametrize("waters", [1, 2, 9, 10, 12, 13, 19, 20, 27])
@pytest.mark.parametrize("n_pts", [5, 300])
def test_k_of_every_tile_count(waters, n_pts):
    mol = molecules.water_cluster(waters, waters)
    info = calc_grid.orbital_info(mol)
    PA = 0.5 * guess.density_guess(mol, info, seed=waters, eps=0.05)
    grid = _points(mol, n_pts, waters)
    print(f"[gpu-case] K of {info.n_aos} AOs, {n_pts} points", flush=True)
    ctx = engine.XcContext(info)
    ctx.set_grid(grid)
    E, K, _ = ctx.build_rks(guess.pack_lower(PA))
    e_ref, K_ref, _ = oracle.calc_xc_rks(oracle.AoTable.from_basis(info), grid, PA)
    assert abs(E - e_ref) <= 1e-10
    np.testing.assert_allclose(guess.unpack_lower(K, info.n_aos), K_ref, rtol=0, atol=1e-10)
    ctx.set_tuning(k_tiles=8)
    K8 = ctx.build_rks(guess.pack_lower(PA))[1]
    ctx.close()
    np.testing.assert_allclose(K8, K, rtol=0, atol=1e-12)


@pytest.mark.parametrize("waters", [3, 11])
def test_pairs_of_blocks_give_the_sum_of_two_grids(waters):
    # 10 units of two blocks per CU and a ragged rest; its halves run block by block
    half = 10 * torch.cuda.get_device_properties(0).multi_processor_count * 128
    mol = molecules.water_cluster(waters, 5)
    info = calc_grid.orbital_info(mol)
    P = guess.pack_lower(0.5 * guess.density_guess(mol, info, seed=5, eps=0.05))
    grid = _points(mol, 2 * half + 77, 5)
    print(f"[gpu-case] pairs of blocks, {len(grid)} points, {info.n_aos} AOs", flush=True)
    ctx = engine.XcContext(info)
    got = []
    for part in (grid, grid[:half], grid[half:]):
        ctx.set_grid(part)
        got.append(ctx.build_rks(P))
    ctx.close()
    # 1e-12 of the sums: the order of about 10^6 terms
    assert abs(got[0][0] - got[1][0] - got[2][0]) <= 1e-12 * abs(got[0][0])
    np.testing.assert_allclose(got[0][1], got[1][1] + got[2][1], rtol=0, atol=1e-12 * np.abs(got[0][1]).max())
