"""Weight term of the gradient where the partition function Z of a point is far
below 1: near the centre of a hollow cage every atom is about as far, every cell
product of n atoms is about 2^-(n - 1) and none of them may be dropped.  The
oracle drops nothing; 1e-10 of the largest component, as elsewhere."""
import numpy as np
import pytest

from oracle import oracle
from proteindf_amd import calc_grid, engine, guess, molecules

pytestmark = pytest.mark.gpu


def _cage(n, radius):
    """n hydrogen atoms spread over a sphere (golden spiral)."""
    k = np.arange(n) + 0.5
    z = 1.0 - 2.0 * k / n
    phi = np.pi * (1.0 + 5.0 ** 0.5) * k
    s = np.sqrt(1.0 - z * z)
    return molecules.Molecule(["H"] * n, radius * np.stack([s * np.cos(phi), s * np.sin(phi), z], 1), f"H{n}")


def _compare(mol, pts, atom, ss):
    rng = np.random.default_rng(7)
    info = calc_grid.orbital_info(mol)
    PA = np.diag(np.full(info.n_aos, 0.2))
    grid = np.concatenate([pts, rng.uniform(0.1, 1.0, (len(pts), 1))], 1)
    print(f"[gpu-case] weight term, {mol.n_atoms} atoms, ss {ss}", flush=True)
    ctx = engine.XcContext(info)
    if ss:  # the grid's partition is the one it was generated with
        o = oracle.grid_opts(n_rad=8, n_ang=50, pruning=0, partitioning=ss)
        opts = engine.GridOpts(**{f: getattr(o, f) for f, _ in engine.GridOpts._fields_})
        ctx.generate_grid_ex(mol.Z, mol.xyz, opts)
        grid, atom = oracle.generate_grid_ex(mol.Z, mol.xyz, o)
        E, gf, gw = ctx.gradient_rks(mol.Z, mol.xyz, guess.pack_lower(PA))
    else:
        ctx.set_grid(grid)
        E, gf, gw = ctx.gradient_rks(mol.Z, mol.xyz, guess.pack_lower(PA), point_atom=atom)
    ctx.close()
    e_ref, gf_ref, gw_ref = oracle.xc_gradient_rks(oracle.AoTable.from_basis(info), info.ao_atom, grid, atom,
                                                   mol.Z, mol.xyz, PA, partition=2 * ss)
    scale = np.abs(gw_ref).max()
    assert scale > 0.0
    assert abs(E - e_ref) <= 1e-10 * abs(e_ref)
    np.testing.assert_allclose(gw, gw_ref, rtol=0, atol=1e-10 * scale)


@pytest.mark.parametrize("n", [60, 100, 240])
def test_points_at_the_centre_of_a_cage(n):
    mol = _cage(n, 0.5 * n ** 0.5)
    rng = np.random.default_rng(n)
    atom = np.sort(rng.integers(0, n, 300)).astype(np.int32)
    _compare(mol, rng.normal(0.0, 0.1, (300, 3)), atom, 0)


def test_generated_ss_grid_of_a_cage():
    # the radius of the atoms' last shell but one: some of its points fall next to the centre
    o = oracle.grid_opts(n_rad=8, n_ang=50, pruning=0, partitioning=1)
    one = oracle.generate_grid_ex(np.array([1], dtype=np.int32), np.zeros((1, 3)), o)[0]
    radius = np.unique(np.round(np.linalg.norm(one[:, :3], axis=1), 9))[-2]
    _compare(_cage(100, radius), np.zeros((1, 3)), None, 1)


@pytest.mark.parametrize("n", [276, 277])
def test_four_waves_and_one_per_workgroup(n):
    # a chain: 276 atoms are the most that leave two workgroups of four waves on a CU
    rng = np.random.default_rng(n)
    xyz = np.zeros((n, 3))
    xyz[:, 0] = 2.1 * np.arange(n)
    mol = molecules.Molecule(["H"] * n, xyz + rng.uniform(-0.2, 0.2, xyz.shape), f"H{n}")
    atom = np.sort(rng.integers(0, n, 600)).astype(np.int32)
    _compare(mol, mol.xyz[atom] + rng.normal(0.0, 0.6, (600, 3)), atom, 0)
