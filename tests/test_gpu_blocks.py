"""Grid blocks made on the device: the same cuts and the same AO lists as a
plain numpy bisection, at the edges of the node sizes (one block, the points
one workgroup cuts, several levels above it), on grids full of equal
coordinates; the per-point results come back in the caller's order."""
import numpy as np
import pytest

from oracle import oracle
from proteindf_amd import calc_grid, engine, guess, molecules

pytestmark = pytest.mark.gpu


def _leaves(xyz):
    """Point indices of every block: cuts at 128 (ceil(n / 128) // 2) along the widest extent, ties by index."""
    out, stack = [], [np.arange(len(xyz))]
    while stack:
        idx = stack.pop()
        n = len(idx)
        if n <= 128:
            out.append(idx)
            continue
        p = xyz[idx]
        ext = p.max(0) - p.min(0)
        d = int(np.argmax(ext))
        idx = idx[np.lexsort((idx, p[:, d]))]
        mid = 128 * (((n + 127) // 128) // 2)
        stack += [idx[mid:], idx[:mid]]
    return out


def _flops(info, xyz):
    """sum 4 n N_b^2 over the blocks, N_b the AOs whose most diffuse primitive reaches the block's box."""
    c = np.asarray(info.ao_center)
    e0 = np.array([min(e) for e in info.ao_exps])
    total = 0.0
    for idx in _leaves(xyz):
        p = xyz[idx]
        lo, hi = p.min(0), p.max(0)
        d = np.maximum(0.0, np.maximum(lo - c, c - hi))
        dm2 = (d * d).sum(1) * (1.0 - 1e-12) ** 2
        total += 4.0 * len(idx) * float((e0 * dm2 <= 30.0).sum()) ** 2
    return total


def _points(kind, n, mol, rng):
    if kind == "cube":  # many equal coordinates
        m = int(np.ceil(n ** (1.0 / 3.0)))
        ax = np.arange(m) * 0.9 - 3.0
        return np.stack(np.meshgrid(ax, ax, ax, indexing="ij"), -1).reshape(-1, 3)[:n]
    if kind == "line":  # two of three coordinates equal, one with repeats and both zeros
        x = np.zeros((n, 3))
        x[:, 1] = rng.integers(-20, 20, n) * 0.5
        x[::2, 1] *= -1.0
        return x
    return mol.xyz[rng.integers(0, mol.n_atoms, n)] + rng.normal(0.0, 3.0, (n, 3))


@pytest.mark.parametrize("kind", ["cloud", "cube", "line"])
@pytest.mark.parametrize("n", [1, 128, 129, 300, 4096, 4097, 8192, 8193, 20001])
def test_blocks_match_a_plain_bisection(kind, n):
    mol = molecules.water_cluster(3, 4)
    info = calc_grid.orbital_info(mol)
    xyz = _points(kind, n, mol, np.random.default_rng(n))
    print(f"[gpu-case] blocks of {n} points, {kind}", flush=True)
    ctx = engine.XcContext(info)
    ctx.set_grid(np.concatenate([xyz, np.ones((n, 1))], 1))
    s = ctx.stats()
    assert s.n_blocks == (n + 127) // 128
    assert s.flops == _flops(info, xyz)
    np.testing.assert_array_equal(ctx.get_grid()[:, :3], xyz)
    ctx.close()


@pytest.mark.parametrize("n", [1, 127, 4097, 13000])
def test_point_results_keep_the_callers_order(n):
    mol = molecules.water_cluster(2, 3)
    info = calc_grid.orbital_info(mol)
    PA = 0.5 * guess.density_guess(mol, info, seed=3, eps=0.05)
    xyz = _points("cloud", n, mol, np.random.default_rng(n))
    print(f"[gpu-case] rho of {n} points", flush=True)
    grid = np.concatenate([xyz, np.full((n, 1), 1e-3)], 1)
    ref = oracle.calc_xc_rks(oracle.AoTable.from_basis(info), grid, PA, want_rho=True)[2]
    ctx = engine.XcContext(info)
    ctx.set_grid(grid)
    rho = ctx.build_rks(guess.pack_lower(PA), want_rho=True)[2]
    rho_p, grad_p = ctx.density_at_points(guess.pack_lower(PA), xyz, want_grad=True)
    rho_1 = ctx.density_at_points(guess.pack_lower(PA), xyz)
    ctx.close()
    scale = np.abs(ref).max()
    np.testing.assert_allclose(rho, ref, rtol=0, atol=1e-12 * scale)
    np.testing.assert_allclose(rho_p, ref[:, 0], rtol=0, atol=1e-12 * scale)
    np.testing.assert_allclose(grad_p, ref[:, 1:4], rtol=0, atol=1e-12 * scale)
    np.testing.assert_array_equal(rho_1, rho_p)
