"""Calls that answer from the context alone may be made while a graph is being
captured on another stream."""
import numpy as np
import pytest
import torch

from proteindf_amd import calc_grid, engine, molecules

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [500, 70000])
def test_grid_is_read_during_a_capture(n, tmp_path):
    mol = molecules.water_cluster(1, 6)
    rng = np.random.default_rng(1)
    grid = rng.normal(size=(n, 4))  # 70,000: rows larger than any workspace its set-up has left behind
    ctx = engine.XcContext(calc_grid.orbital_info(mol))
    ctx.set_grid(grid)
    x = torch.zeros(64, device="cuda")
    print("[gpu-case] grid rows during a capture", flush=True)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        x.add_(1.0)
        rows = ctx.get_grid()
        ctx.save_grid_matrix(tmp_path / "grid.mat", 0)
        x.add_(2.0)
    np.testing.assert_array_equal(rows, grid)
    np.testing.assert_array_equal(engine.load_general_matrix(tmp_path / "grid.mat")[:, :4], grid)
    for k in range(1, 4):
        graph.replay()
        torch.cuda.synchronize()
        assert float(x.sum()) == 64 * 3.0 * k
        np.testing.assert_array_equal(ctx.get_grid(), grid)
    ctx.close()
