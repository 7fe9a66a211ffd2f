"""The non-uniform grid draw dealt by cell and brought back into point order, in order and by runs of 32 points, against the oracle:
numbers of points round a run, a window of 1024 and whole multiples of the cell count, in the caller's and in cell order."""
import numpy as np
import pytest

from tests import helpers
from tests.test_gpu_parity import u32

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("path", ["1", "2"])
@pytest.mark.parametrize("N,C", [((8, 8, 8), 2), ((32, 16, 16), 1), ((32, 16, 16), 5)])
def test_point_order_of_a_draw_dealt_by_cell(gpu, orc, N, C, path, monkeypatch):
    torch = gpu
    monkeypatch.setenv("SRF_GRID_SAMPLE_BY_CELL", path)
    from sphericalrf_amd import api
    cfg = dict(warping_type="ERP", aabb_scale=16, grid_size=N, num_cascades=C, grid_distribution_type="WarpedSpace_Exp", init_grid_with_mask=False,
               maximum_marching_steps=256, sampling_type="Disparity", near_distance=0.05, far_distance=10.0)
    p = helpers.oracle_params(orc, cfg)
    nc = p.n_total // C
    rng = np.random.default_rng(3)
    grid = np.where(rng.random(p.n_total) < 0.3, 1.0, 0.0).astype(np.float32)
    for k, n in enumerate([1, 31, 33, nc - 1, nc, nc + 1, 1023, 1025, 3 * nc + 33]):
        s = api.OccupancySampler(cfg)
        caller, o_caller = api.Pcg32(9 + k), orc.pcg32(9 + k)
        s.init(1, (4, 4), (1.0, 1.0), (0.5, 0.5), None, None, caller)
        o_rng = orc.pcg32(orc.next_uint(o_caller), 1)
        s.set_density_grid(torch.from_numpy(grid).cuda())
        pos, idx = torch.zeros((n, 3), device="cuda"), torch.zeros(n, dtype=torch.int32, device="cuda")
        s.sample_positions_from_grid(0, n, pos, idx)
        orc.advance(o_rng)
        want_pos, want_idx = orc.generate_grid_samples(p, n, o_rng, 0, grid, p.min_optical_thickness)
        assert np.array_equal(u32(idx), want_idx) and np.array_equal(pos.cpu().numpy(), want_pos)
