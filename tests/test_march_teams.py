"""The counting march with teams of lanes and the writing march by log word, against the oracle: the numbers of rays where teams
begin with one lane up to a whole wavefront, dense grids (words full of samples, several windows a wavefront), stepping rules whose
steps go through calc_dt, rays that stop at the sample cap, a capacity that refuses rays, the sphere bound."""
import numpy as np
import pytest

from tests import helpers
from tests.test_gpu_parity import SAMPLER_VARIANTS, u32

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("team", [None, "1", "2", "16", "64"])
@pytest.mark.parametrize("variant,occupancy,n_rays,n_coords", [
    ("disparity", 0.02, 4097, 1 << 22), ("disparity", 0.7, 777, 1 << 22), ("disparity", 0.7, 3000, 100000), ("disparity", 0.1, 1, 1 << 20),
    ("log_stepping", 0.3, 1500, 1 << 22), ("original_stepping_fixed", 0.9, 500, 1 << 22), ("no_grid", 0.0, 300, 1 << 20)])
def test_training_march_by_teams(gpu, orc, variant, occupancy, n_rays, n_coords, team, monkeypatch):
    torch = gpu
    from sphericalrf_amd import api, scene
    if team is not None:
        monkeypatch.setenv("SRF_COUNT_TEAM", team)
    w = scene.workload(3, 1 / 16)
    cfg = dict(w["sampler"], num_cascades=2, maximum_marching_steps=300)
    cfg.update(SAMPLER_VARIANTS.get(variant, {}))
    p = helpers.oracle_params(orc, cfg)
    rng = np.random.default_rng(n_rays)
    s = api.OccupancySampler(cfg)
    bf = None
    if cfg.get("use_grid", True):
        # occupied and empty stretches of 64 cells, so that words are full, empty or mixed
        grid = np.repeat(rng.random(p.n_total // 64) < occupancy, 64).astype(np.float32)
        grid[rng.random(p.n_total) < 0.02] = 1.0
        bf, _ = orc.update_grid_bitfield(p, grid)
        s.set_density_grid(torch.from_numpy(grid).cuda())
        s.update_grid_bitfield()
    o_ds = orc.make_dataset(w["cameras"], w["resolution"], w["focal"], (0.5, 0.5))
    ds = api.Dataset(torch.from_numpy(w["cameras"]).cuda(), w["resolution"], w["focal"], (0.5, 0.5))
    want = orc.generate_training_samples(p, n_rays, 11, n_coords, o_ds, bf, orc.pcg32(5), numsteps_counter=3, coords_capacity=n_coords)
    rays, rgba = torch.zeros((n_rays, 6), device="cuda"), torch.zeros((n_rays, 4), device="cuda")
    ns, coords = torch.zeros((n_rays, 2), dtype=torch.int32, device="cuda"), torch.zeros((n_coords, 7), device="cuda")
    ts, dts, cell = torch.zeros(n_coords, device="cuda"), torch.zeros(n_coords, device="cuda"), torch.zeros(n_coords, dtype=torch.int32, device="cuda")
    rc, nc = torch.zeros(1, dtype=torch.int32, device="cuda"), torch.full((1,), 3, dtype=torch.int32, device="cuda")
    s.sample_coords_from_dataset(n_rays, 11, n_coords, ds, rays, rgba, rc, ns, coords, nc, api.Pcg32(5), ts, dts, cell)
    torch.cuda.synchronize()
    assert int(rc.item()) == want["ray_counter"] and int(u32(nc)[0]) == want["numsteps_counter"]
    n_kept = want["ray_counter"]
    assert np.array_equal(u32(ns)[:n_kept], want["numsteps"][:n_kept]) and np.array_equal(rays.cpu().numpy()[:n_kept], want["rays"][:n_kept])
    assert np.array_equal(u32(cell), want["cell"]) and np.array_equal(coords.cpu().numpy().view(np.uint32), want["coords"].view(np.uint32))
    assert np.array_equal(np.stack([ts.cpu().numpy(), dts.cpu().numpy()], axis=1), want["t_dt"])
