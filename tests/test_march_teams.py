"""The counting march with teams of lanes and the writing march by log word, against the oracle: the numbers of rays where teams
begin with one lane up to a whole wavefront, dense grids (words full of samples, several windows a wavefront), stepping rules whose
steps go through calc_dt, rays that stop at the sample cap, a capacity that refuses rays; then the render marches the same way, and
under a sphere bound."""
import numpy as np
import pytest

from oracle import oracle as O
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


@pytest.mark.parametrize("team", [None, "1", "2", "8", "64"])
@pytest.mark.parametrize("variant,occupancy,sphere", [
    ("disparity", 0.01, False), ("disparity", 0.6, False), ("log_stepping", 0.1, False), ("original_stepping_cone", 0.05, False), ("reciprocal_grid", 0.05, False),
    ("disparity", 0.05, True)])
def test_render_marches_by_teams(gpu, orc, variant, occupancy, sphere, team, monkeypatch):
    """fused frame, first hits, three rounds of coordinates (a ray's last samples in the middle of a team's steps among them), with a
    number of rays that fills neither wavefronts nor teams; under a sphere bound against the march of a ray a lane"""
    torch = gpu
    from sphericalrf_amd import api, scene
    w = scene.workload(3, 1 / 16)
    cfg = dict(w["sampler"], num_cascades=2, maximum_marching_steps=300)
    cfg.update(SAMPLER_VARIANTS.get(variant, {}))
    p = helpers.oracle_params(orc, cfg)
    rng = np.random.default_rng(5)
    grid = np.repeat(rng.random(p.n_total // 64) < occupancy, 64).astype(np.float32)
    grid[rng.random(p.n_total) < 0.01] = 1.0
    bf, _ = orc.update_grid_bitfield(p, grid)
    res, cam, f = (61, 35), w["cameras"][0], (30.0, 30.0)
    n = res[0] * res[1]
    table = scene.field_table(4096, 5)
    table[:, 3] *= 5

    def march(lanes):
        with monkeypatch.context() as env:
            if lanes is not None:
                env.setenv("SRF_MARCH_TEAM", lanes)
            s = api.OccupancySampler(cfg)
        s.set_density_grid(torch.from_numpy(grid).cuda())
        s.update_grid_bitfield()
        if sphere:
            s.set_ray_sphere_bound((0.5, 0.5, 0.5), 0.8)
        m = api.RayMarcher(dict(train_in_linear_color=False, transmittance_threshold=1e-4))
        frame, ns = torch.ones((res[1], res[0], 4), device="cuda"), torch.zeros(n, dtype=torch.int32, device="cuda")
        s.render_frame_fused(m, api.Field(torch.from_numpy(table).cuda(), 77), res, f, (0.5, 0.5), cam, frame, ns, spp=3)
        pay = torch.zeros(n * 40, dtype=torch.uint8, device="cuda")
        s.generate_rays_from_camera_matrix(res, f, (0.5, 0.5), cam, pay)
        out = [frame.cpu().numpy(), u32(ns).reshape(res[1], res[0]), pay.cpu().numpy().view(O.PAYLOAD_DTYPE).copy()]
        for n_steps in (1, 5, 8):
            coords = torch.zeros((n * n_steps, 7), device="cuda")
            s.generate_coords_from_rays(n, n_steps, pay, coords)
            out += [coords.cpu().numpy(), pay.cpu().numpy().view(O.PAYLOAD_DTYPE).copy()]
        return out

    if sphere:
        want = march("1")
    else:
        frame, ns, _ = orc.render_frame(p, orc.make_field(table, 77), bf, res, f, (0.5, 0.5), cam, spp=3, transmittance_threshold=1e-4, train_in_linear_colors=False)
        pay = orc.init_rays_with_payload(p, res, f, (0.5, 0.5), cam)
        orc.advance_pos(p, pay, bf)
        want = [frame, ns, pay.copy()]
        for n_steps in (1, 5, 8):
            coords = np.zeros((n * n_steps, 7), np.float32)
            orc.generate_coords_from_rays(p, n, n_steps, bf, pay, coords)
            want += [coords, pay.copy()]
    got = march(team)
    assert want[1].sum() > 0 and len(got) == len(want)
    for a, b in zip(got, want):
        assert np.array_equal(a, b)
