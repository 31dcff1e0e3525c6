"""Frames of the renderers that shade samples through a wavefront queue, at the sizes where
it can go wrong: one pixel, one ray past a tile, rays of fewer and of several times 64
samples, samples from several rays in one batch, and one or more rays per wavefront."""
import numpy as np
import pytest

import oracle_lib as O
from cpp_volume_rendering_amd import native as N
from cpp_volume_rendering_amd import workloads as W

pytestmark = pytest.mark.gpu
TOL = 2e-3

# (volume side, width, height, alpha limit): 24 voxels give rays of at most 83 samples, 96
# at a low opacity several hundred
SIZES = [(24, 1, 1, 0.95), (24, 17, 3, 0.95), (24, 33, 31, 0.3), (96, 16, 16, 0.02), (96, 5, 18, 0.95)]


# frames of more than one ray per wavefront, the last of them past the image
MANY = [(24, 97, 71, 0.95), (24, 160, 131, 0.3)]


def scene(tech, n, w, h, alpha_max, **params):
    wl = W.cone_blobs(n=n, width=w, height=h, seed=31)
    rgb, a = W.seeded_tf(131, 4, alpha_max=alpha_max)
    r = N.Renderer(tech)
    r.set_volume(wl.volume, wl.scale)
    r.set_transfer_function(rgb, a)
    p = r.params()
    for k, v in params.items():
        if k == "base_res":
            p.base_res[:] = list(v)
        else:
            setattr(p, k, v)
    r.set_params(p)
    r.collect_stats()
    img = r.render(wl.camera(), w, h, light=wl.light())
    return wl, O.OTF(rgb, a), r, r.params(), img


def check(img, ref, m):
    s = O.compare(img, ref, m, TOL, 1)
    print(s)
    assert s["max_abs"] <= TOL, s
    assert s["n_over_tol"] <= 0.005 * s["n_pixels"] + 1, s


@pytest.mark.parametrize("n,w,h,alpha_max", SIZES)
def test_cone(n, w, h, alpha_max):
    wl, tf, r, p, img = scene(N.CONE_TRACE, n, w, h, alpha_max, n_steps=8)
    pyr = O.OPyr.build(wl.volume, tf, nlev=6)
    ref, m = O.render_cone(wl.volume, tf, pyr, O.cone_params(wl.grid, wl.light(), n_steps=8), wl.camera(), w, h)
    check(img, ref, m)


# schedules of one step, of steps of one level only, of two levels from the first on, and remainders of
# the groups in which steps are loaded
@pytest.mark.parametrize("n_steps,n_levels,half,occ,sdw", [(1, 1, 30, 1, 1), (2, 6, 30, 1, 0), (3, 2, 80, 1, 1),
                                                           (5, 6, 5, 0, 1), (64, 3, 30, 1, 1), (7, 6, 89, 1, 1)])
def test_cone_schedules(n_steps, n_levels, half, occ, sdw):
    wl, tf, r, p, img = scene(N.CONE_TRACE, 24, 17, 13, 0.6, n_steps=n_steps, n_levels=n_levels, occ_half_deg=half,
                              apply_occlusion=occ, apply_shadow=sdw)
    pyr = O.OPyr.build(wl.volume, tf, nlev=n_levels)
    prm = O.cone_params(wl.grid, wl.light(), n_steps=n_steps, occ_half_deg=half, apply_occ=occ, apply_sdw=sdw)
    ref, m = O.render_cone(wl.volume, tf, pyr, prm, wl.camera(), 17, 13)
    check(img, ref, m)


@pytest.mark.parametrize("n,w,h,alpha_max", SIZES + MANY)
def test_dos(n, w, h, alpha_max):
    wl, tf, r, p, img = scene(N.DOS, n, w, h, alpha_max, apply_shadow=1, shadow_type=2, base_res=(24, 24, 24))
    pyr = O.OPyr.build(wl.volume, tf, base=(24, 24, 24))
    ref, m = O.render_dos(wl.volume, tf, pyr, O.dos_params(p, wl.grid, wl.light()), wl.camera(), w, h)
    check(img, ref, m)


@pytest.mark.parametrize("n,w,h,alpha_max", SIZES)
@pytest.mark.parametrize("shadow_type", [0, 2])
def test_ground_truth(n, w, h, alpha_max, shadow_type):
    wl, tf, r, p, img = scene(N.CONE_GT, n, w, h, alpha_max, occ_rays=3, sdw_rays=2, shadow_type=shadow_type)
    ref, m = O.render_gt(wl.volume, tf, O.gt_params(p, wl.grid, wl.light()), wl.camera(), w, h)
    check(img, ref, m)


@pytest.mark.parametrize("n,w,h,alpha_max", SIZES + MANY)
@pytest.mark.parametrize("shadow_type", [0, 1])
def test_ebs(n, w, h, alpha_max, shadow_type):
    wl, tf, r, p, img = scene(N.EBS, n, w, h, alpha_max, shadow_type=shadow_type)
    prm = O.ebs_params(p, wl.light())
    prm.sdw_max_dist = np.float32(0.75) * np.float32(np.linalg.norm(wl.grid))
    ref, m = O.render_ebs(wl.volume, tf, O.sat(wl.volume, tf), prm, wl.camera(), w, h)
    check(img, ref, m)


def test_ebs_tables_that_leave_room_for_one_queue():
    """A 4096-entry transfer function and a shadow chain of 2700 boxes: 146 KiB of LDS beside
    a single wavefront's queue."""
    wl = W.cone_blobs(n=24, width=33, height=31, seed=31)
    rgb, a = W.seeded_tf(131, 4, max_density=4095)
    r = N.Renderer(N.EBS)
    r.set_volume(wl.volume, wl.scale)
    r.set_transfer_function(rgb, a, max_density=4095)
    # a sample's chain stops at the volume's edge, far before its table does
    p = r.set_params(shadow_type=1, sdw_max_dist=7300.0)
    img = r.render(wl.camera(), 33, 31, light=wl.light())
    tf = O.OTF(rgb, a, max_density=4095)
    ref, m = O.render_ebs(wl.volume, tf, O.sat(wl.volume, tf), O.ebs_params(p, wl.light()), wl.camera(), 33, 31)
    check(img, ref, m)


@pytest.mark.parametrize("n,w,h,alpha_max", SIZES + MANY + [(24, 257, 259, 0.95)])
def test_surrogate(n, w, h, alpha_max):
    """4 and 16 rays per wavefront, four of them marching side by side."""
    wl = W.cone_blobs(n=n, width=w, height=h, seed=31)
    rgb, a = W.seeded_tf(131, 4, alpha_max=alpha_max)
    r = N.Renderer(N.CONE_NN)
    r.set_volume(wl.volume, wl.scale)
    r.set_transfer_function(rgb, a)
    rng = np.random.default_rng(3)
    wts = rng.normal(0, 0.1, N.lib().cvr_nn_param_count()).astype(np.float32)
    r.nn_set_weights(wts)
    r.collect_stats()
    img = r.render(wl.camera(), w, h, light=wl.light())
    tf = O.OTF(rgb, a)
    pyr = O.OPyr.build(wl.volume, tf, nlev=7)
    ref, m, counts = O.render_nn(wl.volume, tf, pyr, O.cone_params(wl.grid, wl.light()), wts, wl.camera(), w, h)
    check(img, ref, m)
    # near-tied exits may take a sample more or less
    assert abs(int(r.stats().shaded_samples) - int(counts[0])) <= 0.001 * counts[0] + 4


# (density entries, 8 or 16 bits): the smallest tables, the largest staged one, one read from memory
@pytest.mark.parametrize("entries,bits", [(2, 8), (256, 8), (4096, 16), (5000, 16)])
@pytest.mark.parametrize("n,w,h,alpha_max", SIZES + MANY)
@pytest.mark.parametrize("phong", [0, 1])
def test_plain(n, w, h, alpha_max, entries, bits, phong):
    wl = W.cone_blobs(n=n, width=w, height=h, seed=31)
    vol = wl.volume if bits == 8 else (wl.volume.astype(np.uint16) * 257)
    rgb, a = W.seeded_tf(131, 4, alpha_max=alpha_max)
    if entries == 2:
        rgb, a = rgb[[0, -1]], a[[0, -1]]
    rgb[:, 3] = np.round(rgb[:, 3] * (entries - 1) / 255)
    a[:, 1] = rgb[:, 3]
    r = N.Renderer(N.RC1P)
    r.set_volume(vol, wl.scale)
    r.set_transfer_function(rgb, a, max_density=entries - 1)
    p = r.params()
    p.apply_gradient_shading, p.shininess = phong, 20.0
    r.set_params(p)
    img = r.render(wl.camera(), w, h, light=wl.light())
    tf = O.OTF(rgb, a, max_density=entries - 1)
    if phong:
        ph = O.phong(p.gradient_type, wl.light(), ka=p.ka, kd=p.kd, ks=p.ks, shininess=p.shininess)
        ref, m = O.render_rc1p_phong(vol, tf, ph, wl.camera(), w, h)
    else:
        ref, m = O.render_rc1p(vol, tf, wl.camera(), w, h)
    check(img, ref, m)


@pytest.mark.parametrize("n,w,h,alpha_max", SIZES + MANY)
@pytest.mark.parametrize("phong", [0, 1])
def test_light_cache(n, w, h, alpha_max, phong):
    wl, tf, r, p, img = scene(N.EBS, n, w, h, alpha_max, light_cache=1, apply_phong=phong)
    g = r.light_cache()
    if phong:
        ph = O.phong(p.gradient_type, wl.light(), ka=p.ka, kd=p.kd, ks=p.ks, shininess=p.shininess)
        ref, m = O.render_lc_phong(wl.volume, tf, g, 1, 1, p.ka, p.kd, ph, wl.camera(), w, h, scale=wl.scale)
    else:
        ref, m = O.render_lc(wl.volume, tf, g, 1, 1, p.ka, p.kd, wl.camera(), w, h, scale=wl.scale)
    check(img, ref, m)


INSIDE = ((2.0, -1.0, 3.0), (0.0, 0.0, -40.0))


@pytest.mark.parametrize("phong", [0, 1])
@pytest.mark.parametrize("entries,bits", [(256, 8), (5000, 16)])
@pytest.mark.parametrize("w,h,eye,to", [(363, 362, *INSIDE), (1024, 128, *INSIDE), (400, 327, *INSIDE),
                                        (400, 330, (0.0, 0.0, 16.0), (0.0, 0.0, 0.0)),
                                        (400, 330, (0.0, 0.0, 26.0), (0.0, 0.0, 0.0)), (900, 601, (20.0, 9.0, 60.0), (0.0, 0.0, 0.0))])
def test_plain_of_full_frames(w, h, eye, to, entries, bits, phong):
    """A lane to a ray from 2^17 pixels on in frames that the volume fills: one pixel more, just as
    many, and fewer; from inside, from before a face, and from where the corners miss it; and in
    frames of many pixels for the volume's size."""
    wl = W.cone_blobs(n=24, width=w, height=h, seed=31)
    vol = wl.volume if bits == 8 else (wl.volume.astype(np.uint16) * 257)
    rgb, a = W.seeded_tf(131, 4, alpha_max=0.5)
    rgb[:, 3] = np.round(rgb[:, 3] * (entries - 1) / 255)
    a[:, 1] = rgb[:, 3]
    r = N.Renderer(N.RC1P)
    r.set_volume(vol, wl.scale)
    r.set_transfer_function(rgb, a, max_density=entries - 1)
    p = r.params()
    p.apply_gradient_shading, p.shininess = phong, 20.0
    r.set_params(p)
    r.collect_stats()
    cam, light = N.Camera(eye, to, (0.0, 1.0, 0.0), 60.0, w / h), wl.light()
    img = r.render(cam, w, h, light=light)
    tf = O.OTF(rgb, a, max_density=entries - 1)
    if phong:
        ph = O.phong(p.gradient_type, light, ka=p.ka, kd=p.kd, ks=p.ks, shininess=p.shininess)
        ref, m = O.render_rc1p_phong(vol, tf, ph, cam, w, h)
    else:
        ref, m = O.render_rc1p(vol, tf, cam, w, h)
    check(img, ref, m)


@pytest.mark.parametrize("phong", [0, 1])
def test_light_cache_of_a_full_frame(phong):
    w, h = 363, 362
    wl = W.cone_blobs(n=24, width=w, height=h, seed=31)
    rgb, a = W.seeded_tf(131, 4, alpha_max=0.5)
    r = N.Renderer(N.EBS)
    r.set_volume(wl.volume, wl.scale)
    r.set_transfer_function(rgb, a)
    r.set_params(light_cache=1, apply_phong=phong)
    p = r.params()
    cam, light = N.Camera(*INSIDE, (0.0, 1.0, 0.0), 60.0, w / h), wl.light()
    img = r.render(cam, w, h, light=light)
    tf, g = O.OTF(rgb, a), r.light_cache()
    if phong:
        ph = O.phong(p.gradient_type, light, ka=p.ka, kd=p.kd, ks=p.ks, shininess=p.shininess)
        ref, m = O.render_lc_phong(wl.volume, tf, g, 1, 1, p.ka, p.kd, ph, cam, w, h, scale=wl.scale)
    else:
        ref, m = O.render_lc(wl.volume, tf, g, 1, 1, p.ka, p.kd, cam, w, h, scale=wl.scale)
    check(img, ref, m)


def test_buffers_kept_between_volumes_hold_the_new_ones():
    """Volumes, cones and networks of changing and equal sizes through one handle, against new
    handles: what a handle keeps is of the call at hand."""
    def fresh(tech, vol, params):
        r = N.Renderer(tech)
        r.set_volume(vol, (1.0, 1.0, 1.0))
        r.set_transfer_function(*W.seeded_tf(131, 4, alpha_max=0.5))
        r.set_params(**params)
        return r

    rng = np.random.default_rng(5)
    wl = W.cone_blobs(n=24, width=40, height=30, seed=31)
    kept = {t: fresh(t, rng.integers(0, 256, (8, 8, 8), dtype=np.uint8), {}) for t in (N.DOS, N.EBS)}
    for shape in ((20, 24, 28), (20, 24, 28), (30, 10, 12), (20, 24, 28)):
        vol = rng.integers(0, 256, shape, dtype=np.uint8)
        for tech, many in ((N.DOS, [dict(apply_shadow=1, light_cache=c, sigma0=s) for c in (0, 1) for s in (1.0, 1.5)]),
                           (N.EBS, [dict(light_cache=c) for c in (0, 1)])):
            kept[tech].set_volume(vol, (1.0, 1.0, 1.0))
            kept[tech].set_transfer_function(*W.seeded_tf(131, 4, alpha_max=0.5))
            for params in many:
                kept[tech].set_params(**params)
                a = kept[tech].render(wl.camera(), 40, 30, light=wl.light())
                b = fresh(tech, vol, params).render(wl.camera(), 40, 30, light=wl.light())
                assert np.abs(a - b).max() <= 1e-6, (shape, tech, params)  # colours add up in any order
    net, w = N.Renderer(N.CONE_NN), rng.normal(0, 0.2, N.lib().cvr_nn_param_count()).astype(np.float32)
    net.nn_set_weights(w)
    for n in (64, 100, 64, 1):
        x, t = rng.random((n, 16), np.float32), rng.random((n, 2), np.float32)
        new = N.Renderer(N.CONE_NN)
        new.nn_set_weights(w)
        (la, ga), (lb, gb) = net.nn_gradient(x, t), new.nn_gradient(x, t)
        assert la == lb and np.array_equal(ga, gb)


@pytest.mark.parametrize("res", [(1, 1, 1), (5, 3, 2), (7, 11, 3), (33, 2, 4)])
@pytest.mark.parametrize("shadow_type,occ,sdw", [(0, 1, 1), (1, 1, 1), (1, 0, 1), (0, 1, 0)])
def test_light_cache_cells(res, shadow_type, occ, sdw):
    """Eight lanes to a cell: fewer cells than a workgroup's, part of the last one's, and each of
    the terms alone.  The tolerance is that of the cache's own tests."""
    wl = W.banded_noise(n=20, width=16, height=16, seed=12)
    vol = np.ascontiguousarray(wl.volume[:, :13, :9])
    r = N.Renderer(N.EBS)
    r.set_volume(vol, wl.scale)
    r.set_transfer_function(wl.rgb_iso, wl.alpha_iso)
    p = r.params()
    p.shadow_type, p.apply_occlusion, p.apply_shadow, p.light_cache = shadow_type, occ, sdw, 1
    p.light_cache_res[:] = list(res)
    r.set_params(p)
    p = r.params()
    light = wl.light()
    r.render(wl.camera(), 16, 16, light=light)
    prm = O.ebs_params(p, light)
    grid = np.array(vol.shape[::-1]) * np.array(wl.scale)
    prm.sdw_max_dist = np.float32(0.75) * np.float32(float(np.linalg.norm(grid)))
    ref = O.lc_ebs(vol.shape[::-1], wl.scale, O.sat(vol, O.OTF(wl.rgb_iso, wl.alpha_iso)), prm, res)
    d = np.abs(r.light_cache().astype(np.float64) - ref)
    assert d.max() <= 5e-4, d.max()


@pytest.mark.parametrize("bits,entries,ext", [(8, 256, 0), (8, 2, 0), (16, 256, 0), (16, 4096, 0), (16, 70000, 0), (16, 256, 1)])
def test_summed_area_table_of_each_extinction_table(bits, entries, ext):
    """The table's last cell is the sum of every voxel's extinction, each a 32-bit value of the
    table: a step of 2^-23 in one of them stands out less than 1e-6 of the sum."""
    rng = np.random.default_rng(entries)
    vol = rng.integers(0, 1 << bits, (6, 7, 8)).astype(np.uint8 if bits == 8 else np.uint16)
    rgb, a = W.seeded_tf(131, 4, alpha_max=0.9)
    if entries == 2:
        rgb, a = rgb[[0, -1]], a[[0, -1]]
    rgb[:, 3] = np.round(rgb[:, 3] * (entries - 1) / 255)
    a[:, 1] = rgb[:, 3]
    r = N.Renderer(N.EBS)
    r.set_volume(vol, (1.0, 1.0, 1.0))
    r.set_transfer_function(rgb, a, max_density=entries - 1, extinction_input=bool(ext))
    got = r.get_sat(vol.shape[::-1])
    ref = O.sat(vol, O.OTF(rgb, a, max_density=entries - 1, extinction_input=bool(ext)))
    assert np.abs(got - ref).max() <= 1e-6 * ref.max()


# the direct and the separable build of each level, flat and long grids, and a transfer function too
# large for LDS.  The tolerance is that of the pyramid's own tests.
@pytest.mark.parametrize("base,sigma0,entries,bits", [((17, 16, 15), 1.0, 256, 8), ((17, 16, 16), 1.0, 256, 16),
                                                      ((32, 32, 32), 1.0, 256, 8), ((1, 1, 1), 1.0, 256, 8),
                                                      ((70, 5, 1), 0.7, 256, 16), ((40, 33, 9), 1.3, 9000, 16),
                                                      ((64, 64, 64), 1.0, 9000, 16), ((48, 40, 36), 0.7, 9000, 8)])
def test_pyramid_shapes(base, sigma0, entries, bits):
    wl = W.plain_blobs(n=32, width=8, height=8, seed=14)
    vol = wl.volume if bits == 8 else (wl.volume.astype(np.uint16) * 257)
    rgb, a = wl.rgb_iso.copy(), wl.alpha_iso.copy()
    rgb[:, 3] = np.round(rgb[:, 3] * (entries - 1) / 255)
    a[:, 1] = np.round(a[:, 1] * (entries - 1) / 255)
    r = N.Renderer(N.CONE_TRACE)
    r.set_volume(vol)
    r.set_transfer_function(rgb, a, max_density=entries - 1)
    p = r.params()
    p.base_res[:] = list(base)
    p.sigma0, p.n_levels = sigma0, 0
    r.set_params(p)
    g = r.pyramid()
    ref = O.OPyr.build(vol, O.OTF(rgb, a, max_density=entries - 1), base=base, sigma0=sigma0)
    assert len(g) == ref.levels
    for l in range(ref.levels):
        t = ref.level(l)
        assert g[l].shape == t.shape and (np.abs(g[l] - t) / np.maximum(1.0, np.abs(t))).max() <= 1e-4, l


# The samples counted in a frame do not depend on how its rays are spread over workgroups: the shading
# queue and the light-cache march count the same frame alike, again after another frame
@pytest.mark.parametrize("w,h", [(1, 1), (97, 71), (640, 400)])
@pytest.mark.parametrize("tech", [N.EBS, N.DOS])
def test_counted_samples(tech, w, h):
    counts = []
    for cached in (0, 1):
        wl, tf, r, p, img = scene(tech, 24, w, h, 0.3, light_cache=cached)
        s = r.stats()
        counts.append((s.samples, s.shaded_samples))
        r.render(wl.camera(), 2 * w, h, light=wl.light())
        r.render(wl.camera(), w, h, light=wl.light())
        s = r.stats()
        counts.append((s.samples, s.shaded_samples))
    assert counts[0][0] > 0 and len(set(counts)) == 1, counts


# From inside a volume that is dense on one side and clear on the other: tiles of 64 x 64 pixels whose rays end
# after a few samples are dealt out apart from the others.  One tile, ragged ones, a frame too small to be
# looked over, 4 and 16 rays to a wavefront for the other tiles.
@pytest.mark.parametrize("w,h", [(64, 64), (65, 130), (200, 71), (63, 90), (300, 260)])
@pytest.mark.parametrize("tech", [N.CONE_TRACE, N.DOS, N.CONE_GT, N.EBS])
def test_tiles_of_short_rays(tech, w, h):
    n = 40
    vol = np.zeros((n, n, n), np.uint8)
    vol[:, :, : n // 2] = 200
    vol[:, :, n // 2:] = np.linspace(0, 60, n, dtype=np.uint8)[:, None, None]
    rgb = np.array([[0.2, 0.5, 0.9, 0], [0.9, 0.6, 0.3, 255]])
    alpha = np.array([[0.0, 0], [0.0, 50], [0.1, 60], [0.9, 150], [0.95, 255]])
    grid = (float(n),) * 3
    r = N.Renderer(tech)
    r.set_volume(vol)
    r.set_transfer_function(rgb, alpha)
    light = W.light_from_direction((0.3, 0.8, -0.4), grid)
    if tech == N.DOS:
        r.set_params(apply_shadow=1, shadow_type=2)
    elif tech == N.CONE_GT:
        r.set_params(occ_rays=3, sdw_rays=2, shadow_type=2)
    cam, tf = W.orbit_camera(grid, w, h, az_deg=4.0, el_deg=3.0, dist_diag=0.02, fovy=70.0), O.OTF(rgb, alpha)
    img = r.render(cam, w, h, light=light)
    s = 3
    if tech == N.EBS:
        prm = O.ebs_params(r.params(), light)
        prm.sdw_max_dist = np.float32(0.75) * np.float32(np.linalg.norm(grid))
        ref, m = O.render_ebs(vol, tf, O.sat(vol, tf), prm, cam, w, h, stride=s)
    elif tech == N.CONE_GT:
        ref, m = O.render_gt(vol, tf, O.gt_params(r.params(), grid, light), cam, w, h, stride=s)
    else:
        pyr = O.OPyr.wrap(grid, [a.astype(np.float64) for a in r.pyramid()])
        if tech == N.DOS:
            ref, m = O.render_dos(vol, tf, pyr, O.dos_params(r.params(), grid, light), cam, w, h, stride=s)
        else:
            ref, m = O.render_cone(vol, tf, pyr, O.cone_params(grid, light), cam, w, h, stride=s)
    assert ref[::s, ::s, 3].max() > 0.98 and ref[::s, ::s, 3].min() < 0.5
    sparse = np.zeros_like(img)
    sparse[::s, ::s] = img[::s, ::s]
    st = O.compare(sparse, ref, m, 2e-3, s)
    assert st["max_abs"] <= 2e-3 and st["n_over_tol"] <= 0.005 * st["n_pixels"] + 1, st
    r.collect_stats(True)
    again = r.render(cam, w, h, light=light)
    assert np.array_equal(again, img) and r.stats().shaded_samples > 0
