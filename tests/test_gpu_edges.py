"""Calls at the edges of what the entry points accept, against the FP64 oracle."""
import numpy as np
import pytest

import oracle_lib as O
from cpp_volume_rendering_amd import native as N
from cpp_volume_rendering_amd import workloads as W

pytestmark = pytest.mark.gpu
TOL = 2e-3


def handle(tech, wl, **params):
    r = N.Renderer(tech)
    r.set_volume(wl.volume, wl.scale)
    r.set_transfer_function(wl.rgb_iso, wl.alpha_iso)
    if params:
        r.set_params(**params)
    return r


def check(img, ref, m, stride=1):
    s = O.compare(img, ref, m, TOL, stride)
    print(s)
    assert s["max_abs"] <= TOL, s
    assert s["n_over_tol"] <= 0.005 * s["n_pixels"] + 1, s


# a point past each face, past an edge and past a corner, a point on a face and one inside, with cones that
# lead into the box, along the face and away from it; one point a call and 64 of them, whose lanes all
# begin outside.  The tolerance is that of the points inside.
@pytest.mark.parametrize("copies", [1, 64])
@pytest.mark.parametrize("pos", [(-6, 30, 30), (70, 30, 30), (30, -3, 31), (30, 66, 33), (30, 30, -9), (33, 30, 67.5),
                                 (-4, -5, 30), (69, 68, 70), (0, 30, 30), (30, 64, 30), (20, 41, 30)])
def test_cone_points_outside_the_box(pos, copies):
    wl = W.cone_blobs(n=64, width=8, height=8)
    r = handle(N.CONE_TRACE, wl)
    pyr = O.OPyr.wrap(wl.grid, [a.astype(np.float64) for a in r.pyramid()])
    inwards = np.array([32.0, 31.0, 33.0]) - pos
    for light in (inwards, -inwards, np.array([0.3, 0.9, -0.2])):
        light = light / np.linalg.norm(light)
        at, d, li = (np.tile(v, (copies, 1)).astype(np.float32) for v in (np.array(pos, np.float64), -inwards, light))
        occ, sdw, feat = r.cone_eval(at, d, li)
        prm = O.cone_params(wl.grid, light_fwd=light)
        ro, rs, rf = O.cone_points(pyr, prm, at, d)
        for a, b in ((occ, ro), (sdw, rs), (feat, rf)):
            assert np.abs(a - b).max() <= 2e-4


# a threshold below 0 ends a ray with its first opaque sample, whatever came before it
@pytest.mark.parametrize("et", [-1.0, 0.0])
@pytest.mark.parametrize("tech,cached", [(N.EBS, 0), (N.EBS, 1), (N.CONE_TRACE, 0), (N.CONE_NN, 0)])
def test_threshold_not_above_zero(tech, cached, et):
    wl = W.cone_blobs(n=64, width=48, height=37, seed=15)
    wl.rgb_iso, wl.alpha_iso = W.seeded_tf(131, 4)
    wl.alpha_iso[1, 0] = 0.0  # rays of more than 64 transparent samples before the first opaque one
    r, cam, light = handle(tech, wl), wl.camera(), wl.light()
    p = r.params()
    if tech == N.CONE_NN:
        p.cone.et_threshold = et
        wts = np.random.default_rng(3).normal(0, 0.1, N.lib().cvr_nn_param_count()).astype(np.float32)
        r.nn_set_weights(wts)
    else:
        p.et_threshold = et
        if tech == N.EBS:
            p.light_cache = cached
    r.set_params(p)
    if tech == N.CONE_NN:
        r.nn_set_weights(wts)
    img = r.render(cam, 48, 37, light=light)
    tf = O.OTF(wl.rgb_iso, wl.alpha_iso)
    if tech == N.EBS and cached:
        ref, m = O.render_lc(wl.volume, tf, r.light_cache(), 1, 1, p.ka, p.kd, cam, 48, 37, et=et, scale=wl.scale)
    elif tech == N.EBS:
        prm = O.ebs_params(p, light)
        prm.sdw_max_dist = np.float32(0.75) * np.float32(np.linalg.norm(wl.grid))
        ref, m = O.render_ebs(wl.volume, tf, O.sat(wl.volume, tf), prm, cam, 48, 37, et=et)
    else:
        pyr = O.OPyr.wrap(wl.grid, [a.astype(np.float64) for a in r.pyramid()])
        prm = O.cone_params(wl.grid, light)
        if tech == N.CONE_TRACE:
            ref, m = O.render_cone(wl.volume, tf, pyr, prm, cam, 48, 37, et=et)
        else:
            ref, m, _ = O.render_nn(wl.volume, tf, pyr, prm, wts, cam, 48, 37, et=et)
    assert 0 < ref[..., 3].max() < 0.5
    # the margin is the oracle's distance of an opacity from the threshold: none is near one below 0
    check(img, ref, m if et > 0 else None)


def test_frame_of_more_lanes_than_a_launch_may_have():
    """8192 x 8192 pixels of the ground truth, 64 lanes a pixel, in two launches: rows on both sides of
    where the second begins, against the oracle."""
    import torch

    w = h = 8192
    wl = W.cone_blobs(n=24, width=w, height=h, seed=31)
    r = handle(N.CONE_GT, wl, occ_rays=2, sdw_rays=1, shadow_type=2)
    out = torch.full((h, w, 4), -1.0, device="cuda:0")
    r.render(wl.camera(), w, h, light=wl.light(), out=out)
    torch.cuda.synchronize()
    assert float(out.min()) >= 0.0  # every pixel written
    tf = O.OTF(wl.rgb_iso, wl.alpha_iso)
    ref, m = O.render_gt(wl.volume, tf, O.gt_params(r.params(), wl.grid, wl.light()), wl.camera(), w, h, stride=64)
    img = np.zeros((h, w, 4), np.float32)
    img[::64, ::64] = out[::64, ::64].cpu().numpy()
    assert ref[:h // 2, ..., 3].max() > 0.2 and ref[h // 2:, ..., 3].max() > 0.2
    check(img, ref, m, 64)


@pytest.mark.parametrize("edit", ["transfer function", "weights", "checkpoint", "gradient"])
def test_edits_wait_for_frames_in_flight(edit):
    """An edit right after a frame of some milliseconds was queued on a non-blocking stream: the frame is the
    one drawn before the edit, bit for bit (the shared colour sums of a pixel come in any order: to
    rounding)."""
    import torch

    w = h = 1024
    wl = W.cone_blobs(n=96, width=w, height=h, seed=7)
    cam, light = wl.camera(), wl.light()
    if edit in ("weights", "checkpoint"):
        r, rng = handle(N.CONE_NN, wl), np.random.default_rng(5)
        wa, wb = (rng.normal(0, 0.1, N.lib().cvr_nn_param_count()).astype(np.float32) for _ in range(2))
        r.nn_set_weights(wb)
        r.prepare()
        other = r.nn_save()
        r.nn_set_weights(wa)
    elif edit == "gradient":
        r = handle(N.RC1P, wl, apply_gradient_shading=1, step_size=0.01, et_threshold=1.0)
    else:
        r = handle(N.CONE_TRACE, wl)
    r.prepare()
    s = torch.cuda.Stream()
    before, out = (torch.zeros((h, w, 4), device="cuda:0") for _ in range(2))
    torch.cuda.synchronize()
    r.render(cam, w, h, light=light, out=before, stream=s.cuda_stream)
    torch.cuda.synchronize()
    r.render(cam, w, h, light=light, out=out, stream=s.cuda_stream)
    if edit == "transfer function":
        r.set_transfer_function(wl.rgb_iso[:, [1, 2, 0, 3]], wl.alpha_iso * [0.1, 1.0])
    elif edit == "weights":
        r.nn_set_weights(wb)
    elif edit == "checkpoint":
        r.nn_load(other)
    else:
        r.gradient(wl.volume.shape, N.GRADIENT_FINITE_DIFF)
    torch.cuda.synchronize()
    # sums of a thousand samples' colours below 1 in another order: 1000 x 2^-24 at most
    assert float((out - before).abs().max()) <= 6e-5
    if edit != "gradient":
        r.render(cam, w, h, light=light, out=out, stream=s.cuda_stream)
        torch.cuda.synchronize()
        assert float((out - before).abs().max()) > 1e-3  # the edit is in force


def test_volume_that_is_refused_leaves_none():
    """A volume too deep for its corner blocks is refused, and so is a frame after it; the next volume is
    drawn."""
    wl = W.cone_blobs(n=16, width=8, height=8)
    r = handle(N.RC1P, wl)
    deep = np.full((65536, 1, 1), 200, np.uint8)
    with pytest.raises(N.CvrError):
        r.set_volume(deep)
    with pytest.raises(N.CvrError) as e:
        r.render(wl.camera(), 8, 8)
    assert e.value.code == N.ERR_STATE
    r.set_volume(wl.volume, wl.scale)
    assert r.render(wl.camera(), 8, 8)[..., 3].max() > 0.1


def test_pyramid_of_more_workgroups_than_a_launch_may_have():
    """A pyramid of 2^24 workgroups of corner blocks, in three launches: cones around where the second and
    the third begin, and in the first and last slices."""
    vol = W.cone_blobs(n=64, width=8, height=8).volume[:, 16:32, 30:34].copy()
    grid = (4.0, 16.0, 64.0)
    r = N.Renderer(N.CONE_TRACE)
    r.set_volume(vol)
    r.set_transfer_function(*W.seeded_tf(103, 4))
    p = r.params()
    p.base_res[:], p.n_levels = [1, 1025, 65535], 2
    r.set_params(p)
    pyr = O.OPyr.wrap(grid, [a.astype(np.float64) for a in r.pyramid()])
    per = 257  # workgroups of a slice
    z = np.array([0.01, (1 << 23) / per / 65535 * 64, (1 << 24) / per / 65535 * 64, 63.99, 40.0])
    rng = np.random.default_rng(3)
    pos = np.column_stack([rng.uniform(0.5, 3.5, 40), rng.uniform(1, 15, 40), np.tile(z, 8)])
    d = rng.normal(0, 1, (40, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    light = np.array([0.3, 0.2, 0.9]) / np.linalg.norm([0.3, 0.2, 0.9])
    pos, d, li = (np.ascontiguousarray(v, np.float32) for v in (pos, d, np.tile(light, (40, 1))))
    occ, sdw, feat = r.cone_eval(pos, d, li)
    ro, rs, rf = O.cone_points(pyr, O.cone_params(grid, light_fwd=light), pos, d)
    assert ro.min() < 0.9
    for a, b in ((occ, ro), (sdw, rs), (feat, rf)):
        assert np.abs(a - b).max() <= 2e-4


@pytest.mark.parametrize("sizes", [(100, 700, 100, 3000, 64), (5000, 1, 700)])
def test_gradient_of_changing_sample_counts(sizes):
    """Calls of one handle with more and with fewer samples than before: each as a handle's first call,
    which takes other buffers."""
    rng = np.random.default_rng(9)
    w = rng.normal(0, 0.2, N.lib().cvr_nn_param_count()).astype(np.float32)
    kept = N.Renderer(N.CONE_NN)
    kept.nn_set_weights(w)
    for n in sizes:
        X, T = rng.random((n, 16)).astype(np.float32), rng.normal(0, 0.1, (n, 2)).astype(np.float32)
        own = N.Renderer(N.CONE_NN)
        own.nn_set_weights(w)
        (la, ga), (lb, gb) = kept.nn_gradient(X, T), own.nn_gradient(X, T)
        assert la == lb and np.array_equal(ga, gb)


def test_training_and_first_frame_on_a_non_blocking_stream():
    """Optimiser state and second-pass marks are cleared on the call's stream: the network trained there and
    its first frame, some of whose samples leave the training range, are the null stream's bit for bit
    (colours to the rounding of their sums)."""
    import torch

    wl = W.cone_blobs(n=40, width=96, height=80, seed=21)
    out, weights, images = torch.zeros((80, 96, 4), device="cuda:0"), [], []
    for stream in (None, torch.cuda.Stream().cuda_stream):
        r = handle(N.CONE_NN, wl)
        p = r.params()
        p.n_train, p.n_val, p.batch, p.epochs, p.rmse_gate, p.ood_margin = 4096, 1024, 1024, 4, 10.0, -0.02
        r.set_params(p)
        torch.cuda.synchronize()
        r.nn_train(stream=stream)
        r.render(wl.camera(), 96, 80, light=wl.light(), out=out, stream=stream)
        torch.cuda.synchronize()
        weights.append(r.nn_weights())
        images.append(out.clone())
        r.collect_stats(True)
        r.render(wl.camera(), 96, 80, light=wl.light(), out=out, stream=stream)
        assert r.stats().fallback_samples > 0
    assert np.array_equal(weights[0], weights[1])
    assert float((images[0] - images[1]).abs().max()) <= 2e-5  # 300 samples of colours below 1: 300 x 2^-24


@pytest.mark.parametrize("tech,params", [(N.RC1P, {}), (N.RC1P, {"apply_gradient_shading": 1}), (N.EBS, {"light_cache": 1}),
                                         (N.EBS, {}), (N.CONE_TRACE, {})])
@pytest.mark.parametrize("w,h", [(90, 70), (900, 700)])
def test_colours_of_transparent_entries_do_not_count(tech, params, w, h):
    """Entries that are fully transparent, and no opaque sample's neighbours, may hold any colour: NaN gives
    the frame that 0 gives (bit for bit where a pixel's sum has one order)."""
    wl = W.cone_blobs(n=32, width=w, height=h, seed=12)
    frames = []
    for colour in (0.0, float("inf")):  # the table is NaN between an infinite point and the next
        wl.rgb_iso = np.array([[colour] * 3 + [0], [0.6, 0.4, 0.7, 20], [0.9, 0.3, 0.5, 255]])
        wl.alpha_iso = np.array([[0, 0], [0, 40], [0.3, 130], [0.8, 255]])
        frames.append(handle(tech, wl, **params).render(wl.camera(), w, h, light=wl.light()))
    assert frames[0][..., 3].max() > 0.3
    assert np.isfinite(frames[1]).all()
    assert np.abs(frames[0] - frames[1]).max() <= (1e-5 if tech == N.CONE_TRACE or not params else 0.0)


def test_new_jobs_wait_for_the_images_in_flight():
    """New jobs right after a batch was queued on a non-blocking stream, drawn on another into another
    buffer: the first images are those of the first jobs."""
    import torch

    wl = W.cone_blobs(n=64, width=256, height=256, seed=8)
    r = handle(N.CONE_NN, wl)
    r.nn_set_weights(np.random.default_rng(2).normal(0, 0.1, N.lib().cvr_nn_param_count()).astype(np.float32))
    r.prepare()
    b = N.Batch(256, 256)
    m = b.add_volume(r)
    jobs = [[(m, wl.camera(az, 10.0), wl.light()) for az in range(a, a + 32)] for a in (0, 180)]
    s, t = torch.cuda.Stream(), torch.cuda.Stream()
    out = torch.zeros((4, 32, 256, 256, 4), device="cuda:0")
    torch.cuda.synchronize()
    for k in (0, 1):
        b.set_jobs(jobs[k])
        b.render(out[k], stream=s.cuda_stream)
        torch.cuda.synchronize()
    b.set_jobs(jobs[0])
    b.render(out[2], stream=s.cuda_stream)
    torch.cuda.synchronize()
    b.render(out[2], stream=s.cuda_stream)
    b.set_jobs(jobs[1])
    b.render(out[3], stream=t.cuda_stream)
    torch.cuda.synchronize()
    assert float((out[0] - out[1]).abs().max()) > 0.1
    assert float((out[2:] - out[:2]).abs().max()) <= 2e-5  # the order of a pixel's sums: 300 x 2^-24


@pytest.mark.parametrize("tech", [N.CONE_TRACE, N.DOS])
@pytest.mark.parametrize("fwd", [(0.0, 1.0, 0.0), (-0.0, -1.0, 0.0), (0.0, 0.0, 1.0), (1.0, 0.0, -0.0)])
def test_lights_along_an_axis(tech, fwd):
    wl = W.cone_blobs(n=48, width=40, height=33, seed=17)
    cam, light = wl.camera(), W.light_from_direction(fwd, wl.grid)
    light.forward[:] = fwd
    r = handle(tech, wl)
    if tech == N.DOS:
        r.set_params(apply_shadow=1, shadow_type=2)
    img = r.render(cam, 40, 33, light=light)
    tf = O.OTF(wl.rgb_iso, wl.alpha_iso)
    pyr = O.OPyr.wrap(wl.grid, [a.astype(np.float64) for a in r.pyramid()])
    if tech == N.DOS:
        ref, m = O.render_dos(wl.volume, tf, pyr, O.dos_params(r.params(), wl.grid, light), cam, 40, 33)
    else:
        ref, m = O.render_cone(wl.volume, tf, pyr, O.cone_params(wl.grid, light), cam, 40, 33)
    assert ref[..., 3].max() > 0.3
    check(img, ref, m)


def test_volume_of_more_than_4_gib_of_corner_blocks():
    """64-bit block offsets, which volumes from 4 GiB of blocks on take: the camera rays of the plain march
    (lane groups) and of the queue, and light rays, against the oracle."""
    nx, ny, nz = 840, 830, 784
    ax = [np.sin(np.linspace(0, k * np.pi, n)) ** 2 for n, k in ((nx, 3), (ny, 2), (nz, 5))]
    vol = (255.0 * ax[2][:, None, None]).astype(np.float32) * ax[1][:, None].astype(np.float32) * ax[0].astype(np.float32)
    vol = vol.astype(np.uint8)
    assert vol.size * 8 > 1 << 32
    grid, tf = (float(nx), float(ny), float(nz)), W.seeded_tf(107, 4)
    tf[1][:, 0] *= 0.02  # rays go far into the volume
    w, h = 24, 18
    cam, light, otf = W.orbit_camera(grid, w, h, dist_diag=0.9), W.light_from_direction((-0.4, 0.7, 0.6), grid), O.OTF(*tf)
    for tech in (N.RC1P, N.CONE_GT):
        r = N.Renderer(tech)
        r.set_volume(vol)
        r.set_transfer_function(*tf)
        if tech == N.CONE_GT:
            r.set_params(occ_rays=1, sdw_rays=1, shadow_type=2, occ_max_dist=40.0, sdw_max_dist=40.0)
        img = r.render(cam, w, h, light=light)
        if tech == N.RC1P:
            ref, m = O.render_rc1p(vol, otf, cam, w, h)
        else:
            ref, m = O.render_gt(vol, otf, O.gt_params(r.params(), grid, light), cam, w, h)
        assert ref[..., 3].max() > 0.3
        check(img, ref, m)


# 2112 x 2112: a lane to a ray, and with a table that leaves no room for that 16 rays to a wavefront, of which
# more workgroups than there are marks (each takes two sets); from inside with a lane to a ray, a ragged frame
@pytest.mark.parametrize("w,h,entries,dist", [(2112, 2112, 256, 2.0), (2112, 2112, 1024, 2.0), (701, 645, 256, 0.1)])
def test_surrogate_frames_of_many_pixels(w, h, entries, dist):
    """The network's frame against the oracle, the frame of the second pass alone against the cone tracer's,
    and the first again when no mark is left."""
    wl = W.cone_blobs(n=24, width=w, height=h, seed=33)
    md, light = entries - 1, wl.light()
    rgb, al = wl.rgb_iso.copy(), wl.alpha_iso.copy()
    rgb[:, 3], al[:, 1] = np.floor(rgb[:, 3] * md / 255), np.floor(al[:, 1] * md / 255)
    cam = W.orbit_camera(wl.grid, w, h, dist_diag=dist)
    r, c = N.Renderer(N.CONE_NN), N.Renderer(N.CONE_TRACE)
    for x in (r, c):
        x.set_volume(wl.volume)
        x.set_transfer_function(rgb, al, max_density=md)
    p = r.params()
    p.cone.density_precision = 0
    r.set_params(p)
    c.set_params(p.cone)
    wts = np.random.default_rng(4).normal(0, 0.1, N.lib().cvr_nn_param_count()).astype(np.float32)
    r.nn_set_weights(wts)
    first = r.render(cam, w, h, light=light)
    pyr = O.OPyr.wrap(wl.grid, [a.astype(np.float64) for a in r.pyramid()])
    tf, s = O.OTF(rgb, al, max_density=md), 33 if w > 1000 else 11
    ref, m, _ = O.render_nn(wl.volume, tf, pyr, O.cone_params(wl.grid, light), wts, cam, w, h, stride=s)
    img = np.zeros_like(first)
    img[::s, ::s] = first[::s, ::s]
    assert ref[: h // 2, ..., 3].max() > 0.2 and ref[h // 2:, ..., 3].max() > 0.2
    check(img, ref, m, s)
    p.ood_margin = -2e30  # no input is in range
    r.set_params(p)
    r.collect_stats(True)
    exact = r.render(cam, w, h, light=light)
    st = r.stats()
    assert st.fallback_samples == st.shaded_samples > 0
    assert np.abs(exact - c.render(cam, w, h, light=light)).max() <= 2e-5
    p.ood_margin = 0.02
    r.set_params(p)
    assert np.array_equal(r.render(cam, w, h, light=light), first) and r.stats().fallback_samples == 0


def test_gradient_of_more_samples_than_the_kept_buffer_holds():
    """940032 samples (64.5 MiB) go through device buffers: the mean of the halves' gradients.  Sums of 14688
    slabs of one sign in any order: 14688 x 2^-24 of the largest at most."""
    rng, half = np.random.default_rng(6), 470016
    r = N.Renderer(N.CONE_NN)
    r.nn_set_weights(rng.normal(0, 0.2, N.lib().cvr_nn_param_count()).astype(np.float32))
    X, T = rng.random((2 * half, 16), np.float32), np.full((2 * half, 2), 2.0, np.float32)
    assert X.nbytes + T.nbytes > 64 << 20
    (l, g), (la, ga), (lb, gb) = r.nn_gradient(X, T), r.nn_gradient(X[:half], T[:half]), r.nn_gradient(X[half:], T[half:])
    assert abs(l - 0.5 * (la + lb)) <= 9e-4 * l
    assert np.abs(g - 0.5 * (ga + gb)).max() <= 9e-4 * np.abs(g).max()


@pytest.mark.parametrize("tech,entries", [(N.CONE_TRACE, 4096), (N.DOS, 4096), (N.CONE_GT, 4096), (N.EBS, 4096), (N.CONE_NN, 2048)])
def test_largest_transfer_functions(tech, entries):
    """The tables of most entries beside the queues in LDS."""
    wl = W.cone_blobs(n=32, width=40, height=33, seed=19)
    cam, light, md = wl.camera(), wl.light(), entries - 1
    rgb, al = W.seeded_tf(119, 5, max_density=md)
    r = N.Renderer(tech)
    r.set_volume(wl.volume)
    r.set_transfer_function(rgb, al, max_density=md)
    wts = np.random.default_rng(5).normal(0, 0.1, N.lib().cvr_nn_param_count()).astype(np.float32)
    if tech == N.CONE_NN:
        p = r.params()
        p.cone.density_precision = 0
        r.set_params(p)
        r.nn_set_weights(wts)
    elif tech == N.DOS:
        r.set_params(apply_shadow=1, shadow_type=2)
    elif tech == N.CONE_GT:
        r.set_params(occ_rays=4, sdw_rays=2, shadow_type=2)
    img = r.render(cam, 40, 33, light=light)
    tf = O.OTF(rgb, al, max_density=md)
    if tech == N.EBS:
        prm = O.ebs_params(r.params(), light)
        prm.sdw_max_dist = np.float32(0.75) * np.float32(np.linalg.norm(wl.grid))
        ref, m = O.render_ebs(wl.volume, tf, O.sat(wl.volume, tf), prm, cam, 40, 33)
    elif tech == N.CONE_GT:
        ref, m = O.render_gt(wl.volume, tf, O.gt_params(r.params(), wl.grid, light), cam, 40, 33)
    else:
        pyr = O.OPyr.wrap(wl.grid, [a.astype(np.float64) for a in r.pyramid()])
        if tech == N.DOS:
            ref, m = O.render_dos(wl.volume, tf, pyr, O.dos_params(r.params(), wl.grid, light), cam, 40, 33)
        elif tech == N.CONE_TRACE:
            ref, m = O.render_cone(wl.volume, tf, pyr, O.cone_params(wl.grid, light), cam, 40, 33)
        else:
            ref, m, _ = O.render_nn(wl.volume, tf, pyr, O.cone_params(wl.grid, light), wts, cam, 40, 33)
    assert ref[..., 3].max() > 0.3
    check(img, ref, m)


def test_noalloc_of_a_closed_gate_from_inside_allocates_nothing():
    """The exact tracer's frame from inside looks for tiles of short rays in a buffer that is not there yet:
    the call goes without, and gives the frame that cvr_render gives with it."""
    import torch

    w = h = 256
    wl = W.cone_blobs(n=32, width=w, height=h, seed=3)
    wl.alpha_iso[:, 0] = 0.9  # dense: every tile is short
    cam, light = W.orbit_camera(wl.grid, w, h, dist_diag=0.05), wl.light()
    r = handle(N.CONE_NN, wl)
    p = r.params()
    p.force_exact = 1
    r.set_params(p)
    r.nn_set_weights(np.zeros(N.lib().cvr_nn_param_count(), np.float32))
    r.prepare()
    got, ref = (torch.zeros((h, w, 4), device="cuda:0") for _ in range(2))
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    r.render_noalloc(cam, w, h, got, light=light)
    torch.cuda.synchronize()
    assert torch.cuda.mem_get_info()[0] == free
    r.render(cam, w, h, light=light, out=ref)
    torch.cuda.synchronize()
    # a pixel's samples are summed by four wavefronts, or by one: 30 colours of at most 1, 30 x 2^-24
    assert float(ref[..., 3].max()) > 0.9 and float((got - ref).abs().max()) <= 2e-6


def test_captured_frame_from_inside_outlives_larger_ones():
    """A captured frame keeps the buffer in which it looks for tiles of short rays: a larger frame, drawn
    between its replays, takes no new one."""
    import torch

    w, h = 300, 260
    wl = W.cone_blobs(n=32, width=w, height=h, seed=3)
    wl.alpha_iso[:, 0] = 0.9  # dense: every tile is short
    light, fill = wl.light(), torch.empty(4 << 20, device="cuda:0")
    r = handle(N.CONE_TRACE, wl)
    eager, got = (torch.zeros((h, w, 4), device="cuda:0") for _ in range(2))
    cam = W.orbit_camera(wl.grid, w, h, dist_diag=0.05)
    r.render(cam, w, h, light=light, out=eager)
    torch.cuda.synchronize()
    s, g = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        r.render(cam, w, h, light=light, out=got, stream=s.cuda_stream)
    large = torch.zeros((4 * h, 4 * w, 4), device="cuda:0")
    for _ in range(3):
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info()[0]
        r.render(W.orbit_camera(wl.grid, 4 * w, 4 * h, dist_diag=0.05), 4 * w, 4 * h, light=light, out=large)
        torch.cuda.synchronize()
        assert torch.cuda.mem_get_info()[0] == free
        fill.fill_(float("nan"))
        got.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, eager) and float(eager[..., 3].max()) > 0.9
