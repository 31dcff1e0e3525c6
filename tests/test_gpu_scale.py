"""Parity of the GPU multi-scale output resampling (cvr_resample_frame) against the FP64
oracle, for every mode and kernel, on ragged sizes (the digital filter's short-sequence
path included), and on a rendered frame."""
import numpy as np
import pytest
import torch

import oracle_lib as O
from cpp_volume_rendering_amd import native as N
from cpp_volume_rendering_amd import workloads as W

pytestmark = pytest.mark.gpu


def run(frame, dw, dh, mode, kernel, in_place=False):
    src = torch.from_numpy(np.ascontiguousarray(frame, dtype=np.float32)).cuda()
    dst = torch.zeros((dh, dw, 4), dtype=torch.float32, device="cuda")
    work = None
    if mode == N.SCALE_UPSCALE and kernel >= N.FILTER_CARDINAL_BSPLINE3:
        work = src if in_place else torch.empty_like(src)
    N.resample_frame(src, dst, mode, kernel, work=work)
    torch.cuda.synchronize()
    return dst.cpu().numpy(), src.cpu().numpy()


CASES = [(N.SCALE_MULTISAMPLE, 64, 48, 32, 24), (N.SCALE_DOWNSCALE, 66, 50, 33, 25), (N.SCALE_DOWNSCALE, 96, 72, 24, 18),
         (N.SCALE_UPSCALE, 33, 25, 66, 50), (N.SCALE_UPSCALE, 20, 15, 80, 60), (N.SCALE_UPSCALE, 7, 5, 21, 15)]


@pytest.mark.parametrize("kernel", range(6))
@pytest.mark.parametrize("mode,sw,sh,dw,dh", CASES)
def test_resample_matches_fp64(mode, sw, sh, dw, dh, kernel):
    f = np.random.default_rng(sw * 7 + kernel).uniform(0, 1, (sh, sw, 4))
    got, src_after = run(f, dw, dh, mode, kernel)
    ref = O.resample(f.astype(np.float32), dw, dh, mode, kernel)
    err = np.abs(got - ref).max()
    scale = max(1.0, np.abs(ref).max())
    print(mode, kernel, err)
    assert err <= 2e-5 * scale
    assert np.array_equal(src_after, f.astype(np.float32))  # the source is left alone


def weights(n, d, kernel):
    """(d, n) weights of a downscale along one axis: tap positions in 32 bits, as the frame
    filter has them (they lose size * 2^-24 of a tap's width), the kernel in 64."""
    f4 = np.float32
    x = (np.arange(d, dtype=f4) + f4(0.5)) / f4(d)
    x = (x[:, None] - (np.arange(n, dtype=f4) + f4(0.5))[None, :] / f4(n)) * f4(d)
    if kernel == N.FILTER_BOX:
        return ((x > -0.5) & (x <= 0.5)).astype(np.float64)
    x = np.abs(x.astype(np.float64))
    u, v = 2 - x, 1 - x
    outer, inner = {3: ((7 / 18 * u - 1 / 3) * u * u, ((-7 / 6 * v + 1.5) * v + 0.5) * v + 1 / 18),
                    4: (u ** 3, ((-3 * v + 3) * v + 3) * v + 1),
                    5: ((0.875 * u * u + 0.125) * u, ((-2.625 * v + 2.625) * v + 2.25) * v + 1)}[kernel]
    return np.where(x > 2, 0, np.where(x > 1, outer, inner))


def solve(f, kernel):
    """The digital filter along axis 0 in 64 bits, truncated factors and short sequences included."""
    a, m = ((4.0, 8) if kernel == 4 else (3.25, 9))
    L = [1 / (a + 1)]
    while len(L) < m:
        L.append(1 / (a - L[-1]))
    n = len(f)
    while len(f) <= m:
        f = np.concatenate([f, f[::-1]])
    f = f.copy()
    for i in range(1, len(f)):
        f[i] -= L[min(i, m) - 1] * f[i - 1]
    f[-1] *= L[-1] / (1 + L[-1])
    for i in range(len(f) - 2, -1, -1):
        f[i] = L[min(i, m - 1)] * (f[i] - f[i + 1])
    return f[:n]


# The digital filter's chunks (8 elements a lane: rows of 512, columns of 128), rows and
# columns just above the short path, frames narrower than a wavefront's columns, and kernel
# supports that fit the staged weights or not.  Each output is a sum of about 16 weighted taps of
# values below 1 followed by two passes of a recurrence that at most doubles an error: 1e-5
# is about 40 rounding errors of the result.
@pytest.mark.parametrize("kernel", [0, 3, 4, 5])
@pytest.mark.parametrize("sw,sh,dw,dh", [(10, 11, 10, 11), (511, 127, 511, 127), (512, 128, 512, 128),
                                         (513, 129, 513, 129), (3, 300, 3, 300), (1037, 1, 1037, 1), (65, 1, 9, 1),
                                         (300, 290, 37, 10), (290, 300, 9, 37)])
def test_downscale_at_the_edges_of_its_tiles(sw, sh, dw, dh, kernel):
    f = np.random.default_rng(sw * 11 + kernel).uniform(0, 1, (sh, sw, 4))
    got, _ = run(f, dw, dh, N.SCALE_DOWNSCALE, kernel)
    ref = np.einsum("ai,bj,ijc->abc", weights(sh, dh, kernel), weights(sw, dw, kernel), f.astype(np.float32).astype(np.float64),
                    optimize=True) * (dh / sh) * (dw / sw)
    if kernel >= N.FILTER_CARDINAL_BSPLINE3:
        ref = solve(solve(ref.swapaxes(0, 1), kernel).swapaxes(0, 1), kernel)
    assert np.abs(got - ref).max() <= 1e-5 * max(1.0, np.abs(ref).max())


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan])
def test_values_that_are_not_finite_spread_as_in_a_serial_filter(value):
    f = np.random.default_rng(3).uniform(0, 1, (140, 530, 4))
    f[60, 270, 1] = value
    got, _ = run(f, 530, 140, N.SCALE_UPSCALE, N.FILTER_CARDINAL_BSPLINE3)
    ref = O.resample(f.astype(np.float32), 530, 140, N.SCALE_UPSCALE, N.FILTER_CARDINAL_BSPLINE3)
    assert np.array_equal(np.isfinite(got), np.isfinite(ref)) and np.array_equal(np.isnan(got), np.isnan(ref))


def test_upscale_in_place_filters_the_source():
    f = np.random.default_rng(9).uniform(0, 1, (24, 32, 4))
    got, src_after = run(f, 64, 48, N.SCALE_UPSCALE, N.FILTER_CARDINAL_BSPLINE3, in_place=True)
    ref = O.resample(f.astype(np.float32), 64, 48, N.SCALE_UPSCALE, N.FILTER_CARDINAL_BSPLINE3)
    assert np.abs(got - ref).max() <= 2e-5
    assert not np.array_equal(src_after, f.astype(np.float32))


def test_render_at_twice_the_screen_then_downscale():
    wl = W.plain_blobs(n=64, width=128, height=96, seed=51)
    fw, fh = N.multiscale_size(128, 96, 2, 2)
    assert (fw, fh) == (256, 192)
    assert N.multiscale_size(128, 96, -2, -3) == (64, 32)
    r = N.Renderer(N.RC1P)
    r.set_volume(wl.volume)
    r.set_transfer_function(wl.rgb_iso, wl.alpha_iso)
    cam = W.orbit_camera(wl.grid, fw, fh, 30.0, 20.0)
    frame = torch.zeros((fh, fw, 4), dtype=torch.float32, device="cuda")
    r.render(cam, fw, fh, out=frame)
    screen = torch.zeros((96, 128, 4), dtype=torch.float32, device="cuda")
    N.resample_frame(frame, screen, N.SCALE_DOWNSCALE, N.FILTER_MITCHELL_NETRAVALI)
    torch.cuda.synchronize()
    ref = O.resample(frame.cpu().numpy(), 128, 96, N.SCALE_DOWNSCALE, N.FILTER_MITCHELL_NETRAVALI)
    assert np.abs(screen.cpu().numpy() - ref).max() <= 2e-5
    assert ref[..., 3].max() > 0.3


def test_resample_errors():
    src = torch.zeros((8, 8, 4), dtype=torch.float32, device="cuda")
    dst = torch.zeros((16, 16, 4), dtype=torch.float32, device="cuda")
    with pytest.raises(N.CvrError):
        N.resample_frame(src, dst, N.SCALE_UPSCALE, N.FILTER_CARDINAL_OMOMS3)  # needs a work buffer
    with pytest.raises(N.CvrError):
        N.resample_frame(src, dst, 7, N.FILTER_HAT)
    with pytest.raises(N.CvrError):
        N.multiscale_size(128, 96, 0, 2)
