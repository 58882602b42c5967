"""Probe points over source segments (few points: many segments), at the edges
of target blocks and source tiles (needs an MI355X).

Against the FP64 oracle the softening length is below every separation, so no
pair takes the spline: FP32 Newtonian terms carry a few eps = 6e-8 each, and a
sum is within 1e-6 of the sum of its terms' magnitudes (FP64 mode: 1e-12).
Against a call with so many points that the sources stay in one segment, full
target blocks have the same FP32 tile sums and only the order of their FP64
sum differs: at most 12 tiles and 3 waves, 1e-14 of the magnitudes.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode,tol", [("fp64", 1e-12), ("split", 1e-6), ("fp32", 1e-6)])
@pytest.mark.parametrize("n", [1, 256, 3001])
@pytest.mark.parametrize("npts", [1, 64, 257, 1000])
def test_probe_points_in_segments(pkg, orc, mode, tol, n, npts):
    pos, vel, mass = pkg.ics.plummer(n, seed=n)
    pts = np.random.default_rng(npts).standard_normal((npts, 3))
    pts[0] = [3.0, 0.0, 0.0]
    h = 1e-7
    if mode == "fp32":
        pos, mass, pts = (v.astype(np.float32).astype(np.float64) for v in (pos, mass, pts))
    bg = (0.5, 0.1, 0.2, -0.3)   # a point mass
    with pkg._native.Context(n, pkg._native.MODES[mode]) as ctx:
        ctx.set_params(1.0, [h] * 6)
        ctx.upload(pos, vel, mass)
        a, p = ctx.force_at_points(pts, h), ctx.potential_at_points(pts, h)
        again = ctx.force_at_points(pts, h)
        ctx.compute_force()            # (the particles are now in Morton order)
        b = ctx.force_at_points(pts, h)
        ctx.add_background(1, bg)
        abg, pbg = ctx.force_at_points(pts, h), ctx.potential_at_points(pts, h)
    mag, closest = np.zeros(npts), np.inf
    for j in range(n):
        mag += np.linalg.norm(orc.force_at_points(pts, h, pos[j:j + 1], mass[j:j + 1]), axis=1)
        closest = min(closest, np.linalg.norm(pts - pos[j], axis=1).min())
    assert closest > 10 * h
    ref_a, ref_p = orc.force_at_points(pts, h, pos, mass), orc.potential_at_points(pts, h, pos, mass)
    assert np.array_equal(a, again)
    assert np.all(np.linalg.norm(a - ref_a, axis=1) <= tol * mag)
    assert np.all(np.linalg.norm(b - ref_a, axis=1) <= tol * mag)
    assert np.all(np.abs(p - ref_p) <= tol * np.abs(ref_p))
    d = pts - np.array(bg[1:])
    r = np.linalg.norm(d, axis=1)
    ext, extp = -bg[0] * d / r[:, None] ** 3, -bg[0] / r
    assert np.all(np.linalg.norm(abg - ref_a - ext, axis=1) <= tol * (mag + np.linalg.norm(ext, axis=1)))
    assert np.all(np.abs(pbg - ref_p - extp) <= tol * (np.abs(ref_p) + np.abs(extp)))


@pytest.mark.parametrize("mode", ["split", "fp32"])
def test_probe_segments_match_one_segment(pkg, orc, mode):
    n, m, h = 3001, 768, 0.05
    pos, vel, mass = pkg.ics.plummer(n, seed=5)
    pts = np.random.default_rng(9).standard_normal((m, 3))
    many = np.concatenate([pts] + [pts] * (4096 * 256 // m))   # 4096 target blocks: one segment
    with pkg._native.Context(n, pkg._native.MODES[mode]) as ctx:
        ctx.set_params(1.0, [h] * 6)
        ctx.upload(pos, vel, mass)
        a, b = ctx.force_at_points(pts, h), ctx.force_at_points(many, h)[:m]
        p, q = ctx.potential_at_points(pts, h), ctx.potential_at_points(many, h)[:m]
    mag = sum(np.linalg.norm(orc.force_at_points(pts, h, pos[j:j + 1], mass[j:j + 1]), axis=1) for j in range(n))
    assert np.all(np.abs(a - b) <= 1e-14 * mag[:, None])
    assert np.all(np.abs(p - q) <= 1e-14 * np.abs(p))
