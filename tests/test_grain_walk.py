"""The grain-wise kernel's candidate lists and its narrow test
(fg_grainwise.hip, grain_lists_kernel), on the CPU in f32 and on the GPU
against the oracle."""
import numpy as np
import pytest

f32 = np.float32


def members(fx, fy, qa, qb, q, R, eps):
    """splat_lists_body's membership, in its order of operations."""
    half = f32(f32(0.5) / f32(q))
    reach = f32(R + f32(eps + f32(2.0 ** -12)))

    def beyond(f, c):  # distance from the cell's interval on the unit circle
        d = (f - f32(f32(f32(c) / f32(q)) + half)).astype(f32)
        return np.maximum((np.abs((d - np.rint(d)).astype(f32)) - half).astype(f32), f32(0))
    dx, dy = beyond(fx, qa), beyond(fy, qb)
    return ((dx * dx).astype(f32) + (dy * dy).astype(f32)).astype(f32) <= f32(reach * reach)


def box(t, R):
    """bounds() of src/grainwise.rs:126-142 before its clamp."""
    return (np.ceil(((t - R).astype(f32) - f32(0.5)).astype(f32)),
            np.floor(((t + R).astype(f32) - f32(0.5)).astype(f32)))


@pytest.mark.parametrize("side,N,sd,const", [(1280, 64, 0.8, False), (4096, 128, 0.8, True), (4096, 300, 2.0, False),
                                             (16384, 100, 0.8, True), (64, 2048, 0.4, False)])
def test_lists_and_narrow_test_find_every_hit(side, N, sd, const):
    """Every (sample, pixel) that the reference tests (in its box) and that
    passes its disk test is in the grain's list, is pixel floor(t), and the
    box need not be looked at where |dx|, |dy| <= R - C 2^-21."""
    rng = np.random.default_rng(side + N)
    X = rng.normal(0, sd, size=(N, 2)).astype(f32)
    fx, fy = ((X[:, i] - np.floor(X[:, i])).astype(f32) for i in (0, 1))
    rmax = f32(0.45 if const else 0.6)
    C = f32(f32(side) + np.abs(X).max() + rmax + f32(8))
    eps = f32(f32(C * f32(2.0 ** -20)) + f32(2.0 ** -16))
    edge = f32(C * f32(2.0 ** -21))
    narrow_r = f32(f32(0.5) - f32(eps + eps))
    hits = rim = 0
    for i in range(2500):
        R = rmax if const and i % 2 else f32(rng.uniform(0.002, float(rmax)))
        if i % 5 == 0 and not const:
            R = f32(int(rng.integers(1, 32)) / 64 + rng.choice([-1e-6, 0, 1e-6]))  # class edges
        if not R < narrow_r:
            continue
        b = rng.uniform(-4, side + 4, size=2).astype(f32)
        if i % 3 == 0:  # targets of sample 0 at the rim of a pixel's disk
            b = (np.floor(b) + f32(0.5) + rng.choice([-1, 1], 2) * R - X[0] +
                 rng.uniform(-2, 2, 2) * 2.0 ** -12).astype(f32)
        q = 64 if const else 32
        Rl = R if const else f32((int(R * f32(64)) + 1) / 64)
        n = (f32(0.5) - b).astype(f32)
        f = (n - np.floor(n)).astype(f32)
        qa, qb = (min(int(f32(v * f32(q))), q - 1) for v in f)
        sel = members(fx, fy, qa, qb, q, Rl, eps)
        t = (b + X).astype(f32)
        xl, xh = box(t[:, 0], R)
        yl, yh = box(t[:, 1], R)
        for ox in (-1, 0, 1):
            for oy in (-1, 0, 1):
                px, py = np.floor(t[:, 0]) + ox, np.floor(t[:, 1]) + oy
                dx = ((px + f32(0.5)).astype(f32) - t[:, 0]).astype(f32)
                dy = ((py + f32(0.5)).astype(f32) - t[:, 1]).astype(f32)
                disk = ((dx * dx).astype(f32) + (dy * dy).astype(f32)).astype(f32) <= f32(R * R)
                inbox = (xl <= px) & (px <= xh) & (yl <= py) & (py <= yh)
                ref = disk & inbox
                assert not np.any(ref & ~sel), (i, float(R))
                if ox or oy:
                    assert not np.any(disk)
                    continue
                inner = disk & (np.maximum(np.abs(dx), np.abs(dy)) <= f32(R - edge))
                assert not np.any(inner & ~inbox)
                hits += int(ref.sum())
                rim += int((disk & ~inner).sum())
    assert hits > 0 and rim > 0


@pytest.mark.gpu
@pytest.mark.parametrize("r_out,sd", [(0.01, 0.0), (0.2, 0.0), (0.449, 0.0), (0.4501, 0.0), (0.51, 0.0), (1.2, 0.0),
                                      (0.05, 0.03), (0.2, 0.15), (0.45, 0.1), (0.9, 0.5)])
def test_planes_across_the_list_limits(hip_ctx, oracle, r_out, sd):
    """Constant output radii on both sides of the lists' limits and lognormal
    laws with narrow, wide and mixed grains, for several zooms and sample
    counts."""
    from film_grain_amd import synth
    from tests import fgcases
    rng = np.random.default_rng(int(r_out * 1e4))
    for zoom, n in [(0.5, 300), (1.0, 1), (2.0, 64), (3.0, 2048)]:
        w, h = 27, 22
        grains = w * h * 1.4 / (np.pi * (r_out / zoom) ** 2)
        while n > 1 and (round(w * zoom) * round(h * zoom) * n > 2_000_000 or grains * n > 5e8):
            n //= 2
        u = synth.sinusoid_field(w, h, int(rng.integers(0, 1 << 30)), n_waves=3)
        case = fgcases.build_case(oracle, f"gl_{r_out}_{zoom}", u, r_out / zoom, sd / zoom,
                                  "lognorm" if sd else "const", zoom=zoom, n_samples=n,
                                  seed=int(rng.integers(0, 1 << 40)))
        want = oracle.render_grainwise(case.plane, case.lam, case.offsets)
        got = hip_ctx.render_host("grain", case.desc, case.lam, case.offsets)
        assert int(np.sum(got != want)) == 0, (zoom, n)


@pytest.mark.gpu
@pytest.mark.parametrize("sd", [0.0, 0.02])
def test_thin_long_plane(hip_ctx, oracle, sd):
    """Coordinates up to 6000 output pixels: a widening of 6e-3 and a rim of
    3e-3 around radii of 0.04 and up."""
    from film_grain_amd import synth
    from tests import fgcases
    u = synth.sinusoid_field(3000, 3, 5, n_waves=3)
    case = fgcases.build_case(oracle, "thin", u, 0.04, sd, "lognorm" if sd else "const", zoom=2.0, n_samples=24,
                              seed=77)
    want = oracle.render_grainwise(case.plane, case.lam, case.offsets)
    got = hip_ctx.render_host("grain", case.desc, case.lam, case.offsets)
    assert int(np.sum(got != want)) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("w,h,r,sd", [(1, 1, 0.1, 0.0), (63, 1, 0.14, 0.0), (65, 3, 0.05, 0.02), (513, 2, 0.13, 0.0),
                                      (129, 64, 0.3, 0.0), (811, 655, 0.13, 0.0), (700, 750, 0.06, 0.0)])
def test_counts_of_every_pixel(hip_ctx, oracle, w, h, r, sd):
    """Pixels below and above a mean of 12 grains (Knuth's product, the
    rejection sampler with its queue), whole and partial waves, one round of
    the grid's pixels and more; streams resume where the count left them."""
    from film_grain_amd import synth
    from tests import fgcases
    plane = synth.sinusoid_field(w, h, w + h, n_waves=3)
    c = fgcases.build_case(oracle, "count", plane, r, sd, "lognorm" if sd else "const", zoom=1.0, n_samples=2, seed=w)
    want = oracle.render_grainwise(c.plane, c.lam, c.offsets)
    got = hip_ctx.render_host("grain", c.desc, c.lam, c.offsets)
    assert np.array_equal(got, want)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 16, 63, 64, 65, 127, 129, 1000, 2048])
@pytest.mark.parametrize("r,sd,zoom", [(0.25, 0.1, 2.0),   # narrow and wide grains in one round
                                       (0.15, 0.07, 2.0),  # a few wide ones
                                       (0.45, 0.1, 3.0)])  # all wide, boxes of several pixels
def test_wide_grains_among_narrow_ones(hip_ctx, oracle, n, r, sd, zoom):
    """Lognormal radii on both sides of half an output pixel: the narrow grains
    walk lists, each wide one its run of the sample order, 64 samples a step:
    whole and broken steps, and runs past the end of the order."""
    from film_grain_amd import synth
    from tests import fgcases
    c = fgcases.build_case(oracle, "wide", synth.sinusoid_field(13, 11, n, n_waves=3), r, sd, "lognorm", zoom=zoom,
                           n_samples=n, seed=n + 7)
    want = oracle.render_grainwise(c.plane, c.lam, c.offsets)
    for block in (512, 256):
        hip_ctx.set_launch_config(grain_variant=2, grain_block=block)
        try:
            got = hip_ctx.render_host("grain", c.desc, c.lam, c.offsets)
        finally:
            hip_ctx.reset_launch_config()
        assert np.array_equal(got, want), block


def test_room_of_the_class_lists():
    """No class of the lognormal lists holds more entries than its room,
    N min(q, k + 4 + e)^2, up to the widest eps that lists are built for."""
    q, e, N = 32, 4, 96
    assert (2 * 0.0622 + 2.0 ** -11) * q <= e
    rng = np.random.default_rng(3)
    for fx, fy in (rng.random((2, N)).astype(f32), (rng.integers(0, q, (2, N)) / q).astype(f32)):
        for eps in (f32(2.0 ** -16), f32(0.0622)):
            for k in range(q):
                R = f32(f32(k + 1) / f32(2 * q))
                n = sum(int(members(fx, fy, qa, qb, q, R, eps).sum()) for qa in range(q) for qb in range(q))
                assert n <= N * min(q, k + 4 + e) ** 2, (k, float(eps))


@pytest.mark.gpu
@pytest.mark.parametrize("far", [0.0, 30000.0, 64000.0, 65100.0, 70000.0, 300000.0])
def test_far_offsets(hip_ctx, oracle, far):
    """One sample's offset far outside the plane: the lists' widening grows to
    its limit (about 65000) and the grains walk their runs beyond."""
    from film_grain_amd import synth
    from tests import fgcases
    c = fgcases.build_case(oracle, "far", synth.sinusoid_field(24, 17, 3, n_waves=3), 0.1, 0.04, "lognorm", zoom=2.0,
                           n_samples=70, seed=12)
    offs = np.ascontiguousarray(c.offsets).copy()
    offs[5, 0] += np.float32(far)
    offs[6, 1] -= np.float32(far)
    want = oracle.render_grainwise(c.plane, c.lam, offs)
    assert np.array_equal(hip_ctx.render_host("grain", c.desc, c.lam, offs), want)
