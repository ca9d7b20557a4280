"""The splat's concatenated list walk (fg_pixelwise_hbm.hip), on the CPU.

A wave walks the candidate lists of a chunk's grains as one stream, 64 entries
a step in batches of 8, 4 or 2 steps.  An entry's owner is the number of list
ends before it, counted from a bitset of the batch's entries; and the tested
pixel is the one nearest a target taken from the grain's centre in two f32
roundings.  Both are restated here in the kernel's order of operations.
"""
import numpy as np
import pytest

f32 = np.float32
STAGE = 8  # steps of a whole batch


def walk_owners(lens):
    """The kernel's owner (rank among the listed grains) and clamped stream
    entry of every lane of every step it tests."""
    lens = [n for n in lens if n > 0]
    incl = np.cumsum(lens)
    total = int(incl[-1])
    before, sb, out = 0, 0, []

    def batch(stage, sb, before):
        bits = np.zeros(64 * stage, bool)
        for end in incl:
            rel = int(end) - 1 - sb
            if int(end) != total and 0 <= rel < 64 * stage:
                bits[rel] = True
        for i in range(stage):
            step = bits[64 * i:64 * i + 64]
            own = before + np.concatenate([[0], np.cumsum(step)[:-1]])
            before += int(step.sum())
            s0 = sb + 64 * i
            if s0 < total:
                out.append((own, s0 + np.minimum(np.arange(64), total - 1 - s0)))
        return before

    while total - sb > 64 * (STAGE // 2):
        before = batch(STAGE, sb, before)
        sb += 64 * STAGE
    if total - sb > 64 * (STAGE // 4):
        batch(STAGE // 2, sb, before)
    elif total - sb > 0:
        batch(STAGE // 4, sb, before)
    return out


@pytest.mark.parametrize("total_max", [1, 2, 5, 40, 300])
def test_walk_visits_every_entry_with_its_owner(total_max):
    rng = np.random.default_rng(total_max)
    for trial in range(60):
        n = int(rng.integers(1, 65))
        lens = rng.integers(0, total_max + 1, size=n)
        if trial == 0:  # streams that end on a step or batch boundary
            lens = np.full(64, 8)
        if trial == 1:
            lens = np.array([64 * 4] + [0] * 62 + [64 * 4])
        if not lens.any():
            lens[0] = 1
        owner = np.repeat(np.arange(int((lens > 0).sum())), lens[lens > 0])
        seen = np.zeros(len(owner), bool)
        for own, e in walk_owners(lens):
            assert np.array_equal(own, owner[e]), (total_max, trial)
            seen[e] = True
        assert seen.all()


@pytest.mark.parametrize("z,out_side", [(0.3, 512), (1.0, 4096), (2.0, 3840), (4.0, 16384)])
def test_target_from_the_centre_finds_every_passing_pixel(z, out_side):
    """A pixel whose point passes the f32 disk test of a narrow grain (2 rz <
    1) is rint(fma(O + c, zoom, -1/2)) in both axes, for targets within 1e-3
    of half-integers and radii up to the largest narrow one."""
    rng = np.random.default_rng(int(z * 10) + out_side)
    zf, iz = f32(z), f32(f32(1) / f32(z))
    slack = f32(f32(4e-3) + f32(f32(2e-6) * f32(out_side)))
    M, N = 1500, 48
    g = rng.uniform(0, out_side / z, size=(M, 2)).astype(f32)
    o = rng.normal(0, 0.8 / z, size=(N, 2)).astype(f32)
    h = M // 2
    t = np.floor(g[:h] * zf) + f32(0.5) + rng.uniform(-1e-3, 1e-3, size=(h, 2))
    g[:h] = ((t + 0.5) / z - o[0]).astype(f32)
    r_max = float((f32(0.5) - slack) / zf)
    rad = np.minimum(rng.uniform(0, 1, M) ** 0.3 * r_max, r_max * (1 - 1e-6)).astype(f32)
    hits = 0
    for i in range(M):
        assert f32(f32(rad[i] * zf) + slack) * 2 < 1
        s = (o + g[i]).astype(f32)
        near = np.rint((s.astype(np.float64) * float(zf) - 0.5).astype(f32))
        base = np.floor(s.astype(np.float64) * z).astype(np.int64)
        for ddx in range(-2, 3):
            for ddy in range(-2, 3):
                px, py = (base[:, 0] + ddx).astype(f32), (base[:, 1] + ddy).astype(f32)
                dx = (((px + f32(0.5)) * iz).astype(f32) - o[:, 0]).astype(f32) - g[i, 0]
                dy = (((py + f32(0.5)) * iz).astype(f32) - o[:, 1]).astype(f32) - g[i, 1]
                inside = (dx * dx + dy * dy) <= f32(rad[i] * rad[i])
                assert not np.any(inside & ((px != near[:, 0]) | (py != near[:, 1]))), (z, i)
                hits += int(inside.sum())
    assert hits > 0


@pytest.mark.parametrize("z,out_side,n", [(0.3, 512, 64), (1.0, 4096, 100), (2.0, 3840, 256), (4.0, 16384, 33)])
def test_lists_hold_every_passing_sample(z, out_side, n):
    """Every sample with a pixel that passes the f32 disk test of a narrow
    grain is in the list of the grain's class and cell, in the kernels'
    arithmetic."""
    from tests.test_grain_walk import members
    rng = np.random.default_rng(int(z * 10) + out_side + n)
    zf, iz, q = f32(z), f32(f32(1) / f32(z)), 32
    slack = f32(f32(4e-3) + f32(f32(2e-6) * f32(out_side)))
    o = rng.normal(0, 0.8 / z, size=(n, 2)).astype(f32)
    X = (o * zf).astype(f32)
    fx, fy = ((X[:, i] - np.floor(X[:, i])).astype(f32) for i in (0, 1))
    c_out = out_side + 4 * z + 8  # splat_bounds, less its margins
    eps = f32(c_out * 2.0 ** -20 + 2.0 ** -16)
    hits = 0
    for i in range(2500):
        rad = f32(rng.uniform(0.004, (0.5 - float(slack)) * (1 - 1e-6)) / z)
        if i % 4 == 0:  # at the classes' edges
            rad = f32((int(rng.integers(1, 31)) / 64 + rng.choice([-1e-6, 0, 1e-6])) / z)
        g = rng.uniform(0, out_side / z, size=2).astype(f32)
        if i % 3 == 0:  # sample 0's point at the rim, on a diagonal
            px = np.floor(g * zf)
            g = (((px + 0.5) / z) - o[0] + rng.choice([-1, 1], 2) * (rad / np.sqrt(2) * (1 - 1e-6))).astype(f32)
        b = ((g * zf).astype(f32) - f32(0.5)).astype(f32)
        rz = f32(f32(rad * zf) + slack)
        if not rz + rz < 1:
            continue
        # a constant radius is its own class
        R = f32(rad * zf) if i % 2 else f32(f32(int(f32(f32(rad * zf) * f32(2 * q))) + 1) / f32(2 * q))
        f = (-b - np.floor(-b)).astype(f32)
        qa, qb = (min(int(f32(v * f32(q))), q - 1) for v in f)
        sel = members(fx, fy, qa, qb, q, R, eps)
        near = np.rint(((o + g).astype(f32).astype(np.float64) * z - 0.5)).astype(f32)
        dx = ((((near + f32(0.5)) * iz).astype(f32) - o).astype(f32) - g).astype(f32)
        inside = ((dx * dx).astype(f32).sum(axis=1)).astype(f32) <= f32(rad * rad)
        assert not np.any(inside & ~sel), (i, float(rad))
        hits += int(inside.sum())
    assert hits > 0


@pytest.mark.parametrize("side,rm,delta", [(64, 0.1, 0.1), (4096, 0.05, 0.05), (4096, 0.3, 0.11), (1500, 0.012, 0.4),
                                           (16000, 0.1, 0.1)])
def test_points_within_safe_r_have_the_cell_in_their_window(side, rm, delta):
    """A point whose f32 dx is at most safe_r = rm - 12 C 2^-24 has the
    grain's cell in its f32 window, for centres drawn in their cell (at its
    edges too) and dx up to safe_r; and q < i + 1, q >= i on the quotient is
    the window test floor(q) <= i, floor(q) >= i."""
    rng = np.random.default_rng(side + int(rm * 1e3))
    M = 400_000
    rm, delta = f32(rm), f32(delta)
    C = side + float(rm) + 4.0 + 4.0
    lim = float(rm) - 1.5 * C * 2.0 ** -21
    safe_r = f32(lim)
    if float(safe_r) > lim:
        safe_r = np.nextafter(safe_r, f32(-np.inf))
    if not safe_r > 0:
        safe_r = f32(-1)
    i = rng.integers(-int(3 / delta), int(side / delta), M)
    u = rng.uniform(0, 1, M).astype(f32) * delta
    edge = rng.integers(0, 3, M)
    u = np.where(edge == 0, f32(0), np.where(edge == 1, np.nextafter(delta, f32(0)), u)).astype(f32)
    cx = ((i.astype(f32) * delta).astype(f32) + u).astype(f32)
    d = np.where(rng.random(M) < 0.7, safe_r, rng.uniform(-1, 1, M) * rm).astype(f32) * rng.choice([-1, 1], M)
    xg = (cx + d.astype(f32)).astype(f32)
    xg = np.nextafter(xg, (xg + rng.choice([-1, 0, 1], M)).astype(f32)).astype(f32)
    dx = (xg - cx).astype(f32)
    q_lo, q_hi = (xg - rm).astype(f32) / delta, (xg + rm).astype(f32) / delta
    assert q_lo.dtype == f32
    inside = (np.floor(q_lo) <= i) & (i <= np.floor(q_hi))
    near = np.abs(dx) <= safe_r
    assert not np.any(near & ~inside)
    assert near.sum() > 0 or safe_r < 0
    fi = i.astype(f32)
    assert np.array_equal(inside, (q_lo < fi + f32(1)) & (q_hi >= fi))


@pytest.mark.gpu
@pytest.mark.parametrize("w,h,r,zoom,n,cell", [(64, 48, 0.1, 1.0, 32, None), (3001, 5, 0.08, 1.0, 40, None),
                                               (5, 2500, 0.03, 1.0, 16, 0.2), (90, 37, 0.12, 2.0, 256, 0.05),
                                               (41, 33, 0.24, 2.0, 100, None), (33, 40, 0.2, 0.5, 513, 0.31)])
def test_constant_radius_planes_equal_the_oracle(hip_ctx, oracle, w, h, r, zoom, n, cell):
    """A constant radius is the clamp radius itself: its grains walk the lists
    with the window test on points near the clamp distance.  Thin long planes
    take the coordinates (and with them the share of such points) up."""
    from film_grain_amd import synth
    from tests import fgcases
    u = synth.sinusoid_field(w, h, w + h, n_waves=3)
    case = fgcases.build_case(oracle, f"const_{w}x{h}", u, r, 0.0, "const", zoom=zoom, n_samples=n, seed=w * h + n,
                              cell_delta=cell)
    want = oracle.render_pixelwise(case.plane, case.lam, case.offsets_input)
    got = hip_ctx.render_host("pixel", case.desc, case.lam, case.offsets_input)
    assert int(np.sum(got != want)) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 33, 63, 64, 65, 129, 1000, 1024, 2047, 2048])
def test_tables_of_every_level(hip_ctx, oracle, n):
    """Sample counts around the ranks' groups of four, a workgroup's 64
    samples and the levels (16, 32, ..., n), with offsets that tie in x, in y
    and in both: the fixed render and an adaptive one with budgets in every
    level, against the oracle at each pixel's own sample count."""
    import torch
    from film_grain_amd import synth
    from tests import fgcases
    w, h = 24, 16
    u = synth.sinusoid_field(w, h, n, n_waves=3)
    case = fgcases.build_case(oracle, f"tab_{n}", u, 0.12, 0.04, "lognorm", n_samples=n, seed=n + 5)
    offs = np.array(case.offsets_input)
    offs[n // 2:, 0] = offs[:n - n // 2, 0]
    offs[n // 3:, 1] = np.round(offs[n // 3:, 1] * 4) / 4
    case.offsets_input[:] = offs
    want = oracle.render_pixelwise(case.plane, case.lam, case.offsets_input)
    got = hip_ctx.render_host("pixel", case.desc, case.lam, case.offsets_input)
    assert int(np.sum(got != want)) == 0
    rng = np.random.default_rng(n)
    sizes = sorted({max(1, min(n, v)) for v in (1, 15, 16, 17, 32, 100, 128, 500, 1024, n)})
    blocks = rng.choice(sizes, size=(h // 4, w // 4))
    budget = np.kron(blocks, np.ones((4, 4), dtype=np.int64)).astype(np.uint16)
    out = torch.empty((h, w), dtype=torch.float32, device="cuda:0")
    hip_ctx.render_adaptive_device(case.desc, torch.from_numpy(case.lam).to("cuda:0"),
                                   torch.from_numpy(case.offsets_input).to("cuda:0"),
                                   torch.from_numpy(budget.view(np.int16)).to("cuda:0"), out)
    hip_ctx.stream_status()
    out = out.cpu().numpy()
    for b in np.unique(budget):
        p = oracle.plane(case.derived, int(b), case.seed, case.zoom, case.dist, case.radius)
        fixed = oracle.render_pixelwise(p, case.lam, np.ascontiguousarray(case.offsets_input[:b]))
        assert np.array_equal(out[budget == b], fixed[budget == b]), int(b)
