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
