"""The draw pass lists a wave's consecutive bins in groups of at most 256
nonempty cells: grids narrower than a chunk of bins (a chunk then spans several
bin rows), grids of one bin, bins that are all empty or all nonempty, and
enough bins for whole chunks, each cell by cell against the oracle."""
import numpy as np
import pytest

from tests import cellcheck, fgcases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h,r,sd,level", [
    (1, 1, 0.4, 0.0, None),        # a few cells
    (6, 90, 0.5, 0.0, None),       # two bin columns: a chunk spans rows
    (90, 6, 0.3, 0.1, None),
    (24, 24, 0.1, 0.05, 0.0),      # nothing to draw
    (24, 24, 0.1, 0.05, 0.999),    # every cell nonempty: one bin a group
    (40, 33, 0.1, 0.0, None),      # empty and full patches
    (280, 210, 0.1, 0.05, None),   # more than 2048 x 8 bins: whole chunks
])
def test_grouped_draws_equal_the_oracle(hip_ctx, oracle, w, h, r, sd, level):
    import torch
    from film_grain_amd import synth
    u = synth.sinusoid_field(w, h, w * h, n_waves=3, flat_fraction=0.3) if min(w, h) > 8 else \
        np.linspace(0, 0.95, w * h, dtype=np.float32).reshape(h, w)
    if level is not None:
        u = np.full((h, w), level, np.float32)
    case = fgcases.build_case(oracle, f"draw_{w}x{h}", u, r, sd, "lognorm" if sd else "const", n_samples=16, seed=w)
    lam = torch.from_numpy(case.lam).to("cuda:0")
    offs = torch.from_numpy(case.offsets_input).to("cuda:0")
    grains, origin, size = hip_ctx.pixelwise_grains(case.desc, lam, offs)
    q, digest = cellcheck.device_cell_digests(grains, size)
    want_q, want_digest = oracle.cell_digests(case.plane, case.lam, origin, size)
    assert np.array_equal(q, want_q)
    assert np.array_equal(digest, want_digest)
