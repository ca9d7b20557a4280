"""The wave-wide inclusive sum behind the concatenated walks and the draw
groups: list lengths, counts and candidates that put zeros, large values and
uneven totals in every lane, through planes of few and of many grains a cell
(one to hundreds), against the oracle."""
import numpy as np
import pytest

from film_grain_amd import synth
from tests import fgcases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("algo", ["pixel", "grain"])
@pytest.mark.parametrize("r,sd,cell,n", [(0.02, 0.0, 1.0, 16), (0.1, 0.05, 0.1, 64), (0.3, 0.0, 0.05, 33),
                                         (0.05, 0.02, 0.6, 128)])
def test_uneven_sums(hip_ctx, oracle, algo, r, sd, cell, n):
    u = synth.sinusoid_field(23, 19, int(r * 1000) + n, n_waves=4, flat_fraction=0.2)
    case = fgcases.build_case(oracle, f"sum_{r}", u, r, sd, "lognorm" if sd else "const", n_samples=n, seed=n,
                              cell_delta=cell)
    if algo == "pixel":
        want = oracle.render_pixelwise(case.plane, case.lam, case.offsets_input)
        got = hip_ctx.render_host(algo, case.desc, case.lam, case.offsets_input)
    else:
        want = oracle.render_grainwise(case.plane, case.lam, case.offsets)
        got = hip_ctx.render_host(algo, case.desc, case.lam, case.offsets)
    assert int(np.sum(got != want)) == 0
