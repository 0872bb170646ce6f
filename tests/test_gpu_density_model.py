"""The device's form of the disk model (summed exponents, powers by squaring, the azimuth without an
arc tangent) against the host's, over the arm numbers and exponents that take its branches and the
sample counts around the lanes that share a cell."""

import numpy as np
import pytest

from helpers import PC, load_pkg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("arms,index", [(0, 1), (1, 1), (2, 0), (2, 9), (3, 4), (4, 1), (7, 20)])
def test_density_model_matches_host(arms, index):
    pkg = load_pkg()
    md = pkg.disk_model(tau_v=2.0, spiral=arms > 0)
    md.spiral_arms, md.spiral_index, md.perturbation_weight = arms, index, 0.8
    b = [np.linspace(-8 * PC, 8 * PC, q + 1) for q in (5, 4, 3)]
    e = pkg.Engine(0)
    e.grid_cartesian(*b)
    for n in (1, 2, 3, 7, 8, 9, 33):
        print("case density model", arms, index, n, flush=True)
        got = e.sample_density(md, n, 7)
        want = pkg.sample_density_cartesian(*b, md, n, 7)
        # the phase, up to about 50, is off by some 1e-14, which sin^2N (slope below sqrt(2N) cn w
        # < 50) passes on to a density of at least 1 - w = 0.2 of the disk's
        np.testing.assert_allclose(got, want, rtol=4e-12, atol=0)
    e.close()
