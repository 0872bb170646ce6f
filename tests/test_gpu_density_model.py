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


def test_densities_of_more_cells_than_a_launch_has_threads():
    """2^30 cells, four lanes each: more threads than a launch holds along one direction.  One sample per
    cell, so that each density lies between those of the cell's nearest and farthest points."""
    pkg = load_pkg()
    n, h = 1024, 10 * PC
    hR, hz = 3 * PC, 0.3 * PC
    b = np.linspace(-h, h, n + 1)
    md = pkg.disk_model(tau_v=1.0)
    e = pkg.Engine(0)
    e.grid_cartesian(b, b, b)
    print("case density of 2^30 cells", flush=True)
    got = e.sample_density(md, 1, 3)
    e.close()
    assert len(got) == n ** 3
    for first, step in ((0, 99991), (n ** 3 - 5000, 1), (n ** 3 // 4 - 2500, 1), (n ** 3 // 2 - 2500, 1)):
        m = np.arange(first, n ** 3 if step > 1 else first + 5000, step)
        lo, hi = np.empty((3, len(m))), np.empty((3, len(m)))
        for a, q in enumerate((m // (n * n), m // n % n, m % n)):
            c = np.abs(np.stack([b[q], b[q + 1]]))  # (no cell straddles an axis)
            lo[a], hi[a] = c.min(0), c.max(0)
        peak = pkg.disk_density(md, 0.0, 0.0, 0.0)
        least, most = (peak * np.exp(-np.hypot(c[0], c[1]) / hR - c[2] / hz) for c in (hi, lo))
        assert np.all((got[m] >= least * (1 - 1e-12)) & (got[m] <= most * (1 + 1e-12)))
