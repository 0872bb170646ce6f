"""Life cycles on a Voronoi grid with one lane per packet (runs above 512 packets per compute unit)
against the oracle, and, in every variant of the kernel, against the same histories in parts small
enough to have four lanes per packet."""

import numpy as np
import pytest

import oracle as O
from helpers import load_pkg

pytestmark = pytest.mark.gpu

VOR_KEYS = ("sites", "nb_begin", "nb_count", "nb_index", "block_n", "block_begin", "block_count", "block_index", "box")
LIMIT = 512 * 256  # packets: the most with four lanes each
LAM, SEXT, SSCA, G = [0.55e-6, 0.8e-6], [500.0, 350.0], [300.0, 175.0], [0.6, 0.5]


@pytest.fixture(scope="module")
def mesh():
    pkg = load_pkg()
    box = np.array([-1.0, -1.0, -1.0, 1.0, 1.0, 1.0])
    rng = np.random.default_rng(3)
    b = pkg.Voronoi.build(rng.uniform(-1, 1, (1500, 3)), box)
    t = b.export()
    b.close()
    return t, 2e-3 * rng.lognormal(-0.5, 1.0, 1500)


def _frame(inclination, npix=24):
    return dict(inclination=inclination, azimuth=0.3, roll=0.0, nx=npix, ny=npix, fovx=4.0, fovy=4.0)


def _engine(mesh, packets, fp=0):
    pkg = load_pkg()
    t, dens = mesh
    e = pkg.Engine(0)
    e.grid_voronoi(*[t[k] for k in VOR_KEYS])
    e.medium(dens)
    e.dust(LAM, SEXT, SSCA, G)
    f = _frame(1.0)
    e.frame_add(f["inclination"], f["azimuth"], f["roll"], f["nx"], f["ny"], f["fovx"], f["fovy"])
    e.source_point((0.1, -0.05, 0.02), [1.0 / packets] * 2)
    e.options(0.5, 1e4, 0, fp, 31)
    e.tune_pipeline(pkg.SKG_MODE_PERSISTENT)
    return e


@pytest.mark.parametrize("fp", [0, 1], ids=["fp64", "fp32"])
def test_one_lane_life_cycle_matches_oracle(mesh, fp):
    t, dens = mesh
    npk = LIMIT + 9000
    e = _engine(mesh, npk, fp)
    print("case one lane per packet", fp, flush=True)
    e.run_packets(0, npk)
    img, cnt = e.frame_read(0), e.counters()
    e.close()
    ofr, ocnt = O.simulate(O.Grid("voronoi", **{k: t[k] for k in VOR_KEYS}), dens, LAM, SEXT, SSCA, G, [1.0 / npk] * 2,
                           [_frame(1.0)], 0, npk, threads=8, seed=31, src=(0.1, -0.05, 0.02))
    assert cnt[0] == ocnt[0] == npk
    # FP64: the transcendental functions differ in the last bits; FP32: the sums' 1e-7 turns a packet in
    # some thousand another way at a threshold
    assert abs(int(cnt[2]) - int(ocnt[2])) <= 1e-3 * ocnt[2]
    oimg = ofr[0]
    assert abs(img.sum() / oimg.sum() - 1) < (1e-6 if fp == 0 else 1e-4)
    nz = oimg > 0
    assert np.median(np.abs(img[nz] / oimg[nz] - 1)) < (1e-9 if fp == 0 else 1e-4)


@pytest.mark.parametrize("variant", ["plain", "fp32", "field", "perspective", "particles", "guided", "batched"])
def test_one_and_four_lanes_agree(mesh, variant):
    """The same histories in one run above the limit and in two below it: the segments are the same bit
    for bit, so the counters are equal and the images agree up to the order of their sums."""
    pkg = load_pkg()
    npk = LIMIT + 2000
    e = _engine(mesh, npk, 1 if variant == "fp32" else 0)
    if variant == "field":
        e.rf_enable()
    elif variant == "perspective":
        from skirt9_gpu_amd import ski as S
        M, eye, size = S.perspective_setup(np.array([1.0, -3.0, 2.0]), np.zeros(3), np.array([0.0, 0.0, 1.0]), 3.0, 2.0, 30, 30)
        e.perspective_add(M, eye, size, 30, 30)
    elif variant == "particles":
        rng = np.random.default_rng(5)
        lum = rng.uniform(0.1, 3.0, (50, 2))
        e.source_particles(np.hstack([rng.uniform(-0.7, 0.7, (50, 3)), rng.uniform(0.05, 0.2, (50, 1))]), lum, lum.sum(1), npk)
    elif variant == "guided":
        rng = np.random.default_rng(6)
        e.guide_params(np.concatenate([np.concatenate([rng.normal(0, np.sqrt(2 / i), i * o) * (0.1 if o == 40 else 1), np.zeros(o)])
                                       for i, o in ((9, 64), (64, 64), (64, 64), (64, 40))]).astype(np.float32))
        e.guide_mode(1, 0.5, 1.0)
    elif variant == "batched":
        counts = np.array([npk // 2, npk - npk // 2 - 77, 77], np.uint64)
        for q in range(2):
            f = _frame(0.3 + 0.4 * q)
            e.frame_add(f["inclination"], f["azimuth"], f["roll"], f["nx"], f["ny"], f["fovx"], f["fovy"])
        e.instances(counts, [1, 2, 3], [0.5, 1.0, 3.0], np.repeat(1.0 / counts[:, None], 2, axis=1), [0, 1, 2], [1, 1, 1])
    out = []
    for parts in ([npk], [npk // 2, npk - npk // 2]):
        e.frame_clear()
        if variant == "field":
            e.rf_clear()
        print("case lanes", variant, parts, flush=True)
        for first, n in zip((0, parts[0]), parts):
            e.run_packets(first, n)
        out.append((np.array(e.counters()), [e.frame_read(q) for q in range(len(e.frames))],
                    e.rf_read() if variant == "field" else None))
    e.close()
    (c1, f1, r1), (c2, f2, r2) = out
    c1[5] = c2[5] = 0  # atomics after the wavefront's combination
    np.testing.assert_array_equal(c1, c2)
    for a, b in zip(f1, f2):
        assert b.sum() > 0
        np.testing.assert_allclose(a, b, rtol=1e-11, atol=1e-14 * b.max())
    if r1 is not None:
        np.testing.assert_allclose(r1, r2, rtol=1e-11, atol=1e-14 * r2.max())
