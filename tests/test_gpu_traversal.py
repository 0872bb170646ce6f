"""The path generators where their short cuts do not apply, on the GPU and bit for bit against the
oracle: Voronoi cells with ties, close and many neighbours, with one and with four lanes per path;
octrees with fine neighbours, split planes hit exactly, and more planes than the LDS holds; Cartesian
grids beyond the LDS and beyond the packed start hint.  Start hints: the counters and images of
packets from sources on and off the cells' faces."""

import numpy as np
import pytest

import oracle as O
from helpers import frame60, load_pkg

pytestmark = pytest.mark.gpu

VOR_KEYS = ("sites", "nb_begin", "nb_count", "nb_index", "block_n", "block_begin", "block_count", "block_index", "box")


@pytest.fixture(scope="module")
def eng():
    e = load_pkg().Engine(0)
    yield e
    e.close()


def _rays(box, on, seed, n=2000):
    """Random rays, axis-parallel and diagonal ones, from inside, outside and the points `on`."""
    rng = np.random.default_rng(seed)
    lo, hi = box[:3], box[3:]
    r = lo + (hi - lo) * (rng.random((n, 3)) * 1.2 - 0.1)
    r[::4] = on[rng.integers(0, len(on), len(r[::4]))]
    k = rng.normal(size=(n, 3))
    k[1::5] = np.eye(3)[rng.integers(0, 3, len(k[1::5]))] * rng.choice([-1.0, 1.0], (len(k[1::5]), 1))
    k[2::5] = rng.choice([-1.0, 1.0], (len(k[2::5]), 3))
    return np.hstack([r, k / np.linalg.norm(k, axis=1, keepdims=True)])


def _compare(eng, grid, rays, repeat):
    off, m, ds = eng.trace_paths(np.tile(rays, (repeat, 1)), cap=None if repeat == 1 else repeat * 40 * len(rays))
    ooff, om, ods = O.trace(grid, rays)
    cnt = np.diff(ooff)
    np.testing.assert_array_equal(np.diff(off), np.tile(cnt, repeat))
    np.testing.assert_array_equal(m, np.tile(om, repeat))
    np.testing.assert_array_equal(ds, np.tile(ods, repeat))


def _vor_points(name):
    rng = np.random.default_rng(4)
    if name == "lattice":  # every vertex is shared by eight cells, and rays run along faces
        a = (np.arange(6) + 0.5) / 6
        return np.stack(np.meshgrid(a, a, a, indexing="ij"), -1).reshape(-1, 3)
    if name == "close":  # pairs of sites nearer than the FP32 bounds resolve, and a dense clump
        p = rng.random((150, 3))
        return np.clip(np.vstack([p, p[:40] + 3e-10, 0.5 + 1e-6 * rng.random((60, 3))]), 1e-9, 1 - 1e-9)
    if name == "hub":  # one cell with hundreds of neighbours
        k = rng.normal(size=(400, 3))
        return np.vstack([[[0.5, 0.5, 0.5]], 0.5 + 0.4 * k / np.linalg.norm(k, axis=1, keepdims=True)])
    return rng.random((dict(one=1, two=2, few=5).get(name, 700), 3))


@pytest.mark.parametrize("repeat", [1, 70], ids=["four_lanes", "one_lane"])
@pytest.mark.parametrize("name,shift", [("lattice", 0.0), ("close", 0.0), ("hub", 0.0), ("one", 0.0), ("two", 0.0),
                                        ("few", 0.0), ("far", 1e7)])
def test_voronoi_paths_bit_exact(eng, name, shift, repeat):
    pkg = load_pkg()
    box = np.array([0.0, 0.0, 0.0, 1.0, 1.0, 1.0]) + shift
    b = pkg.Voronoi.build(_vor_points(name) + shift, box)
    t = b.export()
    b.upload(eng)
    b.close()
    print("case voronoi", name, repeat, flush=True)
    s = np.asarray(t["sites"])
    on = np.vstack([s, 0.5 * (s + np.roll(s, 1, axis=0))])
    _compare(eng, O.Grid("voronoi", **{k: t[k] for k in VOR_KEYS}), _rays(box, on, 1), repeat)


@pytest.mark.parametrize("name", ["shared", "split", "grid"])
def test_tetra_paths_bit_exact(eng, name):
    """Rays through vertices, along edges and in faces' planes; split: no two cells share vertex ids,
    so that every crossing reads the next cell's vertices."""
    pkg = load_pkg()
    box = np.array([-1.0, -1.0, -1.0, 1.0, 1.0, 1.0])
    rng = np.random.default_rng(7)
    if name == "grid":  # nearly a lattice: flat tetrahedra and rays that graze them
        a = np.linspace(-0.8, 0.8, 5)
        pts = np.stack(np.meshgrid(a, a, a, indexing="ij"), -1).reshape(-1, 3) + rng.normal(0, 1e-7, (125, 3))
    else:
        pts = rng.uniform(-1, 1, (400, 3))
    b = pkg.Tetra.build(pts, box)
    t = b.export()
    b.close()
    v, tv = np.asarray(t["verts"]).reshape(-1, 3), np.asarray(t["tet_verts"]).reshape(-1, 4)
    if name == "split":
        t["verts"], t["tet_verts"] = v[tv.ravel()], np.arange(tv.size, dtype=np.int32).reshape(-1, 4)
    eng.grid_tetra(t["verts"], t["tet_verts"], t["face_nb"], t["face_normal"], t["box"])
    rays = _rays(box, np.vstack([pts, 0.5 * (v[tv[:, 0]] + v[tv[:, 1]])]), 5)
    to = v[tv[rng.integers(0, len(tv), 300), 2]] - rays[:300, :3]  # exactly toward vertices
    rays[:300, 3:] = to / np.maximum(np.linalg.norm(to, axis=1, keepdims=True), 1e-300)
    rays = rays[np.linalg.norm(rays[:, 3:], axis=1) > 0.5]
    print("case tetra", name, len(tv), flush=True)
    _compare(eng, O.Grid("tetra", **t), rays, 1)


def _octree_flags(box, levels, refine):
    """Level-order division flags: nodes that `refine` (lo, hi, level) selects, up to `levels`."""
    flags, row = [], [(tuple(box[:3]), tuple(box[3:]))]
    for level in range(levels + 1):
        nxt = []
        for lo, hi in row:
            d = level < levels and refine(lo, hi, level)
            flags.append(1 if d else 0)
            if d:
                c = [0.5 * (a + b) for a, b in zip(lo, hi)]
                for q in range(8):
                    nxt.append((tuple(c[a] if q >> a & 1 else lo[a] for a in range(3)),
                                tuple(hi[a] if q >> a & 1 else c[a] for a in range(3))))
        row = nxt
    return np.array(flags, np.uint8)


@pytest.mark.parametrize("name", ["root", "random", "lines"])
def test_octree_paths_bit_exact(eng, name):
    pkg = load_pkg()
    box = np.array([-1.0, -1.0, -1.0, 1.0, 1.0, 1.0])
    if name == "root":
        flags = _octree_flags(box, 0, None)
    elif name == "random":
        rng = np.random.default_rng(8)
        flags = _octree_flags(box, 6, lambda lo, hi, level: level < 2 or rng.random() < 0.25)
    else:  # fine along lines parallel to the x and to the y axis: more planes than the LDS table holds
        p = (0.3, 0.7, 0.123, 0.234)
        flags = _octree_flags(box, 12, lambda lo, hi, level: (lo[1] <= p[0] <= hi[1] and lo[2] <= p[1] <= hi[2])
                              or (lo[0] <= p[2] <= hi[0] and lo[2] <= p[3] <= hi[2]))
    tree = pkg.Octree.from_flags(box, flags)
    t = tree.export()
    tree.upload(eng)
    tree.close()
    print("case octree", name, len(flags), flush=True)
    corners = np.asarray(t["bounds"])[:, 3:]
    rays = _rays(box, corners[np.random.default_rng(2).integers(0, len(corners), 500)], 3)
    _compare(eng, O.Grid("octree", **{k: t[k] for k in ("bounds", "child_first", "cell_index", "nb_off", "nb_id")}), rays, 1)


@pytest.mark.parametrize("n", [(1, 1, 1), (7, 5, 3), (1030, 3, 2), (2, 3300, 2)])
def test_cartesian_paths_and_packets(eng, n):
    rng = np.random.default_rng(5)
    b = [np.concatenate([[-1.0], np.sort(rng.uniform(-1, 1, q - 1)), [1.0]]) for q in n]
    eng.grid_cartesian(*b)
    box = np.array([-1.0] * 3 + [1.0] * 3)
    g = O.Grid("cartesian", xb=b[0], yb=b[1], zb=b[2])
    print("case cartesian", n, flush=True)
    _compare(eng, g, _rays(box, np.stack([rng.choice(q, 200) for q in b], 1), 6, 400), 1)
    _packets(eng, g, np.ones(int(np.prod(n))) * 1e-3, (b[0][0 if n[0] == 1 else 1], 0.1, 0.2))


def _packets(eng, grid, dens, src):
    """Few packets (the lanes-per-wave rule) from a source on a face: the oracle's counts and image."""
    eng.medium(dens)
    eng.dust([0.55e-6], [500.0], [300.0], [0.6])
    fr = frame60(npix=20)
    fr["fovx"] = fr["fovy"] = 4.0
    eng.frame_remove_all()
    eng.frame_add(fr["inclination"], fr["azimuth"], fr["roll"], fr["nx"], fr["ny"], fr["fovx"], fr["fovy"])
    for npk, mode in ((1, 1), (700, 1), (700, 0)):  # persistent, persistent, pipeline
        eng.source_point(src, [1.0 / npk])
        eng.options(0.5, 1e4, 0, 0, 13)
        eng.tune_pipeline(mode, 1 << 14, 0, 8)
        eng.frame_clear()
        eng.run_packets(0, npk)
        img, cnt = eng.frame_read(0)[0], eng.counters()
        ofr, ocnt = O.simulate(grid, dens, [0.55e-6], [500.0], [300.0], [0.6], [1.0 / npk], [fr], 0, npk, threads=4, seed=13,
                               src=src)
        # the transcendental functions differ in the last bits: a packet near a threshold may take
        # another turn, one in a thousand at most
        assert cnt[0] == ocnt[0] == npk
        assert abs(int(cnt[2]) - int(ocnt[2])) <= max(1e-3 * ocnt[2], 1)
        assert abs(img.sum() / ofr[0][0].sum() - 1) < 1e-6


@pytest.mark.parametrize("kind", ["octree", "voronoi", "tetra"])
def test_start_hints(eng, kind):
    """Sources on a site, a vertex or a face, and moved from one cell to another without a new grid."""
    pkg = load_pkg()
    box = np.array([-1.0, -1.0, -1.0, 1.0, 1.0, 1.0])
    rng = np.random.default_rng(9)
    if kind == "octree":
        b = pkg.Octree.from_flags(box, _octree_flags(box, 4, lambda lo, hi, level: level < 2 or rng.random() < 0.4))
        keys, srcs = ("bounds", "child_first", "cell_index", "nb_off", "nb_id"), [(0.0, 0.0, 0.0), (0.5, 0.25, -0.1)]
    else:
        pts = rng.uniform(-1, 1, (900, 3))
        b = pkg.Voronoi.build(pts, box) if kind == "voronoi" else pkg.Tetra.build(pts, box)
        keys, srcs = VOR_KEYS if kind == "voronoi" else None, [(0.0, 0.0, 0.0), tuple(pts[17]), tuple(0.5 * (pts[3] + pts[4]))]
    t = b.export()
    b.upload(eng)
    b.close()
    g = O.Grid(kind, **({k: t[k] for k in keys} if keys else t))
    for src in srcs:
        print("case start hint", kind, src, flush=True)
        _packets(eng, g, np.full(eng.num_cells(), 1e-3), src)


def test_service_calls_share_an_engines_buffer():
    """Optical depths and densities of growing and shrinking calls in turn, one beyond the buffer that
    the engine keeps, give what an engine of their own gives."""
    pkg = load_pkg()
    b = np.linspace(-1.0, 1.0, 9)
    rng = np.random.default_rng(3)
    md = pkg.disk_model(tau_v=1.0, scale_length=0.3, scale_height=0.1)

    def engine():
        e = pkg.Engine(0)
        e.grid_cartesian(b, b, b)
        e.medium(np.linspace(0.0, 2e-3, 512))
        e.dust([0.55e-6], [500.0], [300.0], [0.6])
        return e

    shared = engine()
    rays = np.hstack([rng.uniform(-1, 1, (3000, 3)), np.tile([0.6, 0.0, 0.8], (3000, 1))])
    for n in (1, 3000, 7, 4_400_000, 100):
        print("case shared buffer", n, flush=True)
        r = np.resize(rays, (n, 6))
        got = shared.trace_tau(r)
        e = engine()
        want = e.trace_tau(r[:3000])
        for g, w in zip(got, want):
            np.testing.assert_array_equal(g, np.resize(w, n))
        np.testing.assert_array_equal(shared.sample_density(md, 5, n), e.sample_density(md, 5, n))
        e.close()
    shared.close()


@pytest.mark.parametrize("repeat", [1, 70], ids=["four_lanes", "one_lane"])
def test_voronoi_cells_without_a_face_ahead(eng, repeat):
    """Cells whose lists hold no neighbour ahead of the path, or none at all: the path steps on by eps
    until the nearest site is another cell's, as with the oracle."""
    sites = np.array([[-0.5, 0.0, 0.0], [0.5, 0.0, 0.0], [0.5, 0.0, 0.9]])
    lists = [[-1], [-1, -2, -3, -4, -5, 2], []]
    count = np.array([len(q) for q in lists], np.int32)
    box = np.array([-1.0, -1.0, -1.0, 1.0, 1.0, 1.0])
    t = dict(sites=sites, nb_begin=np.array([0, 1, 7], np.int32), nb_count=count,
             nb_index=np.array(sum(lists, []), np.int32), block_n=1, block_begin=np.array([0], np.int32),
             block_count=np.array([3], np.int32), block_index=np.arange(3, dtype=np.int32), box=box)
    eng.grid_voronoi(*[t[k] for k in VOR_KEYS])
    # from a few eps (3.5e-12) before the plane x = 0, and from above the third site's plane z = 0.45
    rng = np.random.default_rng(11)
    n = 2000
    first = np.arange(n) % 2 == 0
    r = np.stack([np.where(first, -4e-11 * rng.random(n), 0.3), 0.2 * rng.normal(size=n).clip(-3, 3),
                  np.where(first, -0.3, 0.45 + 4e-11 * rng.random(n))], 1)
    k = np.stack([np.where(first, 1.0, 0.3), 0.1 * rng.normal(size=n), np.where(first, 0.1, -1.0)], 1)
    print("case voronoi without a face ahead", repeat, flush=True)
    _compare(eng, O.Grid("voronoi", **t), np.hstack([r, k / np.linalg.norm(k, axis=1, keepdims=True)]), repeat)


def test_few_workgroups_use_all_their_lanes(eng):
    """A small run held to one workgroup takes all its 256 lanes: 1000 packets are then four in a row per
    lane instead of one, and full wavefronts take at most about three times as long per step as those of
    four lanes.  (With four lanes of each wavefront they would be 63 in a row.)"""
    b = np.linspace(-1.0, 1.0, 33)
    eng.grid_cartesian(b, b, b)
    eng.medium(np.full(32 ** 3, 1e-3))
    eng.dust([0.55e-6], [5000.0], [3000.0], [0.6])
    eng.frame_remove_all()
    eng.frame_add(1.0, 0.0, 0.0, 20, 20, 4.0, 4.0)
    eng.source_point((0.0, 0.0, 0.0), [1e-3])
    eng.options(0.5, 1e4, 0, 0, 5)
    eng.tune_pipeline(1)
    print("case few workgroups", flush=True)
    ms, flux = {}, {}
    for wg in (0, 1):
        eng.tune(wg, 256, 32)
        runs = []
        for _ in range(4):
            eng.frame_clear()
            eng.run_packets(0, 1000)
            runs.append(eng.last_kernel_ms())
        ms[wg], flux[wg] = min(runs), eng.frame_read(0).sum()
    eng.tune(0, 256, 16)
    assert flux[1] == pytest.approx(flux[0], rel=1e-12)
    assert ms[1] < 12 * ms[0], ms


def test_voronoi_paths_along_faces_are_no_slower(eng):
    """A view in a plane of the lattice's faces against one that no face is parallel to, by time: the
    peel-offs cross as many cells, and no crossing needs the search in FP64."""
    pkg = load_pkg()
    box = np.array([-1.0, -1.0, -1.0, 1.0, 1.0, 1.0])
    a = (np.arange(24) + 0.5) / 12 - 1
    b = pkg.Voronoi.build(np.stack(np.meshgrid(a, a, a, indexing="ij"), -1).reshape(-1, 3), box)
    b.upload(eng)
    b.close()
    eng.medium(np.full(24 ** 3, 1e-3))
    eng.dust([0.55e-6], [2000.0], [1200.0], [0.6])
    eng.source_point((0.01, 0.02, 0.03), [1e-5])
    eng.options(0.5, 1e4, 0, 0, 5)
    eng.tune_pipeline(1)
    ms = []
    for azimuth in (0.3, 0.0):  # at 0, the view has no component along y
        eng.frame_remove_all()
        eng.frame_add(0.9, azimuth, 0.0, 20, 20, 4.0, 4.0)
        print("case voronoi view", azimuth, flush=True)
        runs = []
        for _ in range(4):
            eng.frame_clear()
            eng.run_packets(0, 200_000)
            runs.append(eng.last_kernel_ms())
        ms.append(min(runs))
    assert ms[1] < 1.25 * ms[0], ms


@pytest.mark.parametrize("repeat", [1, 70], ids=["four_lanes", "one_lane"])
@pytest.mark.parametrize("name", ["lattice", "few", "many"])
def test_voronoi_paths_almost_along_faces_bit_exact(eng, name, repeat):
    """Directions 1e-2 to 1e-12 away from a face's plane, around where the FP32 bounds take the face for
    parallel, from inside cells and from close to their faces."""
    pkg = load_pkg()
    box = np.array([0.0, 0.0, 0.0, 1.0, 1.0, 1.0])
    b = pkg.Voronoi.build(_vor_points(name), box)
    t = b.export()
    b.upload(eng)
    b.close()
    rng = np.random.default_rng(12)
    n, s = 2000, np.asarray(t["sites"])
    i, q = rng.integers(0, len(s), n), rng.integers(0, 3, n)
    near = np.argsort(((s[:, None] - s[None]) ** 2).sum(-1), axis=1)[i, 1 % len(s)] if len(s) < 800 else i
    normal = s[near] - s[i]
    wall = (np.arange(n) % 3 == 0) | (np.linalg.norm(normal, axis=1) == 0)
    normal[wall] = np.eye(3)[q[wall]]
    normal /= np.linalg.norm(normal, axis=1, keepdims=True)
    k = np.cross(normal, rng.normal(size=(n, 3)))
    k /= np.linalg.norm(k, axis=1, keepdims=True)
    k += normal * (10.0 ** rng.uniform(-12, -2, (n, 1)) * rng.choice([-1.0, 1.0], (n, 1)))
    r = np.where((np.arange(n) % 2 == 0)[:, None], s[i], 0.5 * (s[i] + s[near]))
    r = np.clip(r + normal * (10.0 ** rng.uniform(-12, -1, (n, 1)) * rng.choice([-1.0, 1.0], (n, 1))), 1e-9, 1 - 1e-9)
    print("case voronoi almost along faces", name, repeat, flush=True)
    _compare(eng, O.Grid("voronoi", **{k_: t[k_] for k_ in VOR_KEYS}),
             np.hstack([r, k / np.linalg.norm(k, axis=1, keepdims=True)]), repeat)


def _tetra_tables(points):
    pkg = load_pkg()
    b = pkg.Tetra.build(points, np.array([-1.0, -1.0, -1.0, 1.0, 1.0, 1.0]))
    t = b.export()
    b.close()
    return t


def test_tetra_records_of_a_large_mesh(eng):
    """Copies of one mesh side by side, more cells than the records are built for at a time (2^20)."""
    t = _tetra_tables(np.random.default_rng(7).uniform(-1, 1, (400, 3)))
    v, tv = np.asarray(t["verts"]).reshape(-1, 3), np.asarray(t["tet_verts"]).reshape(-1, 4)
    fn, nrm = np.asarray(t["face_nb"]).reshape(-1, 4), np.asarray(t["face_normal"]).reshape(-1, 4, 3)
    n = (1 << 20) // len(tv) + 3
    q = np.arange(n)
    big = dict(verts=(v[None] + 2.25 * q[:, None, None] * np.array([1.0, 0.0, 0.0])).reshape(-1, 3),
               tet_verts=(tv[None] + len(v) * q[:, None, None]).reshape(-1, 4).astype(np.int32),
               face_nb=np.where(fn[None] < 0, -1, fn[None] + len(tv) * q[:, None, None]).reshape(-1, 4).astype(np.int32),
               face_normal=np.tile(nrm, (n, 1, 1)), box=np.array([-1.0, -1.0, -1.0, 2.25 * n - 1.25, 1.0, 1.0]))
    eng.grid_tetra(big["verts"], big["tet_verts"], big["face_nb"], big["face_normal"], big["box"])
    copies = np.concatenate([[0, 1, n // 2], np.arange(n - 5, n)])
    rays = np.concatenate([_rays(np.array([-0.9, -0.9, -0.9, 0.9, 0.9, 0.9]), v[8:], 20 + c, 25) + [2.25 * c, 0, 0, 0, 0, 0]
                           for c in copies])
    print("case tetra records of", n * len(tv), "cells", flush=True)
    _compare(eng, O.Grid("tetra", **big), rays, 1)


def test_tetra_tables_refused(eng):
    """Wrong ids anywhere in the tables are refused, also in the last cell of a mesh that several threads
    check, and the grid before stays."""
    pkg = load_pkg()
    t = _tetra_tables(np.random.default_rng(7).uniform(-1, 1, (6000, 3)))
    v, tv, fn = (np.asarray(t[k]) for k in ("verts", "tet_verts", "face_nb"))
    fn = fn.reshape(-1, 4)
    assert len(fn) > 1 << 15
    b = np.linspace(-1.0, 1.0, 5)
    eng.grid_cartesian(b, b, b)
    inner = int(np.flatnonzero((fn >= 0).all(1))[-1])
    stranger = next(m for m in range(len(fn)) if m != inner and m not in fn[inner])
    for cell in (0, inner, len(fn) - 1):
        for name, value, text in (("tet_verts", -1, "vertex"), ("tet_verts", len(v.reshape(-1, 3)), "vertex"),
                                  ("face_nb", -2, "neighbour"), ("face_nb", len(fn), "neighbour")):
            bad = dict(t, **{name: np.array(t[name]).reshape(-1, 4)})
            bad[name][cell, 3] = value
            with pytest.raises(pkg.EngineError, match=text):
                eng.grid_tetra(bad["verts"], bad["tet_verts"], bad["face_nb"], bad["face_normal"], bad["box"])
    bad = np.array(fn)
    bad[inner, 1] = stranger
    with pytest.raises(pkg.EngineError, match="mutual"):
        eng.grid_tetra(v, tv, bad, t["face_normal"], t["box"])
    assert eng.num_cells() == 64


def test_octree_of_several_threads_shares(eng):
    """A tree whose node records several threads prepare: paths bit for bit, and wrong lists in its first
    and last leaf are refused."""
    pkg = load_pkg()
    box = np.array([-1.0, -1.0, -1.0, 1.0, 1.0, 1.0])
    rng = np.random.default_rng(14)
    tree = pkg.Octree.from_flags(box, _octree_flags(box, 6, lambda lo, hi, level: level < 4 or rng.random() < 0.5))
    t = tree.export()
    tree.upload(eng)
    tree.close()
    keys = ("bounds", "child_first", "cell_index", "nb_off", "nb_id")
    print("case octree of", len(t["cell_index"]), "nodes", flush=True)
    assert len(t["cell_index"]) > 50000
    corners = np.asarray(t["bounds"]).reshape(-1, 6)[:, 3:]
    rays = _rays(box, corners[rng.integers(0, len(corners), 500)], 15)
    _compare(eng, O.Grid("octree", **{k: t[k] for k in keys}), rays, 1)
    cells = eng.num_cells()
    leaves = np.flatnonzero(np.asarray(t["cell_index"]) >= 0)
    listed = [n for n in leaves if t["nb_off"][6 * n + 6] > t["nb_off"][6 * n]]
    for n in (listed[0], listed[-1]):
        for value in (-1, len(t["cell_index"]), 0):  # (node 0 is the root, no leaf)
            bad = np.array(t["nb_id"])
            bad[t["nb_off"][6 * n]] = value
            with pytest.raises(pkg.EngineError, match="leaf"):
                eng.grid_octree(t["bounds"], t["child_first"], t["cell_index"], t["nb_off"], bad)
    assert eng.num_cells() == cells


@pytest.mark.parametrize("npk", [3000, 150_000], ids=["table_in_lds", "table_in_memory"])
def test_octree_of_many_coordinates(eng, npk):
    """A tree whose coordinate table leaves room for two of the life cycle's workgroups per compute unit:
    long runs read it from memory, short ones keep it in LDS.  Against the oracle."""
    pkg = load_pkg()
    box = np.array([-1.0, -0.9, -1.1, 1.3, 1.0, 0.8])
    size = box[3:] - box[:3]

    def diagonal(lo, hi, level):
        return max((np.array(lo) - box[:3]) / size) <= min((np.array(hi) - box[:3]) / size)

    tree = pkg.Octree.from_flags(box, _octree_flags(box, 10, diagonal))
    t = tree.export()
    tree.upload(eng)
    tree.close()
    assert 2360 < len(np.unique(t["bounds"])) <= 3200
    dens = 1e-3 * np.random.default_rng(3).lognormal(0.0, 0.5, eng.num_cells())
    eng.medium(dens)
    eng.dust([0.55e-6], [900.0], [540.0], [0.6])
    fr = frame60(npix=20)
    fr["fovx"] = fr["fovy"] = 4.0
    eng.frame_remove_all()
    eng.frame_add(fr["inclination"], fr["azimuth"], fr["roll"], fr["nx"], fr["ny"], fr["fovx"], fr["fovy"])
    src = (0.0, 0.1, -0.1)
    eng.source_point(src, [1.0 / npk])
    eng.options(0.5, 1e4, 0, 0, 13)
    eng.tune_pipeline(1)
    print("case octree of many coordinates", npk, flush=True)
    eng.run_packets(0, npk)
    img, cnt = eng.frame_read(0)[0], eng.counters()
    ofr, ocnt = O.simulate(O.Grid("octree", **{k: t[k] for k in ("bounds", "child_first", "cell_index", "nb_off", "nb_id")}),
                           dens, [0.55e-6], [900.0], [540.0], [0.6], [1.0 / npk], [fr], 0, npk, threads=8, seed=13, src=src)
    assert cnt[0] == ocnt[0] == npk
    assert abs(int(cnt[2]) - int(ocnt[2])) <= 1e-3 * ocnt[2]
    assert abs(img.sum() / ofr[0][0].sum() - 1) < 1e-6
    nz = ofr[0][0] > 0
    assert np.median(np.abs(img[nz] / ofr[0][0][nz] - 1)) < 1e-9
