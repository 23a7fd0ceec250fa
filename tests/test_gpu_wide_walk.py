"""The wide walk at the places where it could part from the binary one (GPU):
hits must equal the oracle's binary walk bit for bit.

* Rays through the shared edges and corners of a regular grid, whose
  coordinates are exact in binary: several triangles in different leaves are
  met at the very same t, and the binary walk's first must be kept.
* Slanted rays at edges and at two layers in one plane, at coordinates that are
  not exact: triangles met within a few roundings of each other.
* Scenes of one to nine triangles: a root that is a leaf, records with one to
  four children.
* Rays along the axes and through the planes of flat boxes, and from inside.
* A chain of nested boxes, every one of them met, and thin triangles as long
  as the scene: more pending nodes than the stack's LDS entries.
"""
import numpy as np
import pytest

import phiray_amd as P
from phiray_amd import scenes as S

pytestmark = pytest.mark.gpu


def rays_of(o, d, tmax=3e38):
    r = np.zeros(len(o), dtype=P.RAY)
    r["o"], r["d"], r["tmax"] = np.asarray(o, np.float32), np.asarray(d, np.float32), np.float32(tmax)
    return r


def same(gpu, orc, corners, rays, what):
    tris = S.tris_from_corners(np.asarray(corners, dtype=np.float32))
    sc = orc.Scene(tris, 4, P.NODE)
    tr = P.Tracer.new(gpu, tris, 4)
    for any_hit in (False, True):
        got = tr.raycast(rays, any_hit=any_hit).view(np.uint32).reshape(-1, 5)
        want = orc.raycast(sc.nodes, sc.tri9, rays, P.HIT, any_hit=any_hit, nthreads=8).view(np.uint32).reshape(-1, 5)
        bad = np.nonzero((got != want).any(1))[0]
        assert len(bad) == 0, f"{what} any={any_hit}: {len(bad)} hits differ, first ray {rays[bad[0]]}"
    return want


def grid(n, tilt=0.0, z=0.0):
    x, y = np.meshgrid(np.arange(n + 1), np.arange(n + 1), indexing="ij")
    p = np.stack([x / 8.0, y / 8.0, tilt * (x + 2 * y) / 8.0 + z], -1)
    a, b, c, d = p[:-1, :-1], p[1:, :-1], p[1:, 1:], p[:-1, 1:]
    return np.concatenate([np.stack([a, b, c], -2).reshape(-1, 3, 3), np.stack([a, c, d], -2).reshape(-1, 3, 3)])


@pytest.mark.parametrize("tilt", [0.0, 0.25])
def test_rays_through_shared_edges(gpu, orc, tilt):
    n = 24
    k = np.arange(4 * n + 1) / 32.0  # corners, edge middles and diagonals
    x, y = np.meshgrid(k, k, indexing="ij")
    o = np.stack([x, y, np.full_like(x, 4.0)], -1).reshape(-1, 3)
    d = np.tile([0.0, 0.0, -1.0], (len(o), 1))
    up = rays_of(np.concatenate([o, o * [1, 1, -1]]), np.concatenate([d, -d]))
    want = same(gpu, orc, grid(n, tilt), up, f"grid tilt {tilt}")
    assert (want[:, 1] != P.NONE).mean() > 0.9


def towards(corners, count, seed, spread):
    """Rays at points on the triangles' edges, from all round them."""
    rng = np.random.default_rng(seed)
    e, k, f = rng.integers(0, len(corners), count), rng.integers(0, 3, count), rng.uniform(0, 1, (count, 1))
    to = corners[e, k] * f + corners[e, (k + 1) % 3] * (1 - f)
    o = to + rng.uniform(-1, 1, (count, 3)) * spread
    d = to - o
    return o, d / np.linalg.norm(d, axis=1)[:, None], np.linalg.norm(d, axis=1)


def layers():
    """Two floors in one plane, at coordinates that are not exact in binary."""
    return np.concatenate([grid(24, z=0.1), grid(23, z=0.1) + np.array([0.03, 0.07, 0.0])]).astype(np.float32)


# Near an edge or in the overlap two triangles are met within a few roundings of
# each other, and t can round below the t of the triangle's own box: which of
# them the binary walk tests depends on its order.
@pytest.mark.parametrize("scene", ["grid", "layers", "spheres"])
def test_slanted_rays_at_edges_and_layers(gpu, orc, scene):
    if scene == "spheres":
        t = S.spheres_scene(8, 3, 1)
        corners = np.stack([t["a"], t["b"], t["c"]], 1)
    else:
        corners = grid(24, z=0.1).astype(np.float32) if scene == "grid" else layers()
    o, d, ln = towards(corners.astype(np.float64), 200_000, 6, np.array([4.0, 4.0, 4.0]))
    same(gpu, orc, corners, rays_of(o, d), scene)
    rays = rays_of(o, d)
    rays["tmax"] = ln  # a ray's end on the surface
    same(gpu, orc, corners, rays, f"{scene}, rays that end on it")


def test_frames_of_layers_are_the_same_in_every_build(gpu, orc):
    """Two floors in one plane: every build, register fit and repeat gives the
    same sums, bit for bit, and they are the oracle's."""
    tris, _ = lit(layers())
    w, h = 64, 48
    cam = S.path_camera(w, h, eye=(1.4, -1.9, 1.7), target=(1.5, 1.5, 0.1), rr_from=3)
    cam["env"] = (0.4, 0.5, 0.6, 0.0)
    px = np.zeros(P.PX_LEN * w * h + 1, dtype=np.uint32)
    sc = orc.Scene(tris, 4, P.NODE)
    for f in range(4):
        sc.sample(cam, w, h, px, f, nthreads=8)
    want = P.planes(px, w, h)
    tr = P.Tracer.new(gpu, tris, 4)
    first = None
    for build, waves in [(0, 2), (0, 4), (1, 4), (2, 4), (3, 4), (3, 4), (3, 5), (3, 2)]:
        tr.set_path_regen(build)
        tr.set_path_waves(waves)
        tr.sample(cam, w, h, 4)
        got = tr.px()
        tr.sample(S.path_camera(w + 1, h), w + 1, h, 1)  # another view: the next call starts over
        if first is None:
            first = got
            a = P.planes(got, w, h)
            for k in ("radiance", "albedo", "normal", "depth", "count", "missed"):
                assert np.allclose(a[k], want[k], rtol=1e-5, atol=0), k  # the tracer's bound against the oracle
        assert np.array_equal(got, first), (build, waves)
    b = P.Batch(gpu, np.concatenate([tris, tris]), np.array([0, len(tris), 2 * len(tris)], dtype=np.uint32))
    for build in (0, 3):
        b.set_path_build(build)
        b.render(cam, w, h, 4)
        for k in range(2):
            got = P.planes(b.px(k), w, h)
            assert np.array_equal(got["radiance"], P.planes(first, w, h)["radiance"]), (build, k)


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 6, 7, 8, 9])
def test_small_scenes(gpu, orc, n):
    corners, _ = S.lbvh_scene(n, 40 + n)
    corners = corners * np.float32(8.0)
    rng = np.random.default_rng(n)
    tgt = corners.reshape(-1, 3)[rng.integers(0, 3 * n, 400)] + rng.normal(0, 0.05, (400, 3))
    o = rng.uniform(-4, 12, (400, 3))
    same(gpu, orc, corners, rays_of(o, (tgt - o) / np.linalg.norm(tgt - o, axis=1)[:, None]), f"{n} triangles")


@pytest.mark.parametrize("n", [1, 2, 4])
@pytest.mark.parametrize("build", [0, 1, 2, 3], ids=["nested", "regen", "wavefront", "split"])
def test_a_leaf_for_a_root(gpu, orc, n, build):
    """One leaf is the whole tree: its box is tested, as the binary walk tests
    it. Some rays at a triangle's corner meet the triangle and not the box; the
    view is of a corner, many pixels to a rounding of its coordinates (with one
    triangle nine pixels have such a ray)."""
    rng = np.random.default_rng(n)
    corners = rng.uniform(0.5, 1, (n, 3, 3)).astype(np.float32)
    if build == 0:
        to = corners.reshape(-1, 3)[rng.integers(0, 3 * n, 20_000)].astype(np.float64)
        o = to + rng.uniform(-3, 3, to.shape)
        d = (to - o) / np.linalg.norm(to - o, axis=1)[:, None]
        same(gpu, orc, corners, rays_of(o, d), f"{n} triangles")
    tris, _ = lit(corners)
    corner = corners[0, 0].astype(np.float64)
    cam = S.path_camera(40, 24, eye=tuple(corner + [3.0, 0.4, 0.2]), target=tuple(corner), fov_deg=1e-5, rr_from=3)
    cam["env"] = (0.4, 0.5, 0.6, 0.0)
    sc = orc.Scene(tris, 4, P.NODE)
    px = np.zeros(P.PX_LEN * 40 * 24 + 1, dtype=np.uint32)
    rays = [0, 0]
    for f in range(8):
        r = sc.sample(cam, 40, 24, px, f, nthreads=8)
        rays = [rays[0] + r[0], rays[1] + r[1]]
    tr = P.Tracer.new(gpu, tris, 4)
    tr.set_path_regen(build)
    tr.set_path_waves(4)
    tr.sample(cam, 40, 24, 8)
    same_planes(tr.px(), px)
    assert list(tr.rays()) == rays


def test_axis_rays_flat_boxes_and_inside(gpu, orc):
    g = grid(12)
    walls = np.concatenate([g, g[:, :, [2, 0, 1]], g[:, :, [1, 2, 0]]])
    rng = np.random.default_rng(3)
    o = rng.integers(0, 49, (3000, 3)) / 32.0
    d = np.eye(3)[rng.integers(0, 3, 3000)] * rng.choice([-1.0, 1.0], 3000)[:, None]
    slant = rng.normal(size=(3000, 3)) * np.where(rng.uniform(size=(3000, 3)) < 0.3, 1e-12, 1.0)
    same(gpu, orc, walls, rays_of(np.concatenate([o, o]), np.concatenate([d, slant])), "walls")
    same(gpu, orc, walls, rays_of(np.concatenate([o, o]), np.concatenate([d, slant]), tmax=0.5), "walls, short rays")


def chain():
    """Centres at 2^-k of the scene along one axis after the other: the tree is
    a chain some 28 levels deep, eight triangles off each level, and every box
    spans the scene's middle, where the rays start: 39 nodes are pending."""
    corners = []
    for k in range(27):
        c = np.array([0.5 ** (k // 3 + (k % 3 > a)) for a in range(3)]) * 4.0 - 2.0
        half = np.minimum(np.abs(c + 4.0), np.abs(4.0 - c))
        for j in range(8):
            e = half * (1.0 - 0.001 * j)
            corners.append([c + e * [1, 1, 1], c + e * [-1, -1, 0.5], c + e * [-1, 0.25 * (j - 4), -1]])
    return np.array(corners)


def test_more_pending_nodes_than_the_stack_holds(gpu, orc):
    rng = np.random.default_rng(5)
    d = rng.normal(size=(2000, 3))
    o = rng.uniform(-0.5, 0.5, (2000, 3))
    same(gpu, orc, chain(), rays_of(o, d / np.linalg.norm(d, axis=1)[:, None]), "chain")


def lit(corners):
    """The triangles with a lamp among them, and a view from their middle."""
    tris = S.tris_from_corners(np.asarray(corners, dtype=np.float32), color=(0.7, 0.6, 0.5, 1.0))
    tris["emit"][::8] = 2.0
    cam = S.path_camera(40, 24, eye=(0.11, -0.23, 0.17), target=(0.4, 0.6, 0.3), fov_deg=90.0, rr_from=3)
    cam["env"] = (0.4, 0.5, 0.6, 0.0)
    return tris, cam


@pytest.fixture(scope="module")
def chain_frame(orc):
    tris, cam = lit(chain())
    px = np.zeros(P.PX_LEN * 40 * 24 + 1, dtype=np.uint32)
    sc = orc.Scene(tris, 4, P.NODE)
    for f in range(2):
        sc.sample(cam, 40, 24, px, f, nthreads=8)
    return tris, cam, px


def same_planes(got, want):
    a, b = P.planes(got, 40, 24), P.planes(want, 40, 24)
    for k in ("radiance", "albedo", "normal", "depth", "count", "missed"):
        assert np.allclose(a[k], b[k], rtol=1e-5, atol=0), k  # the tracer's bound against the oracle


@pytest.mark.parametrize("build", [0, 1, 2, 3], ids=["nested", "regen", "wavefront", "split"])
def test_full_stacks_in_path_frames(gpu, chain_frame, build):
    """The chain as a path frame, closest and shadow rays, at every register
    fit (the split build's stacks hold 27 entries, 19 at five waves)."""
    tris, cam, px = chain_frame
    tr = P.Tracer.new(gpu, tris, 4)
    tr.set_path_regen(build)
    for waves in (2, 3, 4, 5):
        tr.set_path_waves(waves)
        tr.sample(cam, 40, 24, 2)
        same_planes(tr.px(), px)
        tr.sample(S.path_camera(41, 24), 41, 24, 1)  # another view: the next call starts over


@pytest.mark.parametrize("build", [0, 3], ids=["nested", "split"])
def test_full_stacks_in_a_batch(gpu, chain_frame, build):
    tris, cam, px = chain_frame
    b = P.Batch(gpu, np.concatenate([tris, tris]), np.array([0, len(tris), 2 * len(tris)], dtype=np.uint32))
    b.set_path_build(build)
    for waves in (2, 3, 4, 5):
        b.set_path(waves, 0)
        b.render(cam, 40, 24, 2)
        for k in range(2):
            same_planes(b.px(k), px)


def test_a_full_stack_costs_no_second_walk(gpu):
    """4,000 thin triangles as long as the scene: a third of the rays have more
    nodes pending than the split build's 19 entries at five waves. They test
    the triangles that rays with 27 entries test, and hardly a node more."""
    rng = np.random.default_rng(4)
    c = rng.uniform(0, 1, (4000, 1, 3))
    u, v = rng.normal(size=(2, 4000, 1, 3))
    u /= 2 * np.linalg.norm(u, axis=2, keepdims=True)
    v *= 0.002 / np.linalg.norm(v, axis=2, keepdims=True)
    tris, cam = lit(np.concatenate([c - u, c + u, c + v], 1))
    tr = P.Tracer.new(gpu, tris, 4)
    tr.set_path_regen(P.Tracer.PATH_SPLIT)
    tests = {}
    for waves in (2, 5):
        before = tr.counters()[3]
        tr.set_path_waves(waves)
        tr.sample(cam, 40, 24, 1)
        tests[waves] = int(tr.counters()[3] - before)
        tr.sample(S.path_camera(41, 24, eye=(0.0, -60.0, 0.0), target=(0.0, -70.0, 0.0)), 41, 24, 1)
    assert tests[5] < 1.05 * tests[2], tests
