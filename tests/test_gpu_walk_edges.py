"""GPU: the walk's geometry where its short cuts are decided. Triangles and
boxes that touch, cross or cover a cone's window, near and far planes, with
corners exactly on them, must give the oracle's masks, coverage and
irradiance bit for bit: a box settled from its centre and half extents, a
window cut by a triangle's edges in LDS, polygons that outgrow it, and
splatted hulls at the grid's border all have to end where the plain corner
tests and clips do."""
import numpy as np
import pytest

from continuum_amd import _lib
from continuum_amd.kernel import Flat, Scene, receivers_array
from continuum_amd.scenes import box_mesh, meshes_to_arrays, rect_light, sphere_light
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _soup(rng, n, size, lo, hi):
    """`n` random triangles about `size` across, both windings."""
    at = rng.uniform(lo, hi, (n, 1, 3))
    return (at + rng.uniform(-size, size, (n, 3, 3))).astype(np.float32)


def _aligned():
    """Squares between the origin and a 2 x 2 light 4 m up, cut at heights of
    1 and 2 m on the window's own borders, halves and eighths (all exact in
    f32), and one along the far plane."""
    out = []
    for z in (1.0, 2.0):
        s = z / 4.0
        for x0, x1, y0, y1 in ((-1, 1, -1, 1), (-1, 0, -1, 1), (0, 1, 0, 1), (-2, -1, -2, 2), (1, 3, -1, 1),
                               (-0.25, 0.5, -0.75, 0.25), (-3, 3, -3, 3)):
            a, b, c, d = ([x * s, y * s, z] for x, y in ((x0, y0), (x1, y0), (x1, y1), (x0, y1)))
            out += [[[a, c, b], [a, d, c]], [[a, b, c], [a, c, d]]]
    far = [[[-1, -1, 4], [1, 1, 4], [1, -1, 4]], [[-1, -1, 4], [-1, 1, 4], [1, 1, 4]]]
    return [np.array(m, np.float32) for m in out + [far]]


def _check(device, meshes, recv, lights, **kw):
    flat = Flat.build_arrays(*meshes_to_arrays(meshes))
    gv, gf, gt, gc = Scene(device, flat).query(recv, lights, _lib.default_options(hierarchy=2, **kw), True)
    rv, rf, rt, rc, capped, _ = O.irradiance(flat, recv, lights, O.opts_array(hierarchy=2, **kw), True)
    ok = capped == 0
    assert ok.mean() > 0.9
    assert np.array_equal(gf[ok], rf[ok]) and np.array_equal(gt[ok], rt[ok]), "masks differ"
    assert np.array_equal(gc[ok].view(np.uint32), rc[ok].view(np.uint32)), "coverage differs"
    assert np.array_equal(gv[ok].view(np.uint32), rv[ok].view(np.uint32)), "irradiance differs"
    assert int((gt != 0).sum()) > 0
    # The same points as a view, whose walks draw from the lanes' queues.
    import torch
    n, q = len(recv), len(rv)
    scene = Scene(device, flat)
    vis = torch.zeros(q, device="cuda:0")
    full, touched = (torch.zeros(q, dtype=torch.int64, device="cuda:0") for _ in range(2))
    scene.view_query_device(torch.from_numpy(recv).to("cuda:0"), n, 1, torch.from_numpy(lights).to("cuda:0"),
                            _lib.default_options(hierarchy=2, **kw), vis, full, touched, tile_w=64)
    torch.cuda.synchronize()
    assert np.array_equal(full.cpu().numpy().view(np.uint64)[ok], rf[ok]), "a view's full masks differ"
    assert np.array_equal(touched.cpu().numpy().view(np.uint64)[ok], rt[ok]), "a view's touched masks differ"
    assert np.array_equal(vis.cpu().numpy().view(np.uint32)[ok], rv[ok].view(np.uint32)), "a view's irradiance differs"


@pytest.mark.parametrize("offset", [0.0, 1000.0])
@pytest.mark.parametrize("prefilter", [0.0, 1.0, 4.0])
@pytest.mark.parametrize("size", [0.01, 0.3, 4.0])
def test_triangles_across_the_window_match_the_oracle(device, size, prefilter, offset):
    rng = np.random.default_rng(int(100 * size) + int(prefilter))
    shift = np.array([offset, -offset, 0.0], np.float32)
    # big ones cross the near and far planes too; small ones splat
    meshes = [_soup(rng, 200 if size < 4 else 24, size, [-2, -2, -0.5], [2, 2, 4.5]) + shift for _ in range(4)]
    recv = receivers_array(np.concatenate([rng.uniform([-2, -2, 0], [2, 2, 1], (333, 3)) + shift,
                                           np.tile([0.0, 0.0, 1.0], (333, 1))], 1))
    lights = np.stack([rect_light(np.array([-1, 1, 4.0]) + shift, [2, 0, 0], [0, -2, 0], one_sided=True),
                       sphere_light(np.array([1.0, 0.5, 5.0]) + shift, 0.4)])
    _check(device, meshes, recv, lights, prefilter=prefilter)


@pytest.mark.parametrize("prefilter", [0.0, 1.0, 8.0])
def test_corners_exactly_on_the_planes_match_the_oracle(device, prefilter):
    boxes = [box_mesh([x * 0.25, y * 0.25, 1.0], [x * 0.25 + 0.25, y * 0.25 + 0.25, 1.5])
             for x in (-2, -1, 0, 1) for y in (-2, -1, 0, 1)]
    points = [[0, 0, 0], [0, 0, 1], [0.25, 0.25, 0], [0.25, 0, 1.5], [-1, -1, 0], [1, 0, 2], [0, 0, -1e-4],
              [0.5, 0.5, 1.0 - 1e-4], [1.0, 1.0, 3.5]]
    recv = receivers_array([[*p, *n] for p in points for n in ([0, 0, 1], [1, 0, 0], [0.6, 0, 0.8])])
    lights = rect_light([-1, 1, 4.0], [2, 0, 0], [0, -2, 0], one_sided=True)[None]
    for meshes in ([m for m in _aligned()], boxes, [np.concatenate(_aligned())], _aligned() + boxes):
        _check(device, meshes, recv, lights, prefilter=prefilter)


@pytest.mark.parametrize("prefilter", [0.0, 1.0])
def test_sky_faces_over_touching_boxes_match_the_oracle(device, prefilter):
    """The horizon's cull on ground under the receiver and boxes whose faces
    lie in its plane, and cube faces whose diagonals pass through corners."""
    rng = np.random.default_rng(5)
    ground = np.array([[[-8, -8, 0], [8, -8, 0], [8, 8, 0]], [[-8, -8, 0], [8, 8, 0], [-8, 8, 0]]], np.float32)
    meshes = [ground, box_mesh([1, 1, 0], [2, 2, 1]), box_mesh([-2, -1, 0], [-1, 1, 2]), box_mesh([-1, 2, 1], [1, 3, 3]),
              _soup(rng, 100, 0.2, [-3, -3, 0], [3, 3, 2])]
    points = [[0, 0, 0], [0, 0, 1e-4], [0, 0, 1], [3, 3, 1], [-1.5, 0, 2], [0.5, 0.5, 0.25], [7, -7, 1e-4]]
    recv = receivers_array([[*p, *n] for p in points for n in ([0, 0, 1], [0, 1, 0], [0.6, 0, 0.8], [0, 0, -1])])
    flat = Flat.build_arrays(*meshes_to_arrays(meshes))
    out, faces, full = Scene(device, flat).sky(recv, _lib.default_options(hierarchy=2, prefilter=prefilter))
    ro, rfaces, rfull, *_ = O.sky(flat, recv, O.opts_array(hierarchy=2, prefilter=prefilter))
    assert np.array_equal(np.asarray(full).ravel(), np.asarray(rfull).ravel()), "full masks differ"
    assert np.array_equal(faces.ravel().view(np.uint32), np.asarray(rfaces, np.float32).ravel().view(np.uint32))
    assert np.array_equal(out.view(np.uint32), np.asarray(ro, np.float32).view(np.uint32))


@pytest.mark.parametrize("length", [1e-3, 100.0, 1e5])
def test_sky_normals_of_any_length_match_the_oracle(device, length):
    """A receiver's normal is taken as it comes: its horizon's plane runs
    along the faces of boxes and through the corners of a tilted grid."""
    rng = np.random.default_rng(11)
    boxes = [box_mesh([x, y, z], [x + 1, y + 1, z + 1]) for x, y, z in ((1, 0, 0), (-2, 1, -1), (0, -3, 1), (2, 2, -2))]
    n = np.array([0.36, 0.48, 0.8])
    u, v = np.array([0.8, -0.6, 0.0]), np.cross(n, [0.8, -0.6, 0.0])
    flats = np.array([[3 * a * u + 3 * b * v + k * 1e-7 * n for a, b, k in ((i, j, 1), (i + 1, j, -1), (i, j + 1, 0))]
                      for i in range(-2, 2) for j in range(-2, 2)], np.float32)
    meshes = boxes + [flats, _soup(rng, 200, 0.2, [-3, -3, -3], [3, 3, 3])]
    points = [[0, 0, 0], [0, 0, 1], [1, 1, 1], [0.5, -0.5, 0.25], [2, 2, -1]]
    recv = receivers_array([[*p, *(length * np.asarray(d, np.float64))] for p in points
                            for d in (n, [0, 0, 1], [0, 1, 0], [0.6, 0, 0.8], -n)])
    flat = Flat.build_arrays(*meshes_to_arrays(meshes))
    opts = dict(hierarchy=2, prefilter=1.0)
    out, faces, full = Scene(device, flat).sky(recv, _lib.default_options(**opts))
    ro, rfaces, rfull, *_ = O.sky(flat, recv, O.opts_array(**opts))
    assert np.array_equal(np.asarray(full).ravel(), np.asarray(rfull).ravel()), "full masks differ"
    assert np.array_equal(faces.ravel().view(np.uint32), np.asarray(rfaces, np.float32).ravel().view(np.uint32))
    assert np.array_equal(out.view(np.uint32), np.asarray(ro, np.float32).view(np.uint32))


@pytest.mark.parametrize("cap", [150, 190, 233, 300])
def test_a_waiting_splat_counts_once_against_the_node_cap(device, cap):
    """One mesh (whose children's order is fixed) of small clusters that
    splat and larger triangles that are drawn, under a small cap: a lane whose
    splat waits for its queued triangles takes the node again, and still stops
    where the list's walk (no queue) and the oracle's stop, at every query."""
    import torch
    rng = np.random.default_rng(17)
    clusters = (rng.uniform([-1, -1, 0.5], [1, 1, 3], (80, 1, 1, 3)) + rng.uniform(-0.02, 0.02, (80, 12, 1, 3)) +
                rng.uniform(-0.02, 0.02, (80, 12, 3, 3))).reshape(-1, 3, 3)
    mesh = np.concatenate([clusters.astype(np.float32), _soup(rng, 150, 0.25, [-1, -1, 0.5], [1, 1, 3])])
    flat = Flat.build_arrays(*meshes_to_arrays([mesh]))
    recv = receivers_array(np.concatenate([rng.uniform([-1, -1, -0.5], [1, 1, 0.5], (700, 3)),
                                           np.tile([0.0, 0.0, 1.0], (700, 1))], 1))
    lights = np.stack([rect_light([-0.5, 0.5, 4.0], [1, 0, 0], [0, -1, 0], one_sided=True),
                       sphere_light([0.3, 0.2, 5.0], 0.3)])
    kw = dict(hierarchy=2, prefilter=2.0, light_cone_cap=cap, wide_cone_cap=cap)
    opts = _lib.default_options(**kw)
    rv, rf, rt, _, capped, _ = O.irradiance(flat, recv, lights, O.opts_array(**kw))
    assert 0 < int(capped.sum()) < len(capped)
    scene = Scene(device, flat)
    n, q = len(recv), len(rv)
    flags = torch.zeros(q, dtype=torch.uint8, device="cuda:0")
    scene.set_query_flags(flags)
    r, l = torch.from_numpy(recv).to("cuda:0"), torch.from_numpy(lights).to("cuda:0")
    for name in ("view", "list"):
        vis = torch.zeros(q, device="cuda:0")
        full, touched = (torch.zeros(q, dtype=torch.int64, device="cuda:0") for _ in range(2))
        flags.zero_()
        if name == "view":
            scene.view_query_device(r, n, 1, l, opts, vis, full, touched, tile_w=64)
        else:
            scene.query_device(r, l, opts, vis, full, touched)
        torch.cuda.synchronize()
        assert np.array_equal(flags.cpu().numpy() & 1, capped), f"{name}: other queries stop at the cap"
        assert np.array_equal(full.cpu().numpy().view(np.uint64), rf), f"{name}: full masks differ"
        assert np.array_equal(touched.cpu().numpy().view(np.uint64), rt), f"{name}: touched masks differ"
        assert np.array_equal(vis.cpu().numpy().view(np.uint32), rv.view(np.uint32)), f"{name}: irradiance differs"
    scene.set_query_flags(None)
    # Both splats and triangles drawn, several a query.
    scene.set_count_work(True)
    scene.query_device(r, l, opts, vis, full, touched)
    torch.cuda.synchronize()
    work = scene.counters()[1]
    scene.set_count_work(False)
    assert min(int(work[3]), int(work[5])) > q, work
