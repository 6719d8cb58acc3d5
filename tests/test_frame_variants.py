"""Which kernel variants a frame takes (rz_frame_variants) — CPU only.

The raster pass that drops hidden candidates and the bin pass that takes large faces by
windows of tiles cost every frame a few percent; each case here was timed with both
variants, and the faster one is expected (both where they are within 2%)."""
import ctypes as C

import numpy as np
import pytest

import rasteriser_amd as rz
from rasteriser_amd import MaterialSpec, Scene, abi, make_args, make_faces, make_lights, scenes


def variants(scene, args, tile=16):
    desc, keep = scene.desc()
    out = (C.c_int32 * 2)(-1, -1)
    assert rz.load_library().rz_frame_variants(C.byref(desc), C.byref(args), tile, out) == 0
    del keep
    return out[0] == 1, out[1]


def triangles(n, size, edge, seed=1):
    """n raster-space triangles of 0.5..1.5 times `edge` pixels over a square image, half of
    them wound backwards."""
    rng = np.random.default_rng(seed)
    ang = rng.uniform(0, 2 * np.pi, (n, 1)) + np.array([[0, 2.1, 4.2]])
    r = rng.uniform(0.5, 1.5, (n, 1, 1)) * edge / 3 ** 0.5
    xy = rng.uniform(0, size, (n, 1, 2)) + r * np.stack([np.cos(ang), -np.sin(ang)], 2)
    verts = np.concatenate([xy, rng.uniform(0, 1, (n, 3, 1)), np.ones((n, 3, 1))], 2).reshape(-1, 4).astype(np.float32)
    tri = np.arange(3 * n).reshape(n, 3)
    back = rng.random(n) < 0.5
    tri[back] = tri[back][:, [0, 2, 1]]
    return _scene(verts, tri, True), make_args(size, size)


def cloud(n, edge, side, scale=1.0, seed=3):
    """n triangles of up to `edge` in the unit cube before the camera."""
    rng = np.random.default_rng(seed)
    c, e = rng.uniform(0, 1, (n, 3)), rng.uniform(edge / 5, edge, n)[:, None]
    d = rng.normal(size=(2, n, 3))
    d /= np.linalg.norm(d, axis=2, keepdims=True)
    pos = np.concatenate([c, c + e * d[0], c + e * d[1]], 1).reshape(-1, 3).astype(np.float32)
    args = make_args(side, side, fovy=60.0, z_near=0.1, z_far=100.0, scale=scale, displacement=(-0.5 * scale, -0.5 * scale, 0.0))
    return _scene(pos, np.arange(3 * n).reshape(n, 3), False), args


def _scene(verts, tri, raster_space):
    return Scene(verts, np.array([[0.0, 0.0, 1.0]], np.float32), np.zeros((1, 2), np.float32),
                 make_faces(tri, n=np.zeros_like(tri), t=None), [MaterialSpec((1.0, 1.0, 1.0))],
                 make_lights([[0.0, 0.0, -1.0]], [800.0], [[1.0, 1.0, 1.0]]), raster_space=raster_space)


def _n(layers, size, edge):
    return int(layers * size * size / (0.433 * edge * edge * 13 / 12))


@pytest.mark.parametrize("size,edge,layers,drop", [
    (400, 4, 40, False), (400, 8, 12, False), (1024, 8, 30, True), (400, 16, 12, False), (1024, 16, 20, True),
    (400, 16, 30, True), (1024, 32, 6, False), (1024, 32, 24, True), (400, 64, 12, False), (1024, 64, 30, True),
    (1024, 128, 12, False), (1024, 128, 40, True), (400, 300, 30, False), (1024, 300, 20, False), (1024, 300, 40, True)])
def test_hidden_candidates_in_raster_space(size, edge, layers, drop):
    """`layers` counts both windings: half of the faces are culled and hide nothing."""
    assert variants(*triangles(_n(layers, size, edge), size, edge))[0] == drop


@pytest.mark.parametrize("n,size", [(300_000, 400), (1_000_000, 512), (200_000, 300), (1_000_000, 256), (60_000, 200), (20_000, 256)])
def test_pixel_sized_triangles_are_not_overdrawn(n, size):
    assert variants(*scenes.screen_soup_scene(1, n, size)) == (False, 0)


@pytest.mark.parametrize("n,size,drop", [(100, 256, False), (200, 256, True), (400, 512, True), (3000, 1024, True), (800, 1500, True),
                                         (200, 1024, False), (100, 512, False)])
def test_screen_sized_triangles(n, size, drop):
    assert variants(*scenes.large_triangle_scene(5, n, size)) == (drop, 16)


@pytest.mark.parametrize("copies", [1, 2, 40])
@pytest.mark.parametrize("shape", ["triangle", "quad", "strip"])
def test_screen_filling_shapes(shape, copies):
    """A handful of faces, or many in one place: their centroids span no rectangle, their boxes
    do.  They meet thousands of tiles each (a single 1080p triangle's bin pass 111 us by
    atomics, 23 by windows)."""
    corners = {"triangle": [[(-10, -10), (-10, 2200), (3900, -10)]],
               "quad": [[(0, 0), (0, 1080), (1920, 0)], [(1920, 0), (0, 1080), (1920, 1080)]],
               "strip": [[(0, 500), (0, 580), (1920, 500)], [(1920, 500), (0, 580), (1920, 580)]]}[shape] * copies
    xy = np.array(corners, np.float64)
    n = len(xy)
    verts = np.concatenate([xy, np.full((n, 3, 1), 0.5), np.ones((n, 3, 1))], 2).reshape(-1, 4).astype(np.float32)
    scene = _scene(verts, np.arange(3 * n).reshape(n, 3), True)
    drop, parts = variants(scene, make_args(1920, 1080))
    assert parts == 16 and drop == (copies == 40)


def test_front_faces_alone_count():
    """One winding only: seen or culled by wind_clockwise."""
    scene, args = triangles(_n(12, 1024, 64), 1024, 64)
    verts = scene.vertices.reshape(-1, 3, 4)
    a, b = verts[:, 1] - verts[:, 0], verts[:, 2] - verts[:, 0]
    tri = np.arange(3 * len(verts)).reshape(-1, 3)
    back = a[:, 0] * b[:, 1] - a[:, 1] * b[:, 0] > 0
    assert not back.any()   # (y down: anticlockwise on the screen)
    scene = _scene(scene.vertices, tri, True)
    assert variants(scene, args)[0]
    args.wind_clockwise = 1
    assert not variants(scene, args)[0]


@pytest.mark.parametrize("n,edge,side,scale,drop", [
    (5000, 0.15, 400, 0.3, False), (50_000, 0.05, 1024, 1.0, False), (5000, 0.2, 400, 0.3, False), (5000, 0.2, 1024, 1.0, True),
    (10_000, 0.15, 400, 0.3, False), (10_000, 0.15, 1024, 1.0, True), (200_000, 0.05, 400, 1.0, False),
    (200_000, 0.05, 1920, 1.0, True), (50_000, 0.2, 1024, 1.0, True), (50_000, 0.1, 400, 0.3, False)])
def test_hidden_candidates_in_model_space(n, edge, side, scale, drop):
    assert variants(*cloud(n, edge, side, scale))[0] == drop


@pytest.mark.parametrize("detail", [2, 3, 4, 5, 6])
@pytest.mark.parametrize("width,height", [(512, 512), (1920, 1080), (3840, 2160)])
def test_closed_meshes_hide_nothing(detail, width, height):
    scene, args = scenes.icosphere_scene(subdivisions=detail, width=width, height=height, texture_size=4)
    assert not variants(scene, args)[0]


@pytest.mark.parametrize("detail,width,height,scale,wide", [
    (2, 1280, 720, 1.0, True), (2, 1280, 720, 0.4, False), (3, 1920, 1080, 1.0, True), (3, 1920, 1080, 0.6, False),
    (4, 1920, 1080, 0.4, False), (4, 3840, 2160, 1.0, True), (5, 1920, 1080, 1.0, False), (6, 3840, 2160, 1.0, False)])
def test_windows_of_tiles(detail, width, height, scale, wide):
    scene, args = scenes.icosphere_scene(subdivisions=detail, width=width, height=height, texture_size=4)
    args.scale = scale
    assert (variants(scene, args)[1] > 0) == wide


@pytest.mark.parametrize("n,edge,side,parts", [(2000, 0.2, 1024, 16), (20_000, 0.2, 1024, 6), (200_000, 0.2, 1024, 1),
                                               (200_000, 0.4, 1920, 1), (50_000, 0.2, 1920, 5), (10_000, 0.05, 400, 0)])
def test_parts_of_a_block(n, edge, side, parts):
    assert variants(*cloud(n, edge, side))[1] == parts


def test_degenerate_meshes():
    """No faces, faces of no area, and coordinates that are not finite: an answer, and the plain
    variants."""
    tri = np.arange(30).reshape(10, 3)
    for raster_space in (False, True):
        k = 4 if raster_space else 3
        for v in (np.zeros((30, k)), np.full((30, k), np.nan), np.full((30, k), np.inf)):
            assert variants(_scene(v.astype(np.float32), tri, raster_space), make_args(64, 64)) == (False, 0)
        assert variants(_scene(np.zeros((3, k), np.float32), tri[:0], raster_space), make_args(64, 64)) == (False, 0)
    scene, args = cloud(1000, 0.2, 64)
    for bad in (np.nan, np.inf):
        args.displacement[2] = bad
        assert variants(scene, args)[0] is False


def test_rejected_arguments():
    lib = rz.load_library()
    scene, args = cloud(10, 0.2, 64)
    desc, keep = scene.desc()
    out = (C.c_int32 * 2)()
    assert lib.rz_frame_variants(None, C.byref(args), 16, out) == abi.RZ_ERR_INVALID_ARG
    assert lib.rz_frame_variants(C.byref(desc), None, 16, out) == abi.RZ_ERR_INVALID_ARG
    assert lib.rz_frame_variants(C.byref(desc), C.byref(args), 12, out) == abi.RZ_ERR_INVALID_ARG
    assert lib.rz_frame_variants(C.byref(desc), C.byref(args), 16, None) == abi.RZ_ERR_INVALID_ARG
    del keep
