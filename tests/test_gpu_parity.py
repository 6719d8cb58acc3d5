"""GPU parity of the frame path: librz (through its C ABI) against the CPU oracle on
the same seeded inputs.  Face ids, depth bits and colour bytes must match exactly."""
import ctypes as C

import numpy as np
import pytest

import oracle
import rasteriser_amd as rz
from rasteriser_amd import MaterialSpec, Scene, make_args, make_faces, make_lights, scenes
from tests.parity import check

pytestmark = pytest.mark.gpu


def test_uv_sphere_512(ctx):
    scene, args = scenes.uv_sphere_scene()
    gpu, ref = check(ctx, scene, args, label="uv sphere 512")
    assert (gpu[2] >= 0).sum() > 50000


@pytest.mark.parametrize("flat", [False, True])
def test_icosphere_1080p(ctx, flat):
    scene, args = scenes.icosphere_scene(flat=flat)
    gpu, ref = check(ctx, scene, args, label=f"icosphere 1080p flat={flat}")
    assert (gpu[2] >= 0).sum() > 300000


@pytest.mark.parametrize("seed", [3, 4, 5])
def test_icosphere_1080p_more_rotations(ctx, seed):
    """The 1080p workload at further seeded rotations, lights and textures (smooth and,
    for one seed, flat): every face id, depth bit and colour byte as the oracle's."""
    scene, args = scenes.icosphere_scene(seed=seed, flat=(seed == 4))
    gpu, ref = check(ctx, scene, args, label=f"icosphere 1080p seed {seed}")
    assert (gpu[2] >= 0).sum() > 300000


@pytest.mark.parametrize("tile,cap", [(8, 64), (16, 512), (32, 2048), (16, 1), (16, 4)])
def test_tuning_and_overflow(ctx, tile, cap):
    """Every tile size, and tiny bin capacities that force the overflow path."""
    scene, args = scenes.icosphere_scene(flat=False, subdivisions=4, width=640, height=360)
    gpu, ref = check(ctx, scene, args, tuning=(tile, cap), label=f"tile {tile} cap {cap}")
    if cap <= 4:
        assert gpu[3]["overflow_tiles"] > 0


@pytest.mark.parametrize("tile,cap", [(8, 256), (16, 512), (32, 2048)])
def test_large_triangles_and_slivers(ctx, tile, cap):
    """Triangles much larger than a tile, slivers within 1e-3 px of a line and faces with a
    vertex thousands of pixels off screen: the raster pass shrinks large candidate
    rectangles to the triangle's reach, and the fragment count (every (face, pixel)
    passing the inside test) must still equal the oracle's."""
    scene, args = scenes.large_triangle_scene(n=600)
    gpu, ref = check(ctx, scene, args, tuning=(tile, cap), label=f"large triangles tile {tile}")
    assert ref[3]["fragments"] > 5_000_000


def overdraw_scene(n, W, H, seed):
    """n screen-space triangles of 3-120 px over a small image: a third flat at one of a few
    depths (ties between faces, -0 and 0, the depth a cleared pixel holds), a third steep,
    a third slivers; some with infinite or NaN depths; half wound backwards."""
    rng = np.random.default_rng(seed)
    c = rng.uniform(0, 1, (n, 1, 2)) * [W, H]
    ang = rng.uniform(0, 2 * np.pi, (n, 1)) + np.array([[0.0, 2.1, 4.2]])
    rad = np.exp(rng.uniform(np.log(3), np.log(120), (n, 1)))
    xy = c + rad[:, :, None] * np.stack([np.cos(ang), -np.sin(ang)], 2)
    kind = rng.integers(0, 3, n)
    sl = kind == 2
    xy[sl, 2] = xy[sl, 0] + (xy[sl, 1] - xy[sl, 0]) * 0.4 + rng.uniform(-0.5, 0.5, (sl.sum(), 2))
    z = rng.uniform(-1, 1, (n, 3))
    z[kind == 0] = rng.choice([-0.0, 0.0, -0.5, 0.25, 0.25 + 2.0 ** -24, 1.0], ((kind == 0).sum(), 1))
    bad = rng.random(n) < 0.02
    z[bad, rng.integers(0, 3, bad.sum())] = rng.choice([np.inf, -np.inf, np.nan], bad.sum())
    verts = np.concatenate([xy, z[:, :, None], np.ones((n, 3, 1))], 2).reshape(-1, 4).astype(np.float32)
    tri = np.arange(3 * n).reshape(n, 3)
    back = rng.random(n) < 0.5
    tri[back] = tri[back][:, [0, 2, 1]]
    scene = Scene(verts, np.array([[0.0, 0.0, 1.0]], np.float32), np.zeros((1, 2), np.float32),
                  make_faces(tri, n=np.zeros_like(tri), t=None), [MaterialSpec((0.9, 0.8, 0.7))],
                  make_lights([[0.0, 0.0, -1.0]], [200.0 * np.pi], [[1.0, 0.9, 0.8]]), raster_space=True)
    return scene, make_args(W, H)


def _draw_plain(ctx, mesh, scene, args, depth, fused=True, tuning=(16, 0)):
    """A frame drawn without statistics (the raster pass then drops hidden candidates)."""
    ctx.set_tuning(*tuning)
    ctx.set_fused_shade(fused)
    try:
        f = None if depth is None else np.full((3, args.image_height, args.image_width), 7, np.uint8)
        return ctx.draw(mesh, scene.lights_copy(), args, frame=f, depth=None if depth is None else depth.copy(),
                        ids=True)[:3]
    finally:
        ctx.set_tuning(16, 0)
        ctx.set_fused_shade(True)


def _assert_frame(got, ref, label):
    for name, a, b in zip(("face ids", "depth", "colour"), (got[2], got[1].view(np.uint32), got[0]),
                          (ref[2], ref[1].view(np.uint32), ref[0])):
        bad = np.argwhere(a != b)
        assert bad.size == 0, f"{label}: {len(bad)} {name} differ, first at {bad[:3].tolist()}"


@pytest.mark.parametrize("tuning", [(16, 0), (8, 0), (32, 0), (16, 300)])
@pytest.mark.parametrize("n,W,H", [(900, 203, 117), (6000, 64, 48), (4000, 333, 250)])
def test_hidden_candidates_dropped(ctx, n, W, H, tuning):
    """Overdraw from tens to thousands of faces a tile, tiles across the image's edges, ties
    and special depths, cleared buffers and a given depth buffer, both pipelines: frames
    drawn without statistics equal the oracle's bit for bit."""
    scene, args = overdraw_scene(n, W, H, n)
    given = np.random.default_rng(n).uniform(-0.3, 1.0, (H, W)).astype(np.float32)
    given[::7, ::5] = 0.25
    mesh = ctx.upload(scene)
    try:
        for depth in (None, given):
            f = None if depth is None else np.full((3, H, W), 7, np.uint8)
            ref = oracle.draw_frame(scene, args, frame=f, depth=depth)
            for fused in (True, False):
                got = _draw_plain(ctx, mesh, scene, args, depth, fused, tuning)
                _assert_frame(got, ref, f"n {n} {W}x{H} {tuning} depth {depth is not None} fused {fused}")
    finally:
        mesh.close()


@pytest.mark.parametrize("tile", [8, 16, 32])
@pytest.mark.parametrize("largest", [2.0 ** -149, 2.0 ** -140, 2.0 ** -131, 2.0 ** -126, 2.0 ** -101, 2.0 ** -99])
def test_hidden_candidates_dropped_subnormal_depths(ctx, tile, largest):
    """Depths so small that the products with the barycentric weights round by absolute, not
    relative, amounts (a face flat at the smallest subnormal computes 0 where its weights are
    below one half): no face may be taken to lie behind what it ties with.  Frames and batches
    drawn without statistics equal the oracle's."""
    scene, args = overdraw_scene(1500, 90, 70, 11)
    rng = np.random.default_rng(12)
    z = np.where(rng.random((1500, 1)) < 0.5, rng.choice([0.0, -0.0, 1.0, 0.5], (1500, 1)), rng.uniform(-0.2, 1, (1500, 3)))
    scene.vertices[:, 2] = (np.broadcast_to(z, (1500, 3)) * largest).astype(np.float32).ravel()
    ref = oracle.draw_frame(scene, args)
    mesh = ctx.upload(scene)
    outs = (ctx.empty((3, 70, 90), np.uint8), ctx.empty((70, 90), np.float32), ctx.empty((70, 90), np.int32))
    try:
        _assert_frame(_draw_plain(ctx, mesh, scene, args, None, tuning=(tile, 0)), ref, f"frame {tile} {largest}")
        ctx.set_tuning(tile, 0)
        ctx.draw_batch([(mesh, scene.lights_copy(), args, *outs)])
        _assert_frame([b.download() for b in outs], ref, f"batch {tile} {largest}")
    finally:
        ctx.set_tuning(16, 0)
        mesh.close()
        for b in outs:
            b.close()


def test_hidden_candidates_dropped_wide_frame_and_batch(ctx):
    """The same with 64-thread workgroups (a frame of 16,384 tiles) and in a batch, as five
    launches and as one."""
    big, bargs = scenes.large_triangle_scene(n=900, size=2048)
    ref = oracle.draw_frame(big, bargs)
    mesh = ctx.upload(big)
    try:
        _assert_frame(_draw_plain(ctx, mesh, big, bargs, None), ref, "2048x2048")
    finally:
        mesh.close()
    work = [overdraw_scene(5000, 120, 90, 1), scenes.large_triangle_scene(n=500, size=300), overdraw_scene(300, 80, 80, 2)]
    refs = [oracle.draw_frame(s, a) for s, a in work]
    meshes = [ctx.upload(s) for s, _ in work]
    outs = [tuple(ctx.empty(sh, t) for sh, t in (((3, a.image_height, a.image_width), np.uint8),
                                                 ((a.image_height, a.image_width), np.float32),
                                                 ((a.image_height, a.image_width), np.int32))) for _, a in work]
    batch = [(m, s.lights_copy(), a, *o) for m, (s, a), o in zip(meshes, work, outs)]
    try:
        for persistent in (False, True):
            for tuning in ((16, 0), (16, 8192), (8, 0), (32, 0)):
                ctx.set_batch_persistent(persistent)
                ctx.set_tuning(*tuning)
                ctx.draw_batch(batch)
                for k, (o, ref) in enumerate(zip(outs, refs)):
                    _assert_frame([b.download() for b in o], ref, f"batch item {k} persistent {persistent} {tuning}")
    finally:
        ctx.set_batch_persistent(False)
        ctx.set_tuning(16, 0)
        for m in meshes:
            m.close()
        for o in outs:
            for b in o:
                b.close()


@pytest.mark.parametrize("fused", [True, False])
@pytest.mark.parametrize("given", [False, True])
def test_hidden_candidates_dropped_one_wave_of_several_chunks(ctx, given, fused):
    """16-pixel tiles by 64-thread workgroups (16,512 tiles, the last of each row and column cut
    by the image's edge) with several chunks of 64 faces in a tile: those after the first drop
    faces behind the tile's farthest pixel.  Flat faces that tie, -0 and 0, infinite and NaN
    depths, a cleared and a given depth buffer: equal to the oracle's."""
    scene, _ = scenes.large_triangle_scene(3, 6000, 2048)
    W, H = 2041, 2063
    args = make_args(W, H)
    rng = np.random.default_rng(8)
    z = scene.vertices[:, 2].reshape(-1, 3).copy()
    flat = rng.random(len(z)) < 0.4
    z[flat] = rng.choice([-0.0, 0.0, -0.5, 0.25, 0.25 + 2.0 ** -24, 0.5, 0.75], (flat.sum(), 1))
    bad = rng.random(len(z)) < 0.02
    z[bad, rng.integers(0, 3, bad.sum())] = rng.choice([np.inf, -np.inf, np.nan], bad.sum())
    scene.vertices[:, 2] = z.ravel()
    # that the frame reaches what this is about: the variant, and some three chunks in a tile
    desc, keep = scene.desc()
    out = (C.c_int32 * 2)()
    assert rz.load_library().rz_frame_variants(C.byref(desc), C.byref(args), 16, out) == 0 and out[0] == 1
    del keep
    assert (-(-W // 16)) * (-(-H // 16)) >= 16384
    depth = frame = None
    if given:
        depth = rng.uniform(-0.3, 1.0, (H, W)).astype(np.float32)
        depth[::7, ::5] = 0.25
        frame = np.full((3, H, W), 7, np.uint8)
    ref = oracle.draw_frame(scene, args, frame=frame, depth=depth)
    mesh = ctx.upload(scene)
    try:
        _, _, _, st = ctx.draw(mesh, scene.lights_copy(), args, stats=True)
        assert st["bin_pairs"] / st["raster_tiles"] > 150
        _assert_frame(_draw_plain(ctx, mesh, scene, args, depth, fused), ref, f"given {given} fused {fused}")
    finally:
        mesh.close()


@pytest.mark.parametrize("closed,dense", [(4, 0), (4, 1), (1, 3), (0, 2)])
def test_batch_of_closed_and_overdrawn_meshes(ctx, closed, dense):
    """Batches that hide nothing, a little and most of what they draw, without statistics (their
    raster pass drops hidden candidates where that pays for the whole batch): frames, depths
    and ids equal the oracle's."""
    work = [scenes.icosphere_scene(seed=k, width=150 + 20 * k, height=130, subdivisions=3, texture_size=16) for k in range(closed)]
    work += [overdraw_scene(1500, 110, 90, k) for k in range(dense)]
    meshes = [ctx.upload(s) for s, _ in work]
    outs = [tuple(ctx.empty(sh, t) for sh, t in (((3, a.image_height, a.image_width), np.uint8),
                                                 ((a.image_height, a.image_width), np.float32),
                                                 ((a.image_height, a.image_width), np.int32))) for _, a in work]
    batch = [(m, s.lights_copy(), a, *o) for m, (s, a), o in zip(meshes, work, outs)]
    try:
        for persistent in (False, True):
            ctx.set_batch_persistent(persistent)
            ctx.draw_batch(batch)
            for k, (o, (s, a)) in enumerate(zip(outs, work)):
                _assert_frame([b.download() for b in o], oracle.draw_frame(s, a), f"item {k} persistent {persistent}")
    finally:
        ctx.set_batch_persistent(False)
        for x in (*meshes, *(b for o in outs for b in o)):
            x.close()


@pytest.mark.parametrize("tile,flags", [(16, 0), (32, 0), (16, rz.RZ_FLAG_MLP_SHADE), (32, rz.RZ_FLAG_MLP_SHADE)])
def test_time_passes_first_on_a_context(tile, flags):
    """Timing as a context's first call: the shading chain's launch may be larger than the
    frame's, and every launch must use the buffers as they are once both are prepared.  The
    frame it leaves is the plain one's."""
    scene, args = overdraw_scene(4000, 333, 250, 4000)
    with rz.Context(0) as c:
        c.set_tuning(tile, 0)
        c.mlp_init(1)
        mesh = c.upload(scene)
        f, d = c.empty((3, 250, 333), np.uint8), c.empty((250, 333), np.float32)
        us = c.time_passes(mesh, scene.lights_copy(), args, f, d, reps=3, flags=flags)
        assert us["raster"] > 0 and us["chain"] > 0
        got = f.download(), d.download()
        c.draw_device(mesh, scene.lights_copy(), args, f.ptr, d.ptr, flags=flags | rz.RZ_FLAG_CLEARED)
        assert np.array_equal(got[0], f.download())
        assert np.array_equal(got[1].view(np.uint32), oracle.draw_frame(scene, args)[1].view(np.uint32))
        for x in (mesh, f, d):
            x.close()


@pytest.mark.parametrize("fused", [True, False])
@pytest.mark.parametrize("tile", [8, 16, 32])
def test_graphs_outlive_frames_of_other_variants(tile, fused):
    """A captured frame stays valid when its context draws the same mesh and image in other
    ways: with counts, far away, close by, timed: no buffer grows, whichever
    kernel variants those frames take."""
    rng = np.random.default_rng(5)
    pos = (rng.uniform(-0.5, 0.5, (4000, 1, 3)) + rng.uniform(-0.2, 0.2, (4000, 3, 3))).reshape(-1, 3).astype(np.float32)
    tri = np.arange(12000).reshape(4000, 3)
    scene = Scene(pos, np.array([[0.0, 0.0, 1.0]], np.float32), np.zeros((1, 2), np.float32),
                  make_faces(tri, n=np.zeros_like(tri), t=None), [MaterialSpec((0.9, 0.8, 0.7))],
                  make_lights([[0.0, 0.0, -1.0]], [200.0 * np.pi], [[1.0, 0.9, 0.8]]))
    W = H = 300
    with rz.Context(0) as c:
        c.set_tuning(tile, 0)
        c.set_fused_shade(fused)
        mesh = c.upload(scene)
        f, d = c.empty((3, H, W), np.uint8), c.empty((H, W), np.float32)
        views = [make_args(W, H, scale=s) for s in (1.0, 0.01, 2.5)]
        for first in views:
            graph = c.graph(mesh, scene.lights_copy(), first, f.ptr, d.ptr, 2)
            graph.launch()
            c.sync()
            want = f.download(), d.download()
            c.draw_device(mesh, scene.lights_copy(), first, f.ptr, d.ptr, stats=True)
            for other in views:
                c.draw_device(mesh, scene.lights_copy(), other, f.ptr, d.ptr)
            c.time_passes(mesh, scene.lights_copy(), first, f, d, reps=2)
            graph.launch()
            c.sync()
            assert np.array_equal(f.download(), want[0])
            assert np.array_equal(d.download().view(np.uint32), want[1].view(np.uint32))
            graph.close()
        for x in (mesh, f, d):
            x.close()


def test_pass_times_of_a_frame_as_drawn_without_statistics(ctx):
    """RZ_FLAG_TIMES_ONLY: the times of the raster variant that plain calls run (it drops hidden
    candidates; on these triangles the counting one takes more than twice as long), no counts,
    and the frame itself, for single frames and batches of either form."""
    scene, args = scenes.large_triangle_scene(n=3000)
    H, W = args.image_height, args.image_width
    ref = oracle.draw_frame(scene, args)
    mesh = ctx.upload(scene)
    f, d = ctx.empty((3, H, W), np.uint8), ctx.empty((H, W), np.float32)
    batch = [(mesh, scene.lights_copy(), args, f, d, None)]
    flags = rz.RZ_FLAG_CLEARED

    def raster_ms(draw, flags):
        ms = []
        for _ in range(5):
            st = draw(flags)
            ms.append(st["ms_raster"])
        assert np.array_equal(d.download().view(np.uint32), ref[1].view(np.uint32))
        assert np.array_equal(f.download(), ref[0])
        counts = [st[k] for k in ("triangles", "front_triangles", "bin_pairs", "fragments", "covered_pixels", "raster_tiles")]
        assert all(c > 0 for c in counts) if not flags & rz.RZ_FLAG_TIMES_ONLY else not any(counts)
        assert st["ms_frame"] > 0
        return float(np.median(ms))

    ctx.set_profiling(True)
    try:
        for persistent in (None, False, True):
            ctx.set_batch_persistent(bool(persistent))
            draw = (lambda fl: ctx.draw_device(mesh, scene.lights_copy(), args, f.ptr, d.ptr, flags=fl, stats=True)) \
                if persistent is None else (lambda fl: ctx.draw_batch(batch, fl, stats=True))
            counted, plain = raster_ms(draw, flags), raster_ms(draw, flags | rz.RZ_FLAG_TIMES_ONLY)
            assert plain > 0
            if not persistent:   # (the one launch's phases are spans, which overlap)
                assert plain < 0.75 * counted, (persistent, plain, counted)
        ctx.set_profiling(False)
        st = ctx.draw_device(mesh, scene.lights_copy(), args, f.ptr, d.ptr, flags=flags | rz.RZ_FLAG_TIMES_ONLY, stats=True)
        assert not any(st.values())
    finally:
        ctx.set_profiling(False)
        ctx.set_batch_persistent(False)
        for x in (mesh, f, d):
            x.close()


def test_turning_mesh_whose_size_on_screen_changes(ctx):
    """A dense cloud of triangles off the axis it turns about: far away at first, near at the
    end, so that an eager frame's choice of kernel variants changes on the way.  Every frame of
    a graph and of a spin loop equals the eager frame's and the oracle's."""
    rng = np.random.default_rng(5)
    n = 4000
    c = np.array([0.0, 0.0, -1.9]) + rng.uniform(-0.3, 0.3, (n, 1, 3))
    pos = (c + rng.uniform(-0.2, 0.2, (n, 3, 3))).reshape(-1, 3).astype(np.float32)
    tri = np.arange(3 * n).reshape(n, 3)
    scene = Scene(pos, np.array([[0.0, 0.0, 1.0]], np.float32), np.zeros((1, 2), np.float32),
                  make_faces(tri, n=np.zeros_like(tri), t=None), [MaterialSpec((0.9, 0.8, 0.7))],
                  make_lights([[0.0, 0.0, -1.0]], [200.0 * np.pi], [[1.0, 0.9, 0.8]]))
    W, H, frames = 320, 240, 4
    step = float(np.float32(np.pi / (frames - 1)))
    mesh = ctx.upload(scene)
    f, d = ctx.empty((3, H, W), np.uint8), ctx.empty((H, W), np.float32)
    try:
        angles = [np.float32(0.0)]
        for _ in range(frames - 1):
            angles.append(np.float32(angles[-1] + np.float32(step)))
        spin = ctx.spin(mesh, scene.lights_copy(), make_args(W, H), f.ptr, d.ptr)
        for k, ry in enumerate(angles):
            args = make_args(W, H, angles=(0.0, float(ry), 0.0))
            ref = oracle.draw_frame(scene, args)
            graph = ctx.graph(mesh, scene.lights_copy(), make_args(W, H), f.ptr, d.ptr, k + 1, ry_step=step)
            for draw in (lambda: ctx.draw_device(mesh, scene.lights_copy(), args, f.ptr, d.ptr), graph.launch,
                         lambda: spin.frame((0.0, float(ry), 0.0))):
                draw()
                ctx.sync()
                got = f.download(), d.download()
                assert np.array_equal(got[1].view(np.uint32), ref[1].view(np.uint32)), k
                assert np.array_equal(got[0], ref[0]), k
            graph.close()
        spin.close()
    finally:
        for x in (mesh, f, d):
            x.close()


@pytest.mark.parametrize("tile,cap", [(8, 0), (16, 0), (32, 0), (16, 5)])
@pytest.mark.parametrize("wide,tiny", [(1, 0), (40, 0), (300, 200), (6, 9000)])
def test_faces_meeting_many_tiles(ctx, wide, tiny, tile, cap):
    """Faces far larger than the windows of tiles the bin pass takes them by (one face, several
    workgroups per block of faces, faces of a handful of tiles scattered between them, and
    too many faces for more than one workgroup per block), with and without overflowing
    bins: frames, face ids, depths and counts equal the oracle's."""
    W, H = 1500, 700
    rng = np.random.default_rng(wide + tiny)
    n = wide + tiny
    c = rng.uniform(0, 1, (n, 1, 2)) * [W, H]
    rad = np.where(np.arange(n) < wide, rng.uniform(60, 2500, n), rng.uniform(2, 30, n))[:, None, None]
    xy = c + rad * rng.uniform(-1, 1, (n, 3, 2))
    verts = np.concatenate([xy, rng.uniform(0, 1, (n, 3, 1)), np.ones((n, 3, 1))], 2).reshape(-1, 4).astype(np.float32)
    tri = np.arange(3 * n).reshape(n, 3)
    scene = Scene(verts, np.array([[0.0, 0.0, 1.0]], np.float32), np.zeros((1, 2), np.float32),
                  make_faces(tri, n=np.zeros_like(tri), t=None), [MaterialSpec((0.9, 0.8, 0.7))],
                  make_lights([[0.0, 0.0, -1.0]], [200.0 * np.pi], [[1.0, 0.9, 0.8]]), raster_space=True)
    gpu, ref = check(ctx, scene, make_args(W, H), tuning=(tile, cap), label=f"{wide} wide {tiny} tiny tile {tile} cap {cap}")
    mesh = ctx.upload(scene)
    try:
        _assert_frame(_draw_plain(ctx, mesh, scene, make_args(W, H), None, True, (tile, cap)), ref, "without statistics")
    finally:
        mesh.close()


@pytest.mark.parametrize("W,H", [(300, 200), (2048, 2048)])
def test_not_cleared_buffers(ctx, W, H):
    """draw_frame does not clear: the depth test reads the existing depth and pixels it
    does not win keep their old colour (drawing.cpp:119, renderer.cpp:107-108).  2048x2048
    has 16,384 tiles: 64-thread workgroups that compact the covered pixels."""
    scene, args = scenes.uv_sphere_scene(width=W, height=H)
    rng = np.random.default_rng(7)
    frame = rng.integers(0, 256, (3, H, W), dtype=np.uint8)
    depth = rng.uniform(0.85, 1.0, (H, W)).astype(np.float32)
    depth[::7, ::5] = np.float32(2.0)
    check(ctx, scene, args, frame=frame, depth=depth, label="not cleared")


@pytest.mark.parametrize("case", ["all_back", "off_screen", "one_pixel", "huge_coords"])
def test_degenerate_frames(ctx, case):
    """Frames with nothing or almost nothing to draw: (almost) every face turned to face
    away, every face off screen, a 1x1 image, and a third of the vertices at raster
    coordinates of 10^9 pixels."""
    from rasteriser_amd.scene import Scene
    scene, args = scenes.large_triangle_scene(n=300, size=256)
    v = scene.vertices.copy()
    faces = scene.faces.copy()
    if case == "all_back":
        x, y = v[faces[:, 0:3], 0].astype(np.float64), v[faces[:, 0:3], 1].astype(np.float64)
        s2 = (x[:, 0] * y[:, 1] - x[:, 1] * y[:, 0] + x[:, 1] * y[:, 2] - x[:, 2] * y[:, 1]
              + x[:, 2] * y[:, 0] - x[:, 0] * y[:, 2])
        flip = s2 < 0   # front under the raster y flip: wind them the other way
        faces[flip, 1], faces[flip, 2] = faces[flip, 2].copy(), faces[flip, 1].copy()
    elif case == "off_screen":
        v[:, 0] += 100_000.0
    elif case == "one_pixel":
        args = scenes.make_args(1, 1, fovy=60.0, z_near=0.1, z_far=100.0)
        v[:, 0:2] *= 1.0 / 256.0
    elif case == "huge_coords":
        v[::3, 0:2] *= 1e7
    scene = Scene(v, scene.normals, scene.uvs, faces, scene.materials, scene.lights, raster_space=True)
    gpu, ref = check(ctx, scene, args, label=f"degenerate {case}")
    if case == "off_screen":
        assert (gpu[2] < 0).all()
    if case == "all_back":
        assert gpu[3]["front_triangles"] < 10


def test_wind_clockwise(ctx):
    scene, args = scenes.uv_sphere_scene(width=256, height=256)
    args.wind_clockwise = 1
    check(ctx, scene, args, label="wind clockwise")


def test_screen_soup_small(ctx):
    scene, args = scenes.screen_soup_scene(n=200_000, size=1024)
    gpu, ref = check(ctx, scene, args, label="screen soup 200k")
    assert gpu[3]["front_triangles"] > 80_000


def _grid_scene(cells, step, origin, jitter, seed):
    """Screen-space grid of cells x cells quads of `step` pixels at `origin`, two
    triangles each (half wound backwards), vertices moved by up to `jitter` pixels,
    depths random: with no jitter every shared edge passes through pixel centres, whose
    edge values are exactly zero."""
    import math
    from rasteriser_amd.abi import make_args
    from rasteriser_amd.scene import MaterialSpec, Scene, make_faces, make_lights
    rng = np.random.default_rng(seed)
    g = np.arange(cells + 1, dtype=np.float64) * step + origin
    xs, ys = np.meshgrid(g, g, indexing="xy")
    xs = xs + rng.uniform(-jitter, jitter, xs.shape)
    ys = ys + rng.uniform(-jitter, jitter, ys.shape)
    n = (cells + 1) ** 2
    d = rng.uniform(0.5, 50.0, n)
    z = 1.0 - 2.0 / d
    verts = np.stack([xs.ravel(), ys.ravel(), z, 1.0 / d], 1).astype(np.float32)
    i = np.arange(cells)
    a = (i[:, None] * (cells + 1) + i[None, :]).ravel()
    tri = np.concatenate([np.stack([a, a + cells + 1, a + 1], 1), np.stack([a + 1, a + cells + 1, a + cells + 2], 1)])
    back = rng.uniform(size=len(tri)) < 0.5
    tri[back, 1], tri[back, 2] = tri[back, 2].copy(), tri[back, 1].copy()
    faces = make_faces(tri.astype(np.int64), n=np.zeros_like(tri, dtype=np.int64), t=None)
    size = int(math.ceil(origin + cells * step)) + 2
    scene = Scene(verts, np.array([[0.0, 0.0, 1.0]], np.float32), np.zeros((1, 2), np.float32), faces,
                  [MaterialSpec((1.0, 1.0, 1.0))],
                  make_lights([[0.0, 0.0, -1.0]], [255.0 * math.pi], [[1.0, 1.0, 1.0]]), raster_space=True)
    return scene, make_args(size, size, fovy=60.0, z_near=0.1, z_far=100.0)


@pytest.mark.parametrize("cells,step,origin,jitter", [(64, 8.0, 0.0, 0.0), (96, 5.0, 0.5, 0.0),
                                                      (16, 1.0, 0.0, 2.0 ** -19), (24, 0.75, 1.0, 2.0 ** -21)])
def test_edges_through_pixel_centres(ctx, cells, step, origin, jitter):
    """Candidates whose edge values are zero or near 2^-20 — the edge of the range where
    the raster pass takes its quotients from the face's reciprocal — take the general
    test; the frame must still match the oracle bit for bit (ties between faces sharing
    an edge included)."""
    scene, args = _grid_scene(cells, step, origin, jitter, seed=cells)
    for tuning in ((16, 0), (8, 64)):
        check(ctx, scene, args, tuning=tuning, label=f"grid {cells}x{step} jitter {jitter} tiles {tuning}")


def test_shared_reciprocal_quotients(ctx):
    """The raster pass's quotient from a per-face reciprocal equals the IEEE division
    bit for bit on 2^30 random operand pairs in its range (and is not used outside it)."""
    for seed in (1, 2):
        compared, bad = ctx.check_quotients(1 << 30, seed=seed)
        assert bad == 0, f"{bad} of {compared} quotients differ"
        assert compared > 0.9 * (1 << 30)


def test_screen_soup_full_4m(ctx):
    """The small-triangle depth stress at its full size: 4M screen-space triangles at
    4096x4096, about half back-facing, bit for bit against the oracle — once with the
    default bins and once with bins of 40 so that crowded tiles take the overflow path."""
    import oracle
    from tests.parity import assert_same_frame, render_gpu
    scene, args = scenes.screen_soup_scene()
    assert scene.num_faces == 4_000_000 and args.image_width == 4096
    ref = oracle.draw_frame(scene, args)
    gpu = render_gpu(ctx, scene, args)
    assert_same_frame(gpu, ref, "screen soup 4M")
    assert gpu[3]["overflow_tiles"] == 0
    assert 1_900_000 < gpu[3]["front_triangles"] < 2_100_000
    gpu = render_gpu(ctx, scene, args, tuning=(16, 40))
    assert_same_frame(gpu, ref, "screen soup 4M, bins of 40")
    assert gpu[3]["overflow_tiles"] > 1000


@pytest.mark.parametrize("tuning", [(16, 512), (16, 4), (8, 64), (32, 2048)])
def test_split_shade_pass(ctx, tuning):
    """The deferred shade as its own pass over the HBM visibility buffer (the default
    shades non-overflowed tiles inside the raster pass): same bits."""
    ctx.set_fused_shade(False)
    try:
        scene, args = scenes.icosphere_scene(subdivisions=5, width=800, height=600)
        check(ctx, scene, args, tuning=tuning, label=f"split shade {tuning}")
    finally:
        ctx.set_fused_shade(True)
    assert ctx.fused_shade


def test_repeatable(ctx):
    """Two renders of the same frame give identical visibility (order-free atomics)."""
    scene, args = scenes.icosphere_scene(subdivisions=5, width=800, height=600)
    from tests.parity import render_gpu
    a = render_gpu(ctx, scene, args)
    b = render_gpu(ctx, scene, args)
    assert np.array_equal(a[2], b[2]) and np.array_equal(a[0], b[0])
    assert np.array_equal(a[1].view(np.uint32), b[1].view(np.uint32))


def test_frame_graph_spin(ctx):
    """A captured 3-frame spin graph leaves the last frame, rotated by 2*ry_step."""
    import oracle
    from tests.parity import assert_same_frame
    scene, args = scenes.icosphere_scene(subdivisions=4, width=640, height=480)
    W, H = 640, 480
    mesh = ctx.upload(scene)
    frame = ctx.empty((3, H, W), np.uint8)
    depth = ctx.empty((H, W), np.float32)
    ids = ctx.empty((H, W), np.int32)
    lights = scene.lights_copy()
    step = 0.25
    g = ctx.graph(mesh, lights, args, frame.ptr, depth.ptr, 3, ids_ptr=ids.ptr, ry_step=step)
    for _ in range(2):          # replays must give the same result each time
        frame.upload(np.full((3, H, W), 7, np.uint8))
        g.launch()
        ctx.sync()
        last = np.float32(args.tait_bryan_angles[1])
        a2 = type(args).from_buffer_copy(args)
        a2.tait_bryan_angles[1] = float(np.float32(np.float32(last + np.float32(step)) + np.float32(step)))
        ref = oracle.draw_frame(scene, a2)
        gpu = (frame.download(), depth.download(), ids.download(),
               {"fragments": ref[3]["fragments"], "front_triangles": ref[3]["front_triangles"],
                "covered_pixels": int((ref[2] >= 0).sum())}, lights)
        assert_same_frame(gpu, ref, "graph spin")
    g.close()
    mesh.close()


def test_graph_stale_after_realloc():
    """A frame that grows the context buffers makes an older graph refuse to launch (a
    fresh context, whose buffers are sized by this test's frames alone)."""
    import rasteriser_amd as rz
    with rz.Context(0) as ctx:
        scene, args = scenes.uv_sphere_scene(width=64, height=64)
        mesh = ctx.upload(scene)
        frame = ctx.empty((3, 64, 64), np.uint8)
        depth = ctx.empty((64, 64), np.float32)
        g = ctx.graph(mesh, scene.lights_copy(), args, frame.ptr, depth.ptr, 1)
        g.launch()
        ctx.sync()
        big, bargs = scenes.uv_sphere_scene(width=2500, height=2500)
        ctx.draw(mesh, scene.lights_copy(), bargs)
        with pytest.raises(rz.RzError):
            g.launch()


def test_context_close_releases_children():
    """Closing a context first releases its meshes, graphs and device arrays; objects
    collected afterwards do not touch the destroyed context."""
    import gc
    import rasteriser_amd as rz
    ctx = rz.Context(0)
    scene, args = scenes.uv_sphere_scene(width=64, height=64)
    mesh = ctx.upload(scene)
    frame = ctx.empty((3, 64, 64), np.uint8)
    depth = ctx.empty((64, 64), np.float32)
    g = ctx.graph(mesh, scene.lights_copy(), args, frame.ptr, depth.ptr, 2)
    g.launch()
    ctx.close()
    assert mesh.handle is None and g.handle is None and frame.ptr == 0 and depth.ptr == 0
    del mesh, frame, depth, g
    gc.collect()


def _device_outputs(ctx, args, with_ids=True):
    W, H = args.image_width, args.image_height
    return (ctx.empty((3, H, W), np.uint8), ctx.empty((H, W), np.float32),
            ctx.empty((H, W), np.int32) if with_ids else None)


def test_batch_matches_single_frames_and_oracle(ctx):
    """Every mesh of one batched launch equals its own single-mesh frame bit for bit,
    and a few equal the oracle."""
    import oracle
    from tests.parity import assert_same_frame
    work = scenes.batch_scenes(n=12, seed=21, max_faces=20_000)
    meshes = [ctx.upload(s) for s, a in work]
    outs = [_device_outputs(ctx, a) for s, a in work]
    lights = [s.lights_copy() for s, a in work]
    batch = [(m, l, a, f, d, i) for m, l, (s, a), (f, d, i) in zip(meshes, lights, work, outs)]
    st = ctx.draw_batch(batch, stats=True)
    total = {"front_triangles": 0, "fragments": 0, "covered_pixels": 0}
    for k, ((scene, args), (f, d, i), m) in enumerate(zip(work, outs, meshes)):
        fb, db, ib = f.download(), d.download(), i.download()
        single = ctx.draw(m, scene.lights_copy(), args, ids=True, stats=True)
        assert np.array_equal(fb, single[0]) and np.array_equal(ib, single[2]), k
        assert np.array_equal(db.view(np.uint32), single[1].view(np.uint32)), k
        for key in total:
            total[key] += single[3][key]
        if k < 4:
            ref = oracle.draw_frame(scene, args)
            assert_same_frame((fb, db, ib, single[3], lights[k]), ref, f"batch item {k}")
    for key in total:   # the batch's statistics are the sums of its meshes'
        assert st[key] == total[key], key
    for m in meshes:
        m.close()


def test_batch_graph_and_autotune(ctx):
    """The autotuner's choice renders the same pixels; a batch graph replays them."""
    work = scenes.batch_scenes(n=6, seed=22, max_faces=30_000)
    meshes = [ctx.upload(s) for s, a in work]
    outs = [_device_outputs(ctx, a) for s, a in work]
    batch = [(m, s.lights_copy(), a, f, d, i) for m, (s, a), (f, d, i) in zip(meshes, work, outs)]
    ctx.draw_batch(batch)
    before = [(f.download(), d.download(), i.download()) for f, d, i in outs]
    ts, cap, ms = ctx.autotune(batch)
    assert ts in (8, 16, 32) and cap >= 16 and ms > 0
    assert ctx.tuning() == (ts, cap)
    g = ctx.batch_graph(batch, frames=2)
    for _ in range(2):
        for f, d, i in outs:
            f.upload(np.full(f.shape, 3, np.uint8))
        g.launch()
        ctx.sync()
        for (f, d, i), (fb, db, ib) in zip(outs, before):
            assert np.array_equal(f.download(), fb) and np.array_equal(i.download(), ib)
            assert np.array_equal(d.download().view(np.uint32), db.view(np.uint32))
    g.close()
    ctx.set_tuning(16, 0)
    for m in meshes:
        m.close()


@pytest.mark.parametrize("tile,cap", [(16, 2), (8, 1)])
def test_batch_overflow_path(ctx, tile, cap):
    work = scenes.batch_scenes(n=5, seed=23, max_faces=8_000)
    ctx.set_tuning(tile, cap)
    try:
        meshes = [ctx.upload(s) for s, a in work]
        outs = [_device_outputs(ctx, a) for s, a in work]
        batch = [(m, s.lights_copy(), a, f, d, i) for m, (s, a), (f, d, i) in zip(meshes, work, outs)]
        st = ctx.draw_batch(batch, stats=True)
        assert st["overflow_tiles"] > 0
        import oracle
        for (scene, args), (f, d, i) in list(zip(work, outs))[:3]:
            of, od, oi, _, _ = oracle.draw_frame(scene, args)
            assert np.array_equal(i.download(), oi) and np.array_equal(f.download(), of)
            assert np.array_equal(d.download().view(np.uint32), od.view(np.uint32))
    finally:
        ctx.set_tuning(16, 0)


def test_normal_map_and_64_lights(ctx):
    """The learned-shading workload's plain shader (64 lights, cone normal map) at a
    reduced size, bit for bit against the oracle."""
    scene, args = scenes.learned_shading_scene(width=640, height=360, subdivisions=5, map_size=256)
    gpu, ref = check(ctx, scene, args, label="normal map 64 lights")
    assert (gpu[2] >= 0).sum() > 20000


def test_counter_generations_across_calls():
    """Single frames keep two generations of tile counters: each frame's bin pass zeroes
    the one the next frame uses.  Eager frames, frame graphs with odd and even frame
    counts, a change of image size, the overflow path and pass timing interleaved on one
    context must each still match the oracle."""
    import oracle
    import rasteriser_amd as rz
    from tests.parity import assert_same_frame
    big, small = (640, 480), (320, 200)
    with rz.Context(0) as c:
        assert c.tuning() == (16, 0)   # default: automatic bin capacity
        scenes_by_size = {wh: scenes.icosphere_scene(subdivisions=4, width=wh[0], height=wh[1]) for wh in (big, small)}
        meshes = {wh: c.upload(sa[0]) for wh, sa in scenes_by_size.items()}
        bufs = {wh: (c.empty((3, wh[1], wh[0]), np.uint8), c.empty((wh[1], wh[0]), np.float32),
                     c.empty((wh[1], wh[0]), np.int32)) for wh in (big, small)}
        refs = {wh: oracle.draw_frame(*scenes_by_size[wh]) for wh in (big, small)}

        def compare(wh, label, stats=None):
            f, d, i = bufs[wh]
            ref = refs[wh]
            st = stats or {"fragments": ref[3]["fragments"], "front_triangles": ref[3]["front_triangles"],
                           "covered_pixels": int((ref[2] >= 0).sum())}
            assert_same_frame((f.download(), d.download(), i.download(), st, ref[4]), ref, label)

        def eager(wh, label):
            scene, args = scenes_by_size[wh]
            f, d, i = bufs[wh]
            print("eager", label, flush=True)
            st = c.draw_device(meshes[wh], scene.lights_copy(), args, f.ptr, d.ptr, i.ptr,
                               rz.RZ_FLAG_CLEARED, stats=True)
            compare(wh, label, st)

        def graph(wh, frames, label, launches=1):
            scene, args = scenes_by_size[wh]
            f, d, i = bufs[wh]
            g = c.graph(meshes[wh], scene.lights_copy(), args, f.ptr, d.ptr, frames, ids_ptr=i.ptr)
            try:
                for k in range(launches):
                    print("graph", label, frames, "frames, launch", k, flush=True)
                    i.upload(np.full((wh[1], wh[0]), 5, np.int32))
                    g.launch()
                    c.sync()
                    compare(wh, f"{label} launch {k}")
                    eager(wh, f"{label} eager after launch {k}")
            finally:
                g.close()

        eager(big, "first")
        graph(big, 3, "odd graph", launches=2)
        eager(small, "smaller image")
        graph(big, 2, "even graph", launches=2)
        eager(big, "after even graph")
        c.set_tuning(16, 4)   # overflowing bins: the overflow count lives in the counter lines
        eager(big, "overflow 1")
        eager(small, "overflow smaller")
        graph(big, 3, "overflow odd graph", launches=2)
        c.set_tuning(16, 0)
        scene, args = scenes_by_size[big]
        f, d, i = bufs[big]
        for reps in (3, 4):
            print("time_passes reps", reps, flush=True)
            c.time_passes(meshes[big], scene.lights_copy(), args, f, d, reps=reps)
            eager(big, f"after time_passes reps {reps}")
        for m in meshes.values():
            m.close()
        for b in bufs.values():
            for x in b:
                x.close()


def test_many_lights(ctx):
    """The reference shades any number of lights (shading.cpp:24-29): 200 lights (64 in
    the kernel arguments, 136 from device memory) against the oracle, eager, in a frame
    graph (its own copy of the extra lights, kept across a later frame with other lights)
    and as batch items with 65 and 300 lights."""
    import oracle
    from tests.parity import assert_same_frame
    import math
    scene, args = scenes.icosphere_scene(subdivisions=4, width=640, height=360, texture_size=256, lights=200)
    # dim lights, so that no pixel saturates and the 136 beyond the kernel arguments show
    scene.lights = scenes.random_lights(scenes.SplitMix64(0x5EED7000), 200, scale=255 * math.pi / 60)
    gpu, ref = check(ctx, scene, args, label="200 lights")
    assert (gpu[0][:, gpu[2] >= 0] == 255).mean() < 0.01
    W, H = 640, 360
    mesh = ctx.upload(scene)
    f, d, i = _device_outputs(ctx, args)
    g = ctx.graph(mesh, scene.lights_copy(), args, f.ptr, d.ptr, 2, ids_ptr=i.ptr)
    other, _ = scenes.icosphere_scene(seed=9, subdivisions=4, width=640, height=360, texture_size=256,
                                      lights=150)
    ctx.draw(mesh, other.lights_copy(), args)   # rewrites the context's extra lights
    g.launch()
    ctx.sync()
    ref = oracle.draw_frame(scene, args)
    st = {"fragments": ref[3]["fragments"], "front_triangles": ref[3]["front_triangles"],
          "covered_pixels": int((ref[2] >= 0).sum())}
    assert_same_frame((f.download(), d.download(), i.download(), st, ref[4]), ref, "200-light graph")
    g.close()
    work = [scenes.icosphere_scene(seed=s, subdivisions=3, width=256, height=200, texture_size=64, lights=n)
            for s, n in ((11, 65), (12, 300), (13, 3))]
    meshes = [ctx.upload(s) for s, a in work]
    outs = [_device_outputs(ctx, a) for s, a in work]
    batch = [(m, s.lights_copy(), a, bf, bd, bi) for m, (s, a), (bf, bd, bi) in zip(meshes, work, outs)]
    ctx.draw_batch(batch)
    for (s, a), (bf, bd, bi), item in zip(work, outs, batch):
        ref = oracle.draw_frame(s, a)
        st = {"fragments": ref[3]["fragments"], "front_triangles": ref[3]["front_triangles"],
              "covered_pixels": int((ref[2] >= 0).sum())}
        assert_same_frame((bf.download(), bd.download(), bi.download(), st, item[1]), ref,
                          f"batch item with {s.lights.shape[0]} lights")
    for m in meshes + [mesh]:
        m.close()


@pytest.mark.parametrize("W,H", [(40000, 48), (64, 65535)])
def test_image_sides_above_32767(ctx, W, H):
    """Image sides up to 65,535 pixels (bbox corners packed in 16 bits each): a 40,000-pixel
    wide and a 65,535-pixel tall frame against the oracle."""
    scene, args = scenes.uv_sphere_scene(width=W, height=H)
    gpu, ref = check(ctx, scene, args, label=f"{W}x{H}")
    assert (gpu[2] >= 0).sum() > 500


def test_spin_loop_replays(ctx):
    """rz_spin: one frame captured once, replayed with the rotation the spin loop reaches
    (renderer.cpp:117-124) — each replay equals the oracle at its angles, with eager
    frames of another size on the same context in between (they move the tile-counter
    generations the replays rely on)."""
    import oracle
    from tests.parity import assert_same_frame
    scene, args = scenes.icosphere_scene(subdivisions=4, width=640, height=480, texture_size=128)
    other, oargs = scenes.uv_sphere_scene(width=320, height=200)
    mesh, omesh = ctx.upload(scene), ctx.upload(other)
    f, d, i = _device_outputs(ctx, args)
    spin = ctx.spin(mesh, scene.lights_copy(), args, f.ptr, d.ptr, i.ptr)
    a0 = [float(x) for x in args.tait_bryan_angles]
    for k, dy in enumerate([0.0, 0.37, 1.25, 2.5, -0.6]):
        angles = [a0[0], float(np.float32(np.float32(a0[1]) + np.float32(dy))), a0[2]]
        print("spin frame", k, angles, flush=True)
        i.upload(np.full(i.shape, 3, np.int32))
        spin.frame(angles)
        ctx.sync()
        a = type(args).from_buffer_copy(args)
        a.tait_bryan_angles[:] = angles
        ref = oracle.draw_frame(scene, a)
        st = {"fragments": ref[3]["fragments"], "front_triangles": ref[3]["front_triangles"],
              "covered_pixels": int((ref[2] >= 0).sum())}
        assert_same_frame((f.download(), d.download(), i.download(), st, ref[4]), ref, f"spin frame {k}")
        if k in (1, 2):
            ctx.draw(omesh, other.lights_copy(), oargs)
    spin.close()
    for m in (mesh, omesh):
        m.close()


def test_draw_text(ctx):
    """rz_draw_text: 12x16 cells of white glyph pixels on black at (x, y), nothing else
    touched, clipped at the frame's edges."""
    W, H = 120, 40
    f = ctx.empty((3, H, W), np.uint8)
    f.upload(np.full((3, H, W), 7, np.uint8))
    ctx.draw_text(f.ptr, W, H, 5, 5, "12.5")
    ctx.draw_text(f.ptr, W, H, W - 20, H - 8, "88")   # clipped on two sides
    ctx.sync()
    img = f.download()
    box = np.zeros((H, W), bool)
    box[5:21, 5:53] = True
    box[H - 8:, W - 20:] = True
    assert (img[:, ~box] == 7).all()
    cells = img[:, box]
    assert ((cells == 255).all(axis=0) | (cells == 0).all(axis=0)).all()
    lit = (img[0, 5:21, 5:53] == 255)
    assert 40 < lit.sum() < 48 * 16 / 2
    # the four cells differ from each other (distinct glyphs) and the '.' is the smallest
    per = [lit[:, 12 * c:12 * c + 12].sum() for c in range(4)]
    assert per[2] == min(per) and len(set(per)) >= 3
    f.close()


def test_batch_256_meshes_full_size(ctx):
    """The batched workload at its stated size: 256 meshes (log-uniform 500-200k faces,
    8.5M in all, viewports 256^2-1024^2) autotuned and drawn in one batch graph.  Every
    mesh equals its own single-mesh frame at the tuned tile size and capacity, bit for bit;
    16 seeded meshes, and every mesh whose bins overflow at that capacity, equal the
    oracle (drawing.cpp:205-258 per mesh)."""
    import oracle
    from tests.parity import assert_same_frame
    work = scenes.batch_scenes()
    assert len(work) == 256 and sum(s.num_faces for s, a in work) > 8_000_000
    print("uploading 256 meshes", flush=True)
    meshes = [ctx.upload(s) for s, a in work]
    outs = [_device_outputs(ctx, a) for s, a in work]
    lights = [s.lights_copy() for s, a in work]
    batch = [(m, l, a, f, d, i) for m, l, (s, a), (f, d, i) in zip(meshes, lights, work, outs)]
    try:
        ts, cap, ms = ctx.autotune(batch)
        print("autotuned", ts, cap, ms, flush=True)
        g = ctx.batch_graph(batch, frames=2)
        for f, d, i in outs:
            i.upload(np.full(i.shape, 7, np.int32))
        g.launch()
        ctx.sync()
        g.close()
        rng = np.random.default_rng(2026)
        sample = set(rng.choice(256, 16, replace=False).tolist())
        overflowed = 0
        for k, ((scene, args), (f, d, i), m) in enumerate(zip(work, outs, meshes)):
            fb, db, ib = f.download(), d.download(), i.download()
            single = ctx.draw(m, scene.lights_copy(), args, ids=True, stats=True)
            assert np.array_equal(ib, single[2]) and np.array_equal(fb, single[0]), k
            assert np.array_equal(db.view(np.uint32), single[1].view(np.uint32)), k
            if single[3]["overflow_tiles"] > 0:
                overflowed += 1
                sample.add(k)
            if k in sample:
                print("oracle check of mesh", k, scene.num_faces, "faces", flush=True)
                ref = oracle.draw_frame(scene, args)
                assert_same_frame((fb, db, ib, single[3], lights[k]), ref, f"batch mesh {k}")
        print("meshes with overflowing bins:", overflowed, flush=True)
    finally:
        ctx.set_tuning(16, 0)
        for f, d, i in outs:
            f.close(); d.close(); i.close()
        for m in meshes:
            m.close()


@pytest.mark.parametrize("tile,cap", [(16, 512), (32, 2048), (8, 64), (16, 2)])
def test_batch_one_launch_equals_five(ctx, tile, cap):
    """A batch frame as one persistent launch and as five launches, one per pass (the
    default): the same bits and statistics, at every tile size and with overflowing bins;
    a batch graph of three frames replays the one-launch queue frame after frame."""
    work = scenes.batch_scenes(n=9, seed=41, max_faces=25_000)
    meshes = [ctx.upload(s) for s, a in work]
    outs = [_device_outputs(ctx, a) for s, a in work]
    batch = [(m, s.lights_copy(), a, f, d, i) for m, (s, a), (f, d, i) in zip(meshes, work, outs)]
    ctx.set_tuning(tile, cap)
    try:
        results = {}
        for persistent in (False, True):
            ctx.set_batch_persistent(persistent)
            print("batch", tile, cap, "persistent", persistent, flush=True)
            st = ctx.draw_batch(batch, stats=True)
            results[persistent] = (st, [(f.download(), d.download(), i.download()) for f, d, i in outs])
        (s5, r5), (s1, r1) = results[False], results[True]
        for key in ("front_triangles", "bin_pairs", "fragments", "covered_pixels", "overflow_tiles",
                    "raster_tiles", "raster_pixels"):
            assert s1[key] == s5[key], (key, s1[key], s5[key])
        if cap <= 2:
            assert s1["overflow_tiles"] > 0
        for k, (a, b) in enumerate(zip(r1, r5)):
            assert np.array_equal(a[0], b[0]) and np.array_equal(a[2], b[2]), k
            assert np.array_equal(a[1].view(np.uint32), b[1].view(np.uint32)), k
        g = ctx.batch_graph(batch, frames=3)
        for launch in range(2):
            for f, d, i in outs:
                i.upload(np.full(i.shape, 5, np.int32))
            g.launch()
            ctx.sync()
            for (f, d, i), b in zip(outs, r5):
                assert np.array_equal(i.download(), b[2]) and np.array_equal(f.download(), b[0]), launch
        g.close()
    finally:
        ctx.set_tuning(16, 0)
        ctx.set_batch_persistent(False)
        for m in meshes:
            m.close()
