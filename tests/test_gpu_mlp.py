"""GPU tests of the learned shader: the matrix-core network against its numpy statement
(tests/mlp_ref.py), one training step against the numpy gradient, sample collection
against the plain shader, and the MLP-shaded frame against the network evaluated on
the collected inputs.  Coverage, depth and face ids of an MLP-shaded frame must equal
the plain frame's bit for bit; colour is an approximation whose error is measured,
not bounded by parity."""
import numpy as np
import pytest

import mlp_ref as M
import rasteriser_amd as rz
from rasteriser_amd import scenes

pytestmark = pytest.mark.gpu


def _colour_bytes(y: np.ndarray) -> np.ndarray:
    """The shading pass's conversion of network outputs to 8 bits, in float32."""
    v = y.astype(np.float32) * np.float32(255.0)
    v = np.minimum(np.maximum(v, np.float32(0.0)), np.float32(255.0))
    return np.floor(v + np.float32(0.5)).astype(np.uint8)


def test_weights_roundtrip(ctx):
    p = M.random_params(11)
    ctx.mlp_set_weights(p)
    assert np.array_equal(ctx.mlp_get_weights().view(np.uint32), p.view(np.uint32))


@pytest.mark.parametrize("n", [1, 63, 1000, 4096 + 17])
def test_infer_matches_numpy(ctx, n):
    p = M.random_params(12, scale=0.7)
    ctx.mlp_set_weights(p)
    x = np.random.default_rng(n).uniform(-1, 1, (n, M.N_IN)).astype(np.float32)
    y = ctx.mlp_infer(x)
    ref = M.forward(p, x)
    err = np.abs(y - ref)
    scale = 1.0 + np.abs(ref)
    # FP32 accumulation against float64: a hidden unit whose sum lands next to a bf16
    # rounding boundary may round the other way, so a few rows differ by more
    assert (err <= 1e-2 * scale).all(), err.max()
    assert np.mean(err <= 1e-4 * scale) > 0.9


def test_infer_empty(ctx):
    ctx.mlp_init(1)
    assert ctx.mlp_infer(np.zeros((0, 12), np.float32)).shape == (0, 3)


def test_one_training_step_matches_numpy_gradient(ctx):
    p = M.random_params(13, scale=0.5)
    ctx.mlp_set_weights(p)
    rng = np.random.default_rng(14)
    x = rng.uniform(-1, 1, M.N_IN).astype(np.float32)
    t = rng.uniform(0, 1, M.N_OUT).astype(np.float32)
    buf = ctx.empty((1, rz.RZ_MLP_SAMPLE_FLOATS), np.float32)
    try:
        buf.upload(np.concatenate([x, t])[None, :])
        lr = 1e-3
        losses = ctx.mlp_train(buf, 1, steps=1, batch=128, lr=lr, seed=3)
    finally:
        buf.close()
    loss, g = M.loss_and_grad(p, x[None, :], t[None, :])
    assert abs(losses[0] - loss) <= 1e-4 * (1 + loss), (losses[0], loss)
    delta = ctx.mlp_get_weights().astype(np.float64) - p.astype(np.float64)
    # first Adam step: delta = -lr * g / (|g| + 1e-8) = -lr * sign(g) where g is not tiny
    big = np.abs(g) > 1e-4
    assert big.sum() > 1000
    agree = np.abs(delta[big] + lr * np.sign(g[big])) <= 2e-3 * lr
    assert agree.mean() > 0.995, agree.mean()
    zero = g == 0
    assert (np.abs(delta[zero]) <= 1e-6).mean() > 0.995


def _drawn(n, batch, step, seed):
    """The samples a training step draws: SplitMix64's mix of seed, step and place, modulo n."""
    k = np.uint64(step * 1048576 + 1) + np.arange(batch, dtype=np.uint64)
    with np.errstate(over="ignore"):
        z = np.uint64(seed) + np.uint64(0x9E3779B97F4A7C15) * k
        z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        z = z ^ (z >> np.uint64(31))
    return (z % np.uint64(n)).astype(np.int64)


@pytest.mark.parametrize("n, batch", [(1, 64), (37, 64), (1000, 127), (5000, 64 * 256), (5000, 64 * 259)])
def test_training_step_over_chunks(ctx, n, batch):
    """One chunk of 64 samples, one per workgroup, and workgroups with a second chunk: the
    step's loss and the sign of every gradient that is not tiny (the first Adam step is
    -lr * sign(g)), against the numpy gradient over the same drawn samples."""
    p = M.random_params(15, scale=0.5)
    ctx.mlp_set_weights(p)
    rng = np.random.default_rng(n)
    data = np.concatenate([rng.uniform(-1, 1, (n, M.N_IN)), rng.uniform(0, 1, (n, M.N_OUT))], 1).astype(np.float32)
    buf = ctx.empty(data.shape, np.float32)
    lr = 1e-3
    try:
        buf.upload(data)
        losses = ctx.mlp_train(buf, n, steps=1, batch=batch, lr=lr, seed=21)
    finally:
        buf.close()
    rows = data[_drawn(n, batch // 64 * 64, 1, 21)]
    loss, g = M.loss_and_grad(p, rows[:, :M.N_IN], rows[:, M.N_IN:])
    assert abs(losses[0] - loss) <= 1e-4 * (1 + loss), (losses[0], loss)
    delta = ctx.mlp_get_weights().astype(np.float64) - p.astype(np.float64)
    # f32 sums of up to 16,576 terms, and a bf16 rounding of an activation falling the other
    # way for one sample in some hundreds: well under 1e-3 of the largest gradient
    big = np.abs(g) > 1e-3 * np.abs(g).max()
    assert big.sum() > 1000
    agree = np.abs(delta[big] + lr * np.sign(g[big])) <= 2e-3 * lr
    assert agree.mean() > 0.995, agree.mean()


def _grad_and_spread(p, rows):
    """The gradient over the rows, and per parameter the mean size of its samples' terms."""
    X, T = rows[:, :M.N_IN], rows[:, M.N_IN:]
    g = M.loss_and_grad(p, X, T)[1]
    W1, b1, W2, b2, W3, b3 = M.unpack(p)
    r = M._rounder(True)
    w2, w3 = r(W2), r(W3)
    a1 = r(X) @ r(W1).T + b1
    h1 = r(np.maximum(a1, 0))
    a2 = h1 @ w2.T + b2
    h2 = r(np.maximum(a2, 0))
    dy = np.abs(2.0 * (h2 @ w3.T + b3 - T) / len(X))
    d2 = (dy @ np.abs(w3)) * (a2 > 0)
    d1 = (d2 @ np.abs(w2)) * (a1 > 0)
    parts = d1.T @ np.abs(r(X)), d1.sum(0), d2.T @ h1, d2.sum(0), dy.T @ h2, dy.sum(0)
    return g, np.concatenate([q.ravel() for q in parts])


def _second_adam_step(ga, gb):
    """The second Adam update (learning rate 1) after a first one of gradient ga."""
    m, v = 0.09 * ga + 0.1 * gb, 0.000999 * ga * ga + 0.001 * gb * gb
    return -(m / (1 - 0.9 ** 2)) / (np.sqrt(v / (1 - 0.999 ** 2)) + 1e-8)


@pytest.mark.parametrize("chunks", [259, 512, 1027])
def test_gradient_over_chunks_by_value(ctx, chunks):
    """The summed gradient of a step whose workgroups take several chunks, every parameter of
    every block by value.  A step's update is invariant to its gradient's size, so a first step
    of 64 samples with learning rate 0 sets the moments and the second one's update shows the
    ratio of the two gradients.  The samples that a workgroup's first, second, ... and last
    chunks draw have targets scaled so that each of these groups makes up a like share of the
    gradient: a group lost, taken twice or mixed up moves most updates (checked with the numpy
    gradient)."""
    seed, n = 33, 1 << 18
    p = M.random_params(16, scale=0.5)
    rng = np.random.default_rng(chunks)
    data = np.concatenate([rng.uniform(-1, 1, (n, M.N_IN)), rng.uniform(0, 1, (n, M.N_OUT))], 1).astype(np.float32)
    rows_a, rows_b = _drawn(n, 64, 1, seed), _drawn(n, 64 * chunks, 2, seed)
    group = (np.arange(64 * chunks) // 64) // 256          # a workgroup's chunk number
    groups = int(group[-1]) + 1
    for k in range(groups):                                # (later groups overwrite shared rows: still known data)
        data[rows_b[group == k], M.N_IN:] *= np.float32(256.0 * 64 / (group == k).sum())
    ctx.mlp_set_weights(p)
    buf = ctx.empty(data.shape, np.float32)
    try:
        buf.upload(data)
        ctx.mlp_train(buf, n, steps=1, batch=64, lr=0.0, seed=seed)
        assert np.array_equal(ctx.mlp_get_weights(), p)
        ctx.mlp_train(buf, n, steps=1, batch=64 * chunks, lr=1.0, seed=seed)
        got = ctx.mlp_get_weights().astype(np.float64) - p.astype(np.float64)
    finally:
        buf.close()
    (ga, sa), (gb, sb) = _grad_and_spread(p, data[rows_a]), _grad_and_spread(p, data[rows_b])
    # Each gradient to 1e-3 of its terms' mean size: sums of 64 products, five chunks and 16 + 16
    # partials in f32 stay below 400 2^-24 of it, and of 64 samples a few activations may round
    # to bf16 the other way (3 / 64 of 2^-8).  The update's own f32 arithmetic: 5e-5 of it (1 -
    # 0.999^2 cancels all but 2e-3, half of that error through the root), and 2e-6 for the
    # subtraction from a weight of up to 1.
    ends = [_second_adam_step(ga + i * 1e-3 * sa, gb + j * 1e-3 * sb) for i in (-1, 0, 1) for j in (-1, 0, 1)]
    slack = 2e-6 + 5e-5 * np.abs(ends[4])
    lo, hi = np.minimum.reduce(ends) - slack, np.maximum.reduce(ends) + slack
    narrow = (hi - lo < 0.05) & (sb > 0) & (sa > 0)

    def misses(update, block):
        o = sel[block] & narrow
        return np.mean((update[o] < lo[o]) | (update[o] > hi[o])), o.sum()

    sel, at = {}, 0
    for name, size in (("W1", 768), ("b1", 64), ("W2", 4096), ("b2", 64), ("W3", 192), ("b3", 3)):
        sel[name] = np.zeros(M.N_PARAMS, bool)
        sel[name][at:at + size] = True
        at += size
    for name in sel:
        miss, count = misses(got, name)
        assert count >= 0.5 * (sel[name] & (sb > 0) & (sa > 0)).sum(), (name, count)
        assert miss <= 0.002, (name, miss, count)
    for k in range(groups):   # the same check of a gradient without one of the groups fails
        gl = _grad_and_spread(p, data[rows_b[group != k]])[0] * (group != k).mean()
        for name in ("W1", "W2", "W3"):
            assert misses(_second_adam_step(ga, gl), name)[0] > 0.5, (name, k)


def test_collect_train_and_shade(ctx):
    scene, args = scenes.learned_shading_scene(width=320, height=180, subdivisions=4, map_size=128)
    mesh = ctx.upload(scene)
    cap = 200_000
    samples = ctx.empty((cap, rz.RZ_MLP_SAMPLE_FLOATS), np.float32)
    try:
        frame_p, depth_p, ids_p, _ = ctx.draw(mesh, scene.lights_copy(), args, ids=True)
        covered = ids_p >= 0
        n = ctx.mlp_collect(mesh, scene.lights_copy(), args, samples, 0)
        assert n == int(covered.sum()) > 5000
        S = samples.download()[:n]
        feat, target = S[:, :12], S[:, 12:]
        # targets are the plain shader's bytes / 255, one per covered pixel
        got = np.sort(np.round(target * 255).astype(np.int64).view([("", np.int64)] * 3).ravel())
        want = np.sort(frame_p[:, covered].T.astype(np.int64).copy().view([("", np.int64)] * 3).ravel())
        assert np.array_equal(got, want)
        assert np.abs(np.linalg.norm(feat[:, 0:3], axis=1) - 1).max() < 1e-5
        assert np.abs(np.linalg.norm(feat[:, 3:6], axis=1) - 1).max() < 1e-5
        assert (feat[:, 5] > 0).all()   # the eye looks down -z: the view vector has +z
        assert (feat[:, 6:9] >= 0).all() and (feat[:, 6:9] <= 1).all()
        assert (np.abs(feat[:, 9:12]) <= 1).all()
        # a second collect appends behind the first
        n2 = ctx.mlp_collect(mesh, scene.lights_copy(), args, samples, n)
        assert n2 == 2 * n

        ctx.mlp_init(7)
        losses = ctx.mlp_train(samples, n, steps=400, batch=4096, lr=3e-3, seed=9)
        assert np.isfinite(losses).all()
        assert losses[-20:].mean() < 0.5 * losses[:20].mean(), (losses[:5], losses[-5:])

        frame_m, depth_m, ids_m, _ = ctx.draw(mesh, scene.lights_copy(), args, ids=True,
                                              flags=rz.RZ_FLAG_MLP_SHADE)
        assert np.array_equal(ids_m, ids_p)
        assert np.array_equal(depth_m.view(np.uint32), depth_p.view(np.uint32))
        assert (frame_m[:, ~covered] == 0).all()
        # the shaded colours are the network on the collected inputs, fragment for fragment
        y = ctx.mlp_infer(feat)
        want = np.sort(_colour_bytes(y).astype(np.int64).view([("", np.int64)] * 3).ravel())
        got = np.sort(frame_m[:, covered].T.astype(np.int64).copy().view([("", np.int64)] * 3).ravel())
        assert np.array_equal(got, want)
        err = np.abs(frame_m[:, covered].astype(np.int32) - frame_p[:, covered].astype(np.int32))
        assert err.mean() < 12.0, err.mean()
        # the separate shade pass evaluates the same network on the same inputs
        ctx.set_fused_shade(False)
        try:
            frame_s, depth_s, ids_s, _ = ctx.draw(mesh, scene.lights_copy(), args, ids=True,
                                                  flags=rz.RZ_FLAG_MLP_SHADE)
        finally:
            ctx.set_fused_shade(True)
        assert np.array_equal(frame_s, frame_m) and np.array_equal(ids_s, ids_m)
    finally:
        samples.close()
        mesh.close()


def test_learned_shader_with_narrow_workgroups(ctx):
    """At 2048x2048 (16,384 tiles) the raster pass runs 64-thread workgroups with several
    pixels per thread and compacts the covered pixels before shading: the network must
    still see the collected inputs, fragment for fragment, in both pipelines."""
    scene, args = scenes.learned_shading_scene(width=2048, height=2048, subdivisions=4, map_size=128)
    mesh = ctx.upload(scene)
    cap = 2_000_000
    samples = ctx.empty((cap, rz.RZ_MLP_SAMPLE_FLOATS), np.float32)
    try:
        frame_p, depth_p, ids_p, _ = ctx.draw(mesh, scene.lights_copy(), args, ids=True)
        covered = ids_p >= 0
        n = ctx.mlp_collect(mesh, scene.lights_copy(), args, samples, 0)
        assert n == int(covered.sum()) > 100_000
        feat = samples.download()[:n, :12]
        ctx.mlp_init(3)
        ctx.mlp_train(samples, n, steps=50, batch=4096, lr=3e-3, seed=4)
        y = ctx.mlp_infer(feat)
        want = np.sort(_colour_bytes(y).astype(np.int64).view([("", np.int64)] * 3).ravel())
        for fused in (True, False):
            ctx.set_fused_shade(fused)
            try:
                frame_m, depth_m, ids_m, _ = ctx.draw(mesh, scene.lights_copy(), args, ids=True,
                                                      flags=rz.RZ_FLAG_MLP_SHADE)
            finally:
                ctx.set_fused_shade(True)
            assert np.array_equal(ids_m, ids_p)
            assert np.array_equal(depth_m.view(np.uint32), depth_p.view(np.uint32))
            assert (frame_m[:, ~covered] == 0).all()
            got = np.sort(frame_m[:, covered].T.astype(np.int64).copy().view([("", np.int64)] * 3).ravel())
            assert np.array_equal(got, want), f"fused={fused}"
    finally:
        samples.close()
        mesh.close()


def test_mlp_flag_without_weights_is_an_error():
    c = rz.Context(0)
    try:
        scene, args = scenes.uv_sphere_scene()
        mesh = c.upload(scene)
        with pytest.raises(rz.RzError):
            c.draw(mesh, scene.lights_copy(), args, flags=rz.RZ_FLAG_MLP_SHADE)
        mesh.close()
    finally:
        c.close()


def test_batch_network_equals_single_frames(ctx):
    """Batches and single frames evaluate the network per wave inside the pass that
    shades: the same network on the same inputs, so the same bytes."""
    ctx.mlp_set_weights(M.random_params(21, scale=0.4))
    work = scenes.batch_scenes(n=4, seed=31, max_faces=20_000)
    meshes = [ctx.upload(s) for s, a in work]
    outs = []
    for s, a in work:
        W, H = a.image_width, a.image_height
        outs.append((ctx.empty((3, H, W), np.uint8), ctx.empty((H, W), np.float32), ctx.empty((H, W), np.int32)))
    try:
        batch = [(m, s.lights_copy(), a, f, d, i) for m, (s, a), (f, d, i) in zip(meshes, work, outs)]
        ctx.draw_batch(batch, flags=rz.RZ_FLAG_CLEARED | rz.RZ_FLAG_MLP_SHADE)
        for m, (s, a), (f, d, i) in zip(meshes, work, outs):
            fs, ds, ids, _ = ctx.draw(m, s.lights_copy(), a, ids=True, flags=rz.RZ_FLAG_MLP_SHADE)
            assert np.array_equal(i.download(), ids)
            assert np.array_equal(d.download().view(np.uint32), ds.view(np.uint32))
            assert np.array_equal(f.download(), fs)
            assert (ids >= 0).sum() > 1000
    finally:
        for f, d, i in outs:
            f.close(); d.close(); i.close()
        for m in meshes:
            m.close()


def test_learned_shading_full_size(ctx):
    """The learned-shading workload at its stated size: the 81,920-face icosphere at
    1920x1080 with 64 lights and a 1024x1024 cone normal map.  The plain shader equals the
    oracle bit for bit (shading.cpp:24-34 over 64 lights); the network, trained on 2^22
    fragments of the plain shader at seeded rotations, leaves ids and depth unchanged and
    stays within 2/255 mean error per channel of the plain frame at a rotation not used
    for training (the max error is reported)."""
    import oracle
    from tests.parity import check
    scene, args = scenes.learned_shading_scene()
    assert scene.lights.shape[0] == 64 and scene.materials[0].normal_map.shape[:2] == (1024, 1024)
    gpu, ref = check(ctx, scene, args, label="learned-shading workload, plain shader")
    frame_p, depth_p, ids_p = gpu[0], gpu[1], gpu[2]
    W, H = args.image_width, args.image_height
    mesh = ctx.upload(scene)
    n_target = 1 << 22
    samples = ctx.empty((n_target, rz.RZ_MLP_SAMPLE_FLOATS), np.float32)
    try:
        rng = np.random.default_rng(0x5EED2000)
        n = 0
        while n < n_target:
            a_k = rz.make_args(W, H, angles=tuple(rng.uniform(-np.pi, np.pi, 3)))
            a_k.fovy_degrees, a_k.z_near, a_k.z_far = args.fovy_degrees, args.z_near, args.z_far
            n = ctx.mlp_collect(mesh, scene.lights_copy(), a_k, samples, n)
        assert n == n_target
        ctx.mlp_init(0x5EED3000)
        losses = ctx.mlp_train(samples, n, steps=6000, batch=16384, lr=3e-3, seed=0x5EED4000)
        assert np.isfinite(losses).all()
        frame_m, depth_m, ids_m, _ = ctx.draw(mesh, scene.lights_copy(), args, ids=True,
                                              flags=rz.RZ_FLAG_MLP_SHADE)
        assert np.array_equal(ids_m, ids_p)
        assert np.array_equal(depth_m.view(np.uint32), depth_p.view(np.uint32))
        cov = ids_p >= 0
        err = np.abs(frame_m[:, cov].astype(np.int32) - frame_p[:, cov].astype(np.int32))
        mean, mx = err.mean(axis=1), err.max(axis=1)
        print("learned shader error per channel: mean", mean.tolist(), "max", mx.tolist(), flush=True)
        assert (mean <= 2.0).all(), mean
    finally:
        samples.close()
        mesh.close()
