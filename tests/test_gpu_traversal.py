"""Traversal kernels at the edges of their rules: directions outside the quick quotients' range, trees that
are one leaf, stacks that overflow, queues shorter and longer than one batch per wave."""
import numpy as np
import pytest
import torch

import yar_amd
from tests import raygen
from yar_amd import views as yv

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["zero", "two-zero", "tiny", "huge", "denormal", "mixed"])
def test_directions_outside_the_quick_range(kind, c1_path, oracle):
    """Zero, denormal, very small and very large direction components take the divided quotients and the
    case-by-case slab test; hits equal the oracle's bit for bit (the arithmetic is the same)."""
    scene = yar_amd.Scene(c1_path)
    rays = raygen.random_rays(scene, 1 << 14, seed=17)
    d = rays["direction"].astype(np.float64)
    rng = np.random.default_rng(5)
    n = rays.size
    pick = np.zeros((n, 3), bool)
    pick[np.arange(n), rng.integers(0, 3, n)] = True
    if kind == "zero":
        d[pick] = np.where(rng.random(n) < 0.5, 0.0, -0.0)
    elif kind == "two-zero":
        d[~pick] = 0.0
    elif kind == "tiny":
        d *= 2.0 ** -70
    elif kind == "huge":
        d *= 2.0 ** 70
    elif kind == "denormal":
        d[pick] = 2.0 ** -140
    else:
        d *= 2.0 ** rng.integers(-64, 64, (n, 1)).astype(np.float64)
        d[pick] *= 2.0 ** -40
    rays["direction"] = d.astype(np.float32)
    ctx = yar_amd.Context(scene)
    for any_hit in (False, True):
        if any_hit:
            rays["tmax"] = rng.uniform(0.01, 3.0, n).astype(np.float32)
        g = ctx.trace_rays(rays, any_hit=any_hit)
        o = oracle.OracleScene(scene).trace(rays, any_hit=any_hit)
        assert np.array_equal(g["t"], o["t"], equal_nan=True)
        if not any_hit:
            assert np.array_equal(g["object"], o["object"]) and np.array_equal(g["triangle"], o["triangle"])


@pytest.mark.parametrize("depth", [1, 4, 16])
def test_stack_depths_give_the_same_hits(depth, c2_small_path, oracle):
    scene = yar_amd.Scene(c2_small_path)
    rays = raygen.random_rays(scene, 1 << 15, seed=23)
    g = yar_amd.Context(scene, traversal_stack_depth=depth).trace_rays(rays)
    o = oracle.OracleScene(scene).trace(rays)
    assert np.array_equal(g["object"], o["object"]) and np.array_equal(g["triangle"], o["triangle"])
    assert np.array_equal(g["t"], o["t"])


@pytest.mark.parametrize("side,grid", [((1, 1), 1), ((7, 3), 3), ((65, 33), 2), ((256, 256), 4), ((640, 416), 2)])
def test_queue_lengths_and_refill_give_the_same_image(side, grid, c1_path):
    """A ray's result does not depend on the lanes it shares a wave with: queues of one ray, of less than a
    batch per wave (spread over all waves) and of several batches, with lanes refilled at 24, 16 and 64
    idle lanes and in blocks of one and four waves, give the same image bit for bit."""
    scene = yar_amd.Scene(c1_path)
    images = []
    for opts in ({}, {"lane_refill": 1}, {"lane_refill": 2}, {"block_size": 256}, {"max_paths_in_flight": 4096}):
        ctx = yar_amd.Context(scene, **opts)
        ctx.set_views([yv.with_film(ctx.view(0), side[0], side[1], grid, seed_offset=3)])
        img, film, var, st = ctx.render(0)
        images.append((img, film, var))
        ctx.close()
    for img, film, var in images[1:]:
        assert np.array_equal(img, images[0][0]) and np.array_equal(film, images[0][1]) and var == images[0][2]


@pytest.mark.parametrize("opts", [{}, {"use_graph": 1}, {"bin_rays": 2}, {"enable_timing": 1}], ids=["eager", "graph", "binned", "timed"])
@pytest.mark.parametrize("depth,grid,region", [(11, (1, 1), (0, 0, 33, 17)), (12, (3, 3), (100, 60, 171, 131)), (24, (4, 5), (90, 90, 140, 113))])
def test_deep_paths_in_flight_match_one_sample_per_pass(depth, grid, region, opts, scene_dir):
    """Beyond ten bounces: all samples in flight with the pixel's parked samples resumed in order, against
    one sample per pixel per pass (paths in flight below one tile's samples), bit for bit and ray for ray."""
    path = yar_amd.generate_scene(1, str(scene_dir / f"c1_depth{depth}.pbrt"), seed=1)
    text = open(path).read()
    # a white room keeps more paths alive past the tables
    lines = [l if not l.startswith('Material "matte"') else 'Material "matte" "rgb Kd" [ 0.95 0.95 0.95 ]' for l in text.splitlines()]
    text = "\n".join(lines).replace('"integer maxdepth" [ 5 ]', f'"integer maxdepth" [ {depth} ]') + "\n"
    open(path, "w").write(text)
    scene = yar_amd.Scene(path)
    out = []
    for o in (opts, {"max_paths_in_flight": 16}):
        ctx = yar_amd.Context(scene, **o)
        ctx.set_views([yv.with_film(ctx.view(0), 256, 256, grid, seed_offset=5, region=region)])
        for _ in range(2):
            img, film, var, st = ctx.render(0)
            out.append((img, film, var, st.closest_rays, st.any_rays))
        ctx.close()
    for img, film, var, closest, any_rays in out[1:]:
        assert np.array_equal(img, out[0][0]) and np.array_equal(film, out[0][1]) and var == out[0][2]
        assert (closest, any_rays) == (out[0][3], out[0][4])


@pytest.mark.parametrize("objects", [2, 6, 40])
def test_objects_in_many_scene_leaves(objects, scene_dir, oracle):
    """Long thin boxes across each other, so every one lies in many leaves of the scene tree: a ray passes
    over an object it searched before (the last four), and must still find the oracle's hits."""
    rng = np.random.default_rng(objects)
    text = ['LookAt 0 0 6 0 0 0 0 1 0', 'Camera "perspective" "float fov" [ 60 ]',
            'Film "image" "integer xresolution" [ 64 ] "integer yresolution" [ 64 ] "string filename" "o.exr"',
            'Sampler "stratified" "integer xsamples" [ 1 ] "integer ysamples" [ 1 ]', 'Integrator "path" "integer maxdepth" [ 3 ]',
            'PixelFilter "box"', 'WorldBegin', 'LightSource "point" "point from" [ 0 3 3 ] "rgb I" [ 9 9 9 ]',
            'Material "matte" "rgb Kd" [ 0.6 0.6 0.6 ]']
    corner = np.array([[x, y, z] for x in (-1, 1) for y in (-1, 1) for z in (-1, 1)], float)
    quads = [(0, 1, 3, 2), (4, 6, 7, 5), (0, 4, 5, 1), (2, 3, 7, 6), (0, 2, 6, 4), (1, 5, 7, 3)]
    idx = " ".join(f"{a} {b} {c} {a} {c} {d}" for a, b, c, d in quads)
    for k in range(objects):
        half = np.full(3, 0.04)
        half[k % 3] = 2.5
        pts = corner * half + rng.uniform(-1.5, 1.5, 3)
        text.append(f'Shape "trianglemesh" "integer indices" [ {idx} ] "point P" [ {" ".join(f"{v:.7g}" for v in pts.reshape(-1))} ]')
    path = scene_dir / f"bars{objects}.pbrt"
    path.write_text("\n".join(text) + "\nWorldEnd\n")
    scene = yar_amd.Scene(str(path))
    assert scene.desc.object_count == objects
    rays = raygen.random_rays(scene, 1 << 15, seed=objects)
    osc = oracle.OracleScene(scene)
    for any_hit in (False, True):
        if any_hit:
            rays["tmax"] = rng.uniform(0.1, 6.0, rays.size).astype(np.float32)
        g = yar_amd.Context(scene).trace_rays(rays, any_hit=any_hit)
        o = osc.trace(rays, any_hit=any_hit)
        assert np.array_equal(g["t"], o["t"])
        if not any_hit:
            assert np.array_equal(g["object"], o["object"]) and np.array_equal(g["triangle"], o["triangle"])


@pytest.mark.parametrize("grid", [(8, 16), (3, 43), (16, 16), (1, 257), (5, 103), (32, 32), (33, 32), (64, 64)],
                         ids=lambda g: f"{g[0] * g[1]}spp")
def test_long_shuffle_runs(grid, c1_path, oracle):
    """Sampler tables whose runs take 64, 32, 16, 8 and 4 lanes of a block, in bytes and 16-bit entries, in
    whole words and not: every sampler dimension of the pixels against the oracle's paths."""
    scene = yar_amd.Scene(c1_path)
    ctx = yar_amd.Context(scene)
    v = yv.with_film(ctx.view(0), 256, 256, grid, seed_offset=11, region=(120, 130, 127, 133))
    ctx.set_views([v])
    img, film, var, st = ctx.render(0)
    oimg, ofilm, ovar, _, _ = oracle.OracleScene(scene).render(v)
    rel = np.abs(img - oimg) / np.maximum(np.abs(oimg), 1e-3)
    # a wrong permutation entry moves a sample to another stratum; device sin and cos move a path by an ulp
    assert np.all(rel <= 1e-4, axis=-1).mean() >= 0.95
    assert (film["weight_sum"] == ofilm["weight_sum"]).all()
    assert abs(var - ovar) <= 1e-3 * ovar


def test_short_and_long_runs_in_one_batch(c1_path):
    """Views of different sample counts share a chunk's tables (runs of different lengths in one block)."""
    scene = yar_amd.Scene(c1_path)
    ctx = yar_amd.Context(scene)
    base = ctx.view(0)
    views = [yv.with_film(base, 64, 64, g, seed_offset=i, region=(20, 20, 33, 31))
             for i, g in enumerate([(2, 2), (20, 20), (1, 1), (7, 11), (16, 17)])]
    ctx.set_views(views)
    imgs, var, _ = ctx.render_batch(list(range(len(views))))
    for i, v in enumerate(views):
        ctx.set_views([v])
        img, _, rvar, _ = ctx.render(0, want_film=False)
        assert np.array_equal(img, imgs[i]) and rvar == var[i]


@pytest.mark.parametrize("count", [1, 63, 64, 65, 5119, 327679, 327681, 700001])
def test_ray_batches_of_every_length(count, c1_path):
    """A batch is answered ray by ray whatever its length: lengths around one wave, one ray per wave, the
    rays all waves take first (320K) and several runs per wave, as prefixes of one batch."""
    scene = yar_amd.Scene(c1_path)
    ctx = yar_amd.Context(scene)
    rays = raygen.random_rays(scene, 700001, seed=29)
    rays["tmax"] = np.where(np.arange(rays.size) % 3 == 0, 1.0, np.inf).astype(np.float32)
    for any_hit in (False, True):
        whole = np.concatenate([ctx.trace_rays(rays[i:i + 100000], any_hit=any_hit) for i in range(0, rays.size, 100000)])
        got = ctx.trace_rays(rays[:count], any_hit=any_hit)
        assert got.tobytes() == whole[:count].tobytes()


@pytest.mark.parametrize("count", [64, 400001])
def test_device_rays_and_hits_in_one_buffer(count, c1_path):
    """Hits written over the rays they answer: every ray is read before."""
    scene = yar_amd.Scene(c1_path)
    ctx = yar_amd.Context(scene)
    rays = raygen.random_rays(scene, count, seed=31)
    want = ctx.trace_rays(rays).tobytes()
    for entry in (ctx.trace_rays_device, ctx.trace_rays_device_noalloc):
        buf = torch.from_numpy(rays.view(np.uint8).reshape(-1).copy()).cuda()
        torch.cuda.synchronize()
        entry(buf.data_ptr(), count, buf.data_ptr())
        torch.cuda.synchronize()
        assert buf[:24 * count].cpu().numpy().tobytes() == want
