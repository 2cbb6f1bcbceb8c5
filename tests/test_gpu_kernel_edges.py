"""GPU tests of kernel variants at the sizes where their dispatch or their
tiling changes, against the host step or the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# (tiles across, tiles down): partial and full waves, the edges of one, four
# and eight values a thread, and the most tiles that the kernel sorts
@pytest.mark.parametrize("tiles", [(1, 1), (2, 1), (3, 2), (8, 8), (13, 5), (17, 15), (16, 16), (257, 1), (23, 89), (64, 64), (17, 241),
                                   (128, 64)])
def test_device_exposure_tile_counts(sr, scenes, env, tiles):
    """The device exposure step's sort and trimmed sum over 1 to 8192 tiles
    equal the host step's to 1e-5 relative: the order of the sum is the
    host's, so only the two libms' last bits differ, once per luminance and
    a few times in the step (1e-7 each, averaged)."""
    W, H = 64 * tiles[0], 64 * tiles[1]
    scene, spec = scenes.make_c1(width=W, height=H, subdiv=1)
    scene.prepare(env, grid=16)
    gscene = sr.Scene(scene)
    spec["yaw"] += 0.2
    r = sr.Renderer(W, H)
    r.render_scene(gscene, scenes.make_camera(spec))
    lum = r.read_tile_luminance()
    assert lum.size == tiles[0] * tiles[1]
    r.update_auto_exposure_device(0.5)
    dev = r.exposure
    r.set_exposure(2.0)
    r.update_auto_exposure(0.5)
    host = r.exposure
    r.close()
    assert abs(dev - host) <= 1e-5 * host, (dev, host)


def _glass_layers(sr, scenes, n, levels, seed):
    """n small translucent triangles facing the camera in one 64-px tile, at
    `levels` distinct depths (few levels: long runs of equal sort keys)."""
    rng = np.random.Generator(np.random.PCG64(seed))
    c = rng.uniform(-0.8, 0.8, (n, 1, 2))
    a = rng.uniform(0, 2 * np.pi, (n, 1)) + np.array([0.0, 2.1, 4.2])
    xy = c + 0.25 * np.stack([np.cos(a), np.sin(a)], -1)
    z = -2.0 - 0.5 * rng.permutation(np.arange(n) % levels) / levels
    pos = np.concatenate([xy, np.broadcast_to(z[:, None, None], (n, 3, 1))], -1).astype(np.float32).reshape(-1, 3)
    prims, mats, nodes, meshes = [], [], [], []
    for k, part in enumerate(np.array_split(np.arange(n), min(n, 5))):
        p = pos.reshape(n, 3, 3)[part].reshape(-1, 3)
        prims.append({"positions": p, "normals": np.tile(np.float32([0, 0, 1]), (len(p), 1)), "texcoords": None,
                      "tangents": None, "indices": np.arange(len(p), dtype=np.uint32), "material": k})
        mats.append({"base_color": tuple(rng.uniform(0.5, 1, 3)) + (1.0,), "metallic": 0.1, "roughness": 0.4,
                     "is_translucent": 1, "transmission": 0.7})
        meshes.append((k, 1))
        nodes.append((np.eye(4, dtype=np.float32), k))
    return sr.SceneData(prims, meshes, nodes, mats, [], name=f"glass_{n}_{levels}")


# the sort's sizes (one, two, four and eight values a thread, in LDS up to
# 4096, then blocks of 4096 merged in memory), each without and with runs of
# equal keys, down to one key for all
@pytest.mark.parametrize("n,levels", [(2, 1), (63, 63), (65, 7), (512, 512), (513, 40), (1025, 1), (2049, 2049),
                                      (2500, 700), (4096, 3), (4096, 4000), (4097, 4097), (5000, 1), (9001, 2500)])
def test_translucent_sort_sizes(sr, orc, scenes, env, n, levels):
    """Lists of 2 to 9001 translucent triangles in one tile blend in the
    oracle's order: the linear colour, which the order decides, is the
    oracle's bit for bit."""
    W = H = 60
    scene = _glass_layers(sr, scenes, n, levels, n + levels)
    scene.prepare(env, grid=16)
    cam = scenes.make_camera(scenes.camera_spec((0, 0, 0), 0.0, 0.0, np.pi / 3, W, H, 20.0))
    r = sr.Renderer(W, H)
    r.render_scene(sr.Scene(scene), cam)
    rgb = r.read_color()
    r.close()
    o = orc.OracleRenderer(W, H)
    o.render_scene(orc.OracleScene(scene), cam)
    want = o.read_frame()["rgb"]
    assert np.array_equal(rgb.view(np.uint32), np.ascontiguousarray(want, np.float32).view(np.uint32))


def test_translucent_long_list_later(sr, orc, scenes, env):
    """The room to sort a list of more than 4096 is taken when a frame first
    has one: after a frame of 7000 triangles in two tiles, whose lists fit,
    one of 5000 in one tile outgrows no other buffer and has the oracle's
    colour, and so has the next of each."""
    W, H = 128, 64
    cam = scenes.make_camera(scenes.camera_spec((0, 0, 0), 0.0, 0.0, np.pi / 3, W, H, 20.0))
    pairs = []
    for n, sides in ((7000, (-1.15, 1.15)), (5000, (1.15, 1.15))):
        scene = _glass_layers(sr, scenes, n, n, n)
        for prim in scene.primitives:
            p = prim["positions"].reshape(-1, 3, 3)
            p[::2, :, 0] += np.float32(sides[0])
            p[1::2, :, 0] += np.float32(sides[1])
        scene.rebuild()
        scene.prepare(env, grid=16)
        o = orc.OracleRenderer(W, H)
        o.render_scene(orc.OracleScene(scene), cam)
        pairs.append((sr.Scene(scene), np.ascontiguousarray(o.read_frame()["rgb"], np.float32)))
    r = sr.Renderer(W, H)
    for k in (0, 1, 0, 1):
        r.render_scene(pairs[k][0], cam)
        assert np.array_equal(r.read_color().view(np.uint32), pairs[k][1].view(np.uint32)), k
    r.close()


@pytest.mark.parametrize("size", [(16, 16), (63, 65), (130, 97)])
def test_translucent_walk_edges(sr, orc, scenes, env, size):
    """The forward pass keeps only the entries that meet each 16x16 block
    and masks them per pixel 64 at a time: 300 triangles from a few pixels
    to the whole view (kept counts below and above 64 and 256), partly off
    screen, some behind an opaque triangle, over blocks cut by the view's
    edges.  The linear colour and the tiles' luminance are the oracle's bit
    for bit."""
    W, H = size
    rng = np.random.Generator(np.random.PCG64(W))
    scene = _glass_layers(sr, scenes, 300, 300, 11)
    for k, prim in enumerate(scene.primitives):
        p = prim["positions"].reshape(-1, 3, 3)
        mid = p.mean(1, keepdims=True)
        p[:] = mid + (p - mid) * np.exp(rng.uniform(np.log(0.2), np.log(12.0), (len(p), 1, 1))) * \
            np.array([1.0, 1.0, 0.0], np.float32)
    quad = np.array([[-0.5, -2, -2.3], [2, -2, -2.3], [2, 2, -2.3]], np.float32)
    scene.primitives.append({"positions": quad, "normals": np.tile(np.float32([0, 0, 1]), (3, 1)), "texcoords": None,
                             "tangents": None, "indices": np.arange(3, dtype=np.uint32),
                             "material": len(scene.materials)})
    scene.materials.append({"base_color": (0.4, 0.5, 0.6, 1.0), "metallic": 0.0, "roughness": 0.6})
    scene.meshes.append((len(scene.primitives) - 1, 1))
    scene.nodes.append((np.eye(4, dtype=np.float32), len(scene.meshes) - 1))
    scene.rebuild()
    scene.prepare(env, grid=16)
    cam = scenes.make_camera(scenes.camera_spec((0, 0, 0), 0.0, 0.0, np.pi / 3, W, H, 20.0))
    r = sr.Renderer(W, H)
    r.render_scene(sr.Scene(scene), cam)
    rgb, lum = r.read_color(), r.read_tile_luminance()
    r.close()
    o = orc.OracleRenderer(W, H)
    o.render_scene(orc.OracleScene(scene), cam)
    want = o.read_frame()["rgb"]
    assert np.array_equal(rgb.view(np.uint32), np.ascontiguousarray(want, np.float32).view(np.uint32))
    assert np.array_equal(lum.view(np.uint32), np.asarray(o.tile_luminance(), np.float32).view(np.uint32))


@pytest.mark.parametrize("blocks", [1, 3, 8, 64, 100, 4096])
def test_persistent_raster_block_counts(sr, scenes, env, blocks):
    """Persistent raster workgroups below, at and above the item count (one
    workgroup for all items, counts that do not divide them, more workgroups
    than items): every view equals the batch with one workgroup per item."""
    scene, spec = scenes.make_c1(width=160, height=90, spheres=6, subdiv=2)
    scene.prepare(env, grid=16)
    gscene = sr.Scene(scene)
    views = []
    for k, (w, h) in enumerate(((160, 90), (1, 1), (65, 130), (96, 64))):
        s = dict(spec)
        s["yaw"] = 0.05 * k
        views.append((gscene, scenes.make_camera(s, w, h), w, h, 0.0))
    b = sr.Batch()
    out = []
    for persistent in (-1, blocks):
        b.configure(persistent_blocks=persistent)
        b.render(views)
        out.append([(*b.read_vbuffer(i), b.read_pixels(i)) for i in range(len(views))])
    b.close()
    for want, got in zip(*out):
        for x, y in zip(want, got):
            assert np.array_equal(x.view(np.uint32), y.view(np.uint32))


# list lengths around the groups of 64 and the batches of 256 that the
# overdraw raster sorts; "hole" leaves part of the view uncovered, so no
# quadrant there ever rejects, and "flat" puts all triangles at two depths
@pytest.mark.parametrize("n", [40, 64, 65, 129, 256, 257, 520])
@pytest.mark.parametrize("kind", ["full", "hole", "flat"])
def test_overdraw_raster_list_lengths(sr, orc, n, kind):
    """n large triangles over every tile of a 64x48 view (odd tile rows off
    screen): the frame takes the overdraw raster on its second rendering and
    both renderings have the oracle's visibility buffer."""
    from util import attach_dummy, screen_triangle_scene
    W, H = 64, 48
    rng = np.random.default_rng(1000 * n + len(kind))
    c = rng.uniform([0, 0], [W * 16, H * 16], (n, 1, 2))
    ang = rng.uniform(0, 2 * np.pi, (n, 1)) + np.array([0.0, 2.1, 4.2]) + rng.uniform(-0.4, 0.4, (n, 3))
    rad = rng.uniform(40, 90, (n, 3)) * 16
    tris = np.round(c + np.stack([np.cos(ang), np.sin(ang)], -1) * rad[..., None])
    if kind == "hole":
        tris[..., 0] = np.minimum(tris[..., 0], 40 * 16)
    a = (tris[:, 1, 0] - tris[:, 0, 0]) * (tris[:, 2, 1] - tris[:, 0, 1]) - \
        (tris[:, 2, 0] - tris[:, 0, 0]) * (tris[:, 1, 1] - tris[:, 0, 1])
    tris[a > 0] = tris[a > 0][:, ::-1]
    depths = rng.uniform(2.0, 90.0, (n, 1)) * rng.uniform(0.9, 1.1, (n, 3))
    if kind == "flat":
        depths = np.where(rng.random((n, 1)) < 0.5, 10.0, 20.0) * np.ones((n, 3))
    scene, spec = screen_triangle_scene(sr, tris, depths, W, H)
    attach_dummy(sr, scene)
    import swraster_viewer_amd.scenes as sc
    cam = sc.make_camera(spec)
    o = orc.OracleRenderer(W, H)
    o.render_scene(orc.OracleScene(scene), cam)
    want = o.read_frame()
    gscene = sr.Scene(scene)
    r = sr.Renderer(W, H)
    for k in range(2):
        r.render_scene(gscene, cam)
        ids, depth = r.read_vbuffer()
        assert np.array_equal(ids, want["ids"]), f"frame {k}"
        assert np.array_equal(depth.view(np.uint32), want["depth"].view(np.uint32)), f"frame {k}"
    assert r.stats()["depth_rejection"] == 1
    r.close()


# pairs a tile on both sides of the overdraw raster's line: 56 with fewer than
# 512 tiles (320 here), 32 from there on (512)
@pytest.mark.parametrize("W,H,pairs,near", [(320, 240, 45, 0), (320, 240, 80, 1), (512, 256, 24, 0), (512, 256, 45, 1)])
def test_overdraw_raster_line(sr, orc, W, H, pairs, near):
    """The raster that a second frame takes follows the pairs a tile, and both
    frames have the oracle's visibility buffer."""
    from util import attach_dummy, screen_triangle_scene
    import swraster_viewer_amd.scenes as sc
    rng = np.random.default_rng(pairs)
    n = pairs * W * H // 256 // 25                 # 40-px triangles take about 25 tiles each
    c = rng.uniform([0, 0], [W * 16, H * 16], (n, 1, 2))
    ang = rng.uniform(0, 2 * np.pi, (n, 1)) + np.array([0.0, 2.1, 4.2])
    tris = np.round(c + np.stack([np.cos(ang), np.sin(ang)], -1) * 640)
    a = (tris[:, 1, 0] - tris[:, 0, 0]) * (tris[:, 2, 1] - tris[:, 0, 1]) - \
        (tris[:, 2, 0] - tris[:, 0, 0]) * (tris[:, 1, 1] - tris[:, 0, 1])
    tris[a > 0] = tris[a > 0][:, ::-1]
    scene, spec = screen_triangle_scene(sr, tris, rng.uniform(2.0, 90.0, n), W, H)
    attach_dummy(sr, scene)
    cam = sc.make_camera(spec)
    o = orc.OracleRenderer(W, H)
    o.render_scene(orc.OracleScene(scene), cam)
    want = o.read_frame()
    gscene = sr.Scene(scene)
    r = sr.Renderer(W, H)
    for k in range(2):
        r.render_scene(gscene, cam)
        ids, depth = r.read_vbuffer()
        assert np.array_equal(ids, want["ids"]), f"frame {k}"
        assert np.array_equal(depth.view(np.uint32), want["depth"].view(np.uint32)), f"frame {k}"
    st = r.stats()
    r.close()
    assert st["depth_rejection"] == near, st["binned_pairs"] / st["tiles"]


# sizes that leave part of a tile, whole quadrants or whole tiles off the
# screen, the centre quad of a 64-px tile among them (32 rows: just off it)
@pytest.mark.parametrize("size", [(64, 32), (70, 40), (33, 97), (47, 34), (640, 360)])
def test_overdraw_raster_screen_edges(sr, orc, size):
    """Large triangles reaching past the right and bottom edge: both
    renderings (the second by the overdraw raster) have the oracle's
    visibility buffer and tile luminance."""
    from util import attach_dummy, screen_triangle_scene
    import swraster_viewer_amd.scenes as sc
    W, H = size
    n = 300 + W * H // 80
    rng = np.random.default_rng(W + H)
    c = rng.uniform([0, 0], [(W + 20) * 16, (H + 20) * 16], (n, 1, 2))
    ang = rng.uniform(0, 2 * np.pi, (n, 1)) + np.array([0.0, 2.1, 4.2]) + rng.uniform(-0.4, 0.4, (n, 3))
    tris = np.round(c + np.stack([np.cos(ang), np.sin(ang)], -1) * (rng.uniform(40, 90, (n, 3)) * 16)[..., None])
    a = (tris[:, 1, 0] - tris[:, 0, 0]) * (tris[:, 2, 1] - tris[:, 0, 1]) - \
        (tris[:, 2, 0] - tris[:, 0, 0]) * (tris[:, 1, 1] - tris[:, 0, 1])
    tris[a > 0] = tris[a > 0][:, ::-1]
    scene, spec = screen_triangle_scene(sr, tris, rng.uniform(2.0, 90.0, (n, 1)) * rng.uniform(0.9, 1.1, (n, 3)), W, H)
    attach_dummy(sr, scene)
    cam = sc.make_camera(spec)
    o = orc.OracleRenderer(W, H)
    o.render_scene(orc.OracleScene(scene), cam)
    want = o.read_frame()
    gscene = sr.Scene(scene)
    r = sr.Renderer(W, H)
    for k in range(2):
        r.render_scene(gscene, cam)
        ids, depth = r.read_vbuffer()
        assert np.array_equal(ids, want["ids"]), f"frame {k}"
        assert np.array_equal(depth.view(np.uint32), want["depth"].view(np.uint32)), f"frame {k}"
        assert np.array_equal(r.read_tile_luminance().view(np.uint32),
                              np.asarray(o.tile_luminance(), np.float32).view(np.uint32)), f"frame {k}"
    assert r.stats()["depth_rejection"] == 1
    r.close()


# the raster variants with the alpha test: each tile size, and the overdraw
# raster (tile 16, a list of 300); "far" minifies the texture to its last levels
@pytest.mark.parametrize("n,tile,far", [(24, 8, False), (24, 16, True), (24, 32, False), (300, 16, False),
                                        (300, 16, True), (300, 32, True)])
def test_alpha_raster_variants(sr, orc, n, tile, far):
    """n large triangles over a 64x48 view, two in three cut out by their
    texture's alpha, the rest opaque: both renderings have the oracle's
    visibility buffer, the second of 300 at 16-px tiles by the overdraw raster."""
    from util import attach_dummy, screen_triangle_scene
    import swraster_viewer_amd.scenes as sc
    W, H = 64, 48
    rng = np.random.default_rng(n + tile)
    c = rng.uniform([0, 0], [W * 16, H * 16], (n, 1, 2))
    ang = rng.uniform(0, 2 * np.pi, (n, 1)) + np.array([0.0, 2.1, 4.2]) + rng.uniform(-0.4, 0.4, (n, 3))
    tris = np.round(c + np.stack([np.cos(ang), np.sin(ang)], -1) * (rng.uniform(40, 90, (n, 3)) * 16)[..., None])
    a = (tris[:, 1, 0] - tris[:, 0, 0]) * (tris[:, 2, 1] - tris[:, 0, 1]) - \
        (tris[:, 2, 0] - tris[:, 0, 0]) * (tris[:, 1, 1] - tris[:, 0, 1])
    tris[a > 0] = tris[a > 0][:, ::-1]
    scene, spec = screen_triangle_scene(sr, tris, rng.uniform(2.0, 90.0, (n, 1)) * rng.uniform(0.9, 1.1, (n, 3)), W, H)
    p, mat = scene.primitives[0], scene.materials[0]
    uv = (rng.uniform(-2, 2, (3 * n, 2)) * (40.0 if far else 1.0)).astype(np.float32)
    tex = (32, 32, sr.SR_TEX_SRGB, sr.pack_rgba(rng.integers(0, 256, (32 * 32, 4), dtype=np.uint8)).ravel())
    prims, mats = [], []
    for k, part in enumerate(np.array_split(np.arange(3 * n).reshape(n, 3), 3)):
        part = part.reshape(-1)
        prims.append({"positions": p["positions"][part], "normals": p["normals"][part], "texcoords": uv[part],
                      "tangents": None, "indices": np.arange(len(part), dtype=np.uint32), "material": k})
        mats.append(dict(mat, **({} if k == 1 else {
            "alpha_mode": sr.SR_ALPHA_MASK, "alpha_cutoff": 0.3 + 0.2 * k,
            "base_color_tex": (0, sr.SR_WRAP_REPEAT, sr.SR_WRAP_MIRRORED_REPEAT)})))
    scene = sr.SceneData(prims, [(0, 3)], list(scene.nodes), mats, [tex], name="cut")
    attach_dummy(sr, scene)
    cam = sc.make_camera(spec)
    o = orc.OracleRenderer(W, H)
    o.render_scene(orc.OracleScene(scene), cam)
    want = o.read_frame()
    r = sr.Renderer(W, H, tile_size=tile)
    gscene = sr.Scene(scene)
    for k in range(2):
        r.render_scene(gscene, cam)
        ids, depth = r.read_vbuffer()
        assert np.array_equal(ids, want["ids"]), f"frame {k}"
        assert np.array_equal(depth.view(np.uint32), want["depth"].view(np.uint32)), f"frame {k}"
    assert n < 300 or r.stats()["depth_rejection"] == int(tile == 16)
    r.close()


def _with_backfacing(sr, scene, n):
    """scene plus a last primitive of n copies of one backfacing triangle in
    every mesh-bearing node's place: they make records without bins, so the
    tiles' lists stay the same while the frame has n more triangles."""
    import copy
    prims = [dict(p) for p in scene.primitives]
    tri = np.array([[0.0, 0.0, 0.0], [0.0, 1e-3, 0.0], [1e-3, 0.0, 0.0]], np.float32)
    prims.append({"positions": tri, "normals": np.tile(np.float32([0, 0, 1]), (3, 1)), "texcoords": None,
                  "tangents": None, "indices": np.tile(np.arange(3, dtype=np.uint32), n), "material": 0})
    first, count = scene.meshes[-1]
    assert first + count == len(prims) - 1
    meshes = list(scene.meshes[:-1]) + [(first, count + 1)]
    out = sr.SceneData(prims, meshes, list(scene.nodes), copy.deepcopy(scene.materials), list(scene.textures))
    return out


# small frames by direct binning against the same frames by radix passes,
# which 262,144 more triangles (1024 chunks) make them take: tile counts of
# one, a few and exactly 8192, sizes that leave tiles off screen, all tile
# sizes; "near" stands close to the terrain, so many triangles cross the
# frustum, "mixed" has rectangles of more than 32 tiles among small ones and
# more pairs than a first frame has room for (it runs again, direct still)
@pytest.mark.parametrize("kind,W,H,tile", [("cluster", 16, 16, 32), ("cluster", 64, 64, 16), ("cluster", 333, 202, 8),
                                           ("cluster", 2048, 1024, 16), ("near", 640, 360, 16), ("near", 500, 301, 32),
                                           ("mixed", 640, 480, 16), ("mixed", 1023, 130, 8)])
def test_direct_binning_equals_radix(sr, scenes, env, kind, W, H, tile):
    """The tiles' lists, the visibility buffer and the pair count of a small
    frame are those that the radix passes give, and so are the views of a
    batch of three."""
    if kind == "cluster":
        scene, spec = scenes.make_c1(width=W, height=H)
        # one node: all spheres in world space, so the copies come last
        prims = []
        for (t, m) in scene.nodes:
            p = dict(scene.primitives[m])
            p["positions"] = (p["positions"] @ np.asarray(t, np.float32)[:3, :3].T + np.asarray(t, np.float32)[:3, 3])
            prims.append(p)
        scene = sr.SceneData(prims, [(0, len(prims))], [(np.eye(4, dtype=np.float32), 0)], scene.materials,
                             scene.textures)
    elif kind == "near":
        scene, spec = scenes.make_c2(width=W, height=H, grid=120, tex_size=64)
        spec["position"] = [0.0, 4.0, 10.0]
    else:
        from util import mixed_triangle_scene
        scene, spec = mixed_triangle_scene(sr, W, H, 12000, 4 * tile)
    more = _with_backfacing(sr, scene, 262144)
    scene.prepare(env, grid=16)
    more.attach(scene.environment, scene.voxels)
    cam = scenes.make_camera(spec, W, H)
    out = []
    for data in (scene, more):
        r = sr.Renderer(W, H, tile_size=tile)
        gscene = sr.Scene(data)
        r.render_scene(gscene, cam)
        ids, depth = r.read_vbuffer()
        out.append((ids, depth.view(np.uint32), *r.read_bins(), r.stats()["binned_pairs"]))
        assert r.direct_binning() == (data is scene)
        r.close()
        if data is scene:
            b = sr.Batch(tile_size=tile)
            b.render([(gscene, cam, W, H, 0.0), (gscene, cam, 50, 70, 0.0), (gscene, cam, W, H, 0.0)])
            views = [b.read_vbuffer(k) for k in (0, 2)]
            b.close()
    if kind == "mixed":
        assert out[0][5] > 2 * (12000 + 12000 // 8 + 1024)       # the first frame's room
    for ids, depth in views:
        assert np.array_equal(ids, out[1][0]) and np.array_equal(depth.view(np.uint32), out[1][1])
    assert out[0][5] == out[1][5] and out[0][5] > 0
    for a, b in zip(out[0][:5], out[1][:5]):
        assert np.array_equal(a, b)
    assert np.all(np.diff(out[0][2].astype(np.int64)) >= 0) and out[0][3][-1] == out[0][5]


def _mixed(sr, scenes, W, H, n, radius, huge=0):
    from util import attach_dummy, mixed_triangle_scene
    scene, spec = mixed_triangle_scene(sr, W, H, n, radius, huge)
    attach_dummy(sr, scene)
    return scene, scenes.make_camera(spec, W, H)


def test_large_triangles_leave_direct_binning(sr, scenes):
    """A frame with three screen-filling triangles among small ones is binned
    by the radix passes: a renderer's first frame, a frame after small ones,
    and as long as the last one had such triangles; frames without them go
    back to the direct binning.  All have the frame that radix passes give."""
    W, H = 640, 360
    small, cam = _mixed(sr, scenes, W, H, 3000, 40)
    large, _ = _mixed(sr, scenes, W, H, 3000, 40, huge=3)
    want = {}
    for name, data in (("small", small), ("large", large)):
        more = _with_backfacing(sr, data, 262144)
        more.attach(data.environment, data.voxels)
        r = sr.Renderer(W, H)
        r.render_scene(sr.Scene(more), cam)
        assert not r.direct_binning()
        want[name] = (*r.read_vbuffer(), *r.read_bins())
        r.close()
    gpu = {"small": sr.Scene(small), "large": sr.Scene(large)}
    r = sr.Renderer(W, H)
    for k, (name, direct) in enumerate((("large", False), ("large", False), ("small", False), ("small", True),
                                        ("large", False), ("small", False), ("small", True))):
        r.render_scene(gpu[name], cam)
        got = (*r.read_vbuffer(), *r.read_bins())
        assert r.direct_binning() == direct, (k, name)
        for x, y in zip(got, want[name]):
            assert np.array_equal(x.view(np.uint32), y.view(np.uint32)), (k, name)
    r.close()


def _gi(sr, scene, env, grid, device):
    g = sr.sr_voxel_grid()
    scene.environment = env
    scene.desc.environment = sr.C.pointer(env.desc)
    sr.check(sr.lib().sr_prepare_gi(sr.C.byref(scene.desc), grid, device, 8, sr.C.byref(g)))
    sh4 = np.ctypeslib.as_array(g.sh4, shape=(grid ** 3 * 16,)).copy()
    sr.lib().sr_voxel_grid_free(sr.C.byref(g))
    return sh4.view(np.uint32)


# a tree whose root is a leaf (up to four triangles), one inner node, a few
# levels; grids whose active voxels leave waves of the last workgroup empty;
# the translucent variant with rays through many layers
@pytest.mark.parametrize("n,grid,glass", [(1, 5, False), (4, 9, False), (5, 9, False), (9, 7, True), (40, 13, False),
                                          (40, 13, True), (700, 16, True)])
def test_gi_tree_sizes(sr, scenes, env, n, grid, glass):
    """The device GI bake over trees of 1 to 700 triangles equals the host
    bake bit for bit."""
    rng = np.random.Generator(np.random.PCG64(n))
    pos = (rng.uniform(-2, 2, (n, 1, 3)) + rng.normal(0, 0.8, (n, 3, 3))).astype(np.float32).reshape(-1, 3)
    half = 3 * (n // 2)
    prims, mats = [], []
    for k, (a, b) in enumerate(((0, half), (half, 3 * n))):
        if a == b:
            continue
        prims.append({"positions": pos[a:b], "normals": np.tile(np.float32([0, 0, 1]), (b - a, 1)), "texcoords": None,
                      "tangents": None, "indices": np.arange(b - a, dtype=np.uint32), "material": len(mats)})
        mats.append({"base_color": (0.8, 0.5, 0.3, 1.0), "metallic": 0.0, "roughness": 0.5,
                     "emissive": (0.2 * k, 0.1, 0.0), "is_translucent": int(glass and k == 0), "transmission": 0.6})
    scene = sr.SceneData(prims, [(0, len(prims))], [(np.eye(4, dtype=np.float32), 0)], mats, [], name=f"gi_{n}")
    assert np.array_equal(_gi(sr, scene, env, grid, 0), _gi(sr, scene, env, grid, -1))


# (depth of vertex 0, of the other two, pixel): a covered sample of the
# triangle at which the interpolated 1/w is exactly zero
@pytest.mark.parametrize("w0,w1,px,py", [(21.636152, 67.772125, 4963, 1629), (15.870249, 80.99527, 5004, 1632),
                                         (5.1477737, 84.73842, 4949, 1749)])
def test_zero_denominator_sample(sr, orc, scenes, w0, w1, px, py):
    """A triangle whose integer edge constants wrap covers samples far outside
    itself, one of them where the interpolated 1/w is zero: w and the depth
    are infinite there, as IEEE division gives them, and the pixel is the
    triangle's, in the raster and in the shading."""
    from util import attach_dummy, screen_triangle_scene
    W, H = 5120, 2880
    tri = np.array([[[81888, 28748], [81888, 24724], [65594, 46048]]])
    scene, spec = screen_triangle_scene(sr, tri, np.float32([[w0, w1, w1]]), W, H)
    attach_dummy(sr, scene)
    cam = scenes.make_camera(spec)
    o = orc.OracleRenderer(W, H)
    o.render_scene(orc.OracleScene(scene), cam, threads=16)
    want = o.read_frame()
    assert want["ids"][py, px] == 0 and np.isinf(want["depth"][py, px])
    r = sr.Renderer(W, H)
    r.render_scene(sr.Scene(scene), cam)
    ids, depth = r.read_vbuffer()
    rgb = r.read_color()
    r.close()
    assert np.array_equal(ids, want["ids"]), (ids[py, px], int((ids != want["ids"]).sum()))
    assert np.array_equal(depth.view(np.uint32), want["depth"].view(np.uint32))
    assert np.array_equal(rgb, want["rgb"], equal_nan=True)


def test_short_divisions_and_roots_are_ieee(sr):
    """The reciprocal and 1 / sqrt in their short forms for every float in
    [2^-96, 2^96], the quotient for 4e9 random pairs with exponents within
    +-40: all equal IEEE division and square root bit for bit."""
    bad = (sr.C.c_uint64 * 3)()
    sr.check(sr.lib().sr_check_short_forms(0, 20240229, 4 * 10 ** 9, bad))
    assert list(bad) == [0, 0, 0]


# heights of the floor over the grid's corner, down to where the quotient by
# the voxel's size is denormal
@pytest.mark.parametrize("y", [1e-30, 3e-34, 1.3e-36, 2e-38])
def test_voxel_lookup_tiny_offsets(sr, orc, scenes, y):
    """A floor a hair above the voxel grid's corner, dark below and lit above:
    the light is the height over the voxel's size, in sizes that are no power
    of two, and it is the oracle's to the bit however small."""
    from util import dark_environment
    W, H = 96, 64
    rng = np.random.default_rng(5)
    n = 40
    p = np.zeros((n * n, 3), np.float32)
    g = np.linspace(-2, 2, n)
    p[:, 0], p[:, 2] = np.tile(g, n), np.repeat(g, n)
    p[:, 1] = (y * rng.uniform(0.2, 1.0, n * n)).astype(np.float32)
    i = (np.arange(n - 1)[:, None] * n + np.arange(n - 1)).reshape(-1, 1)
    idx = np.concatenate([i, i + n, i + 1, i + 1, i + n, i + n + 1], 1).reshape(-1).astype(np.uint32)
    prim = {"positions": p, "normals": np.tile(np.float32([0, 1, 0]), (n * n, 1)), "texcoords": None, "tangents": None,
            "indices": idx, "material": 0}
    mat = {"base_color": (1.0, 1.0, 1.0, 1.0), "metallic": 0.0, "roughness": 0.5}
    scene = sr.SceneData([prim], [(0, 1)], [(np.eye(4, dtype=np.float32), 0)], [mat], [], name="floor")
    light = np.repeat(np.float32([0.0, 1.0]), 2)[None].repeat(2, 0).reshape(-1)      # [z][y][x]: by y
    scene.attach(dark_environment(sr), sr.VoxelGrid((2, 2, 2), np.float32([-3, 0, -3]), np.float32([3, 3.4567, 3]), light))
    cam = scenes.make_camera(scenes.camera_spec((0, 1.5, 3), 0.0, 0.5, np.pi / 3, W, H, 50.0))
    o = orc.OracleRenderer(W, H)
    o.render_scene(orc.OracleScene(scene), cam)
    want = np.ascontiguousarray(o.read_frame()["rgb"], np.float32)
    r = sr.Renderer(W, H)
    r.render_scene(sr.Scene(scene), cam)
    ids, rgb = r.read_vbuffer()[0], r.read_color()
    r.close()
    lit = rgb[ids != sr.NO_ID]
    assert len(lit) > 1000 and 0 < lit.max() < 10 * y
    assert np.array_equal(rgb.view(np.uint32), want.view(np.uint32)), int((rgb != want).any(-1).sum())
