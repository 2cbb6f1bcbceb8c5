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
