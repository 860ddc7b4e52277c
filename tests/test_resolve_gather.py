"""The resolve's gathered shading (hvvr_amd/csrc/gpu/resolve.hip): samples with as many
triangles as subsamples, with one, with none, and mixed in a wave, against the oracle's
colours (within 1/255). Triangles from smaller than a subsample's spacing up to the whole
view."""

import numpy as np
import pytest

from conftest import rgba_delta

pytestmark = pytest.mark.gpu


def _scene(H, n, size):
    rng = np.random.default_rng(n)
    v = np.zeros(3 * n, H.DTYPES["vertex"])
    centre = rng.uniform([-1.4, -1.4, -6], [1.4, 1.4, -4], (n, 1, 3))
    v["pos"] = (centre + rng.uniform(-size, size, (n, 3, 3))).reshape(-1, 3)
    v["normal"][:, 2] = np.float16(1).view(np.uint16)
    m = np.zeros(4, H.DTYPES["material"])
    m["diffuse"] = [(0.9, 0.1, 0.1, 1), (0.1, 0.8, 0.2, 1), (0.2, 0.3, 0.9, 1), (0.7, 0.7, 0.1, 1)]
    m["specular"] = (0.04, 0.04, 0.04, 1)
    m["glossiness"] = 0.4
    m["textureIDsAndShadingModel"] = 1 | (0xFFFF << 16) | (0xFFFF << 32) | (0xFFFF << 48)
    tri = np.arange(3 * n, dtype=np.uint32).reshape(n, 3)
    return H.HostScene.from_meshes([(v, tri, (np.arange(n) % 4).astype(np.uint32), None)], m)


@pytest.mark.parametrize("n,size", [(1, 8.0), (40, 0.05), (3000, 0.02), (3000, 0.3)])
@pytest.mark.parametrize("A,half", [(1, False), (2, False), (4, False), (4, True), (8, False), (8, True), (16, False)])
def test_gathered_shading(H, O, ctx, n, size, A, half):
    scene = _scene(H, n, size)
    t = 0.35
    view = H.HostView.from_samples(H.grid_samples(40, 40), 40, 40, (-t, -t, t, t))
    m = np.eye(4, dtype=np.float32).reshape(16)
    ref = O.render_view(scene, view, A, camera_to_world=m)
    gs, gv = H.GpuScene(ctx, scene), H.GpuView(ctx, view, A)
    if half:
        gv.set_shading_precision(16)
    gv.render(gs, m)
    assert rgba_delta(gv.read_sample_colors(), ref["colors"]).max() <= (2 if half else 1)
    gv.close()
    gs.close()
