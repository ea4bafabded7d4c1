"""Calls that share a context's scratch and pinned memory: ray batches longer
than one pass of their grid, calls of different sizes and kinds in turn, and
frames averaged and flipped on the device. Every result is what the same work
gives in small pieces or in a context of its own, bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _rays(n, seed):
    rng = np.random.default_rng(seed)
    r = np.empty((n, 8), np.float32)
    r[:, 0:3] = rng.uniform(-0.9, 0.9, (n, 3)) + [0.0, 1.0, 0.0]
    d = rng.normal(size=(n, 3))
    r[:, 3:6] = d / np.linalg.norm(d, axis=1, keepdims=True)
    r[:, 6] = 1e-3
    r[:, 7] = 1e30
    return r


@pytest.fixture(scope="module")
def scene():
    from xenon_amd import HipScene, scenes
    desc = scenes.cornell(33, 17, spp=2)
    return HipScene(desc), desc


def _renderer(scene):
    from xenon_amd import HipRenderer
    hs, desc = scene
    r = HipRenderer(desc.width, desc.height, desc.max_bounces, desc.min_bounces)
    r.upload_scene(hs)
    return r


@pytest.mark.parametrize("n", [1, 255, 257, 262145, 700001])
def test_ray_batches_in_pieces(scene, n):
    rays = _rays(n, n)
    with _renderer(scene) as r:
        print(f"[scratch] {n} rays", flush=True)
        hits, occ = r.trace_closest(rays), r.trace_any(rays)
        piece = 50000
        for a in range(0, n, piece):
            assert hits[a:a + piece].tobytes() == r.trace_closest(rays[a:a + piece]).tobytes()
            assert occ[a:a + piece].tobytes() == r.trace_any(rays[a:a + piece]).tobytes()


def test_mixed_calls_share_scratch(scene):
    rng = np.random.default_rng(4)
    meshes = []
    for t in (1, 7, 3000):
        v = rng.random((3 * t, 3)).astype(np.float32)
        meshes.append((v, np.arange(3 * t, dtype=np.int32).reshape(t, 3)))
    rays = _rays(4001, 9)

    def work(r, k):
        out = []
        for n in (4001, 3, 900):
            out.append(r.trace_closest(rays[:n]).tobytes())
            nodes, prims = r.build_blas(*meshes[(k + n) % 3])[:2]
            out.append(nodes.tobytes() + prims.tobytes())
        return out

    want = []
    for k in range(3):
        with _renderer(scene) as r:
            want.append(work(r, k))
    with _renderer(scene) as r:
        for k in (0, 1, 2, 0):
            print(f"[scratch] mixed calls {k}", flush=True)
            assert work(r, k) == want[k]


def test_frame_is_the_average_flipped(scene):
    hs, desc = scene
    with _renderer(scene) as r, _renderer(scene) as q:
        for k in range(1, 4):
            frame = r.render_frame(hs.camera())
            avg = q.render(hs.camera(), k, 1)
            assert frame.tobytes() == np.ascontiguousarray(
                np.asarray(avg).reshape(desc.height, desc.width, 3)[::-1]).tobytes(), k
