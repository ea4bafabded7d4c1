"""NoiseStats where its launches change shape: images without interior, one
pixel short of, at and past a work-group and the largest number of
work-groups, and keys that all fall on one or two values. Exact as
test_gpu_image.py has it: the counts, the selected ranks and the maximum are
the oracle's bits; what comes from the double sums is held to 1 ulp."""
import numpy as np
import pytest

from test_gpu_image import _same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["noise", "flat", "two"])
@pytest.mark.parametrize("w,h", [(1, 1), (2, 9), (3, 3), (3, 85), (16, 16), (257, 1), (257, 3), (129, 33),
                                 (1023, 256), (512, 512), (2049, 128), (1031, 521)])
def test_noise_stats_edges(oracle, w, h, kind):
    from xenon_amd import HipRenderer
    rng = np.random.default_rng(w * 4099 + h)
    img = rng.uniform(0.0, 2.0, (h, w, 3)).astype(np.float32)
    if kind == "flat":
        img[:] = 0.25
    elif kind == "two":
        img = (rng.random((h, w, 1)) < 0.01).astype(np.float32) * np.ones(3, np.float32)
    print(f"[image] {kind} {w}x{h}", flush=True)
    with HipRenderer(8, 8) as r:
        _same(r.noise_stats(img), oracle.noise_stats(img, w, h), (kind, w, h))
        _same(r.noise_stats(img), oracle.noise_stats(img, w, h), (kind, w, h, "again"))
