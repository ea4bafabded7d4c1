"""Materials at the edges of the rule that skips a dielectric's reflection lobe
of weight 0: IOR 1 (skipped), next to 1 (a small weight) and 1.5, each smooth,
anisotropic, rougher than the rule takes and partly metal. Images against the
oracle, which evaluates every lobe. Skipped or not, the arithmetic is the
oracle's but for the last bit of a few transcendentals, so most pixel sums are
bit-identical, as in the other scenes."""
import dataclasses

import numpy as np
import pytest

from test_gpu_render import SAME_PIXELS_MIN, _render_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ior", [1.0, 1.001, 1.5])
@pytest.mark.parametrize("rough,aniso,metal", [(1.0, 0.0, 0.0), (0.04, 0.9, 0.0), (4.5, 0.0, 0.0), (0.5, 0.3, 0.4)])
def test_dielectrics_by_ior(oracle, ior, rough, aniso, metal):
    from xenon_amd import scenes
    desc = scenes.cornell(32, 24, spp=4)
    desc.materials = [dataclasses.replace(m, ior=ior, roughness=rough, anisotropy=aniso, metallic=metal)
                      for m in desc.materials]
    print(f"[lobe] ior {ior} roughness {rough} anisotropy {aniso} metal {metal}", flush=True)
    _, acc, ref, _, _ = _render_pair(oracle, desc, 4)
    acc, ref = np.asarray(acc).reshape(-1, 3), np.asarray(ref).reshape(-1, 3)
    same = np.all((acc == ref) | (np.isnan(acc) & np.isnan(ref)), axis=1)
    assert same.mean() >= SAME_PIXELS_MIN
