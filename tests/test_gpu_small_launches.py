"""Renders at the sizes where the launches hand out their work differently:
fewer 64-entry units than the grid has waves (parts of units, smaller shading
windows), one more than that, ragged last units, and several jobs in one
batch. A sample's path is a function of its pixel, sample index and scene, so
the same samples rendered in other batches, sizes of batch and orders give
the same bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _bits(a):
    return np.ascontiguousarray(a).view(np.uint32)


@pytest.fixture(scope="module")
def built():
    from xenon_amd import HipScene, scenes
    return {"cornell": HipScene(scenes.cornell(64, 64)),
            "mesh": HipScene(scenes.big_mesh(width=64, height=36, level=4)),
            "instancing": HipScene(scenes.instancing(width=64, height=36, n_inst=80, tri_range=(500, 2000),
                                                     n_emit=8)),
            "prims": HipScene(scenes.prim_shapes(width=64, height=36))}


# paths per batch: one, a unit less one, a unit, a unit and one, parts of units at several splits, about the
# grid's waves in units, and above them
@pytest.mark.parametrize("name,w,h", [("cornell", 1, 1), ("cornell", 9, 7), ("mesh", 8, 8), ("instancing", 13, 5),
                                      ("prims", 97, 31), ("mesh", 160, 121), ("cornell", 331, 247),
                                      ("instancing", 333, 217), ("mesh", 577, 570), ("cornell", 700, 701)])
def test_batches_of_any_size_give_the_same_sums(built, name, w, h):
    from xenon_amd import HipRenderer
    scene = built[name]
    sums = []
    for spp_per_launch in (1, 3, 0):
        with HipRenderer(w, h, 6, 2, spp_per_launch=spp_per_launch) as r:
            r.upload_scene(scene)
            print(f"[small launches] {name} {w}x{h}, {spp_per_launch or 'default'} samples a batch", flush=True)
            r.render(scene.camera(w, h), 5, 7, want_image=False)
            st = r.stats()
            sums.append((r.read_accum()[0], st["closest_rays"], st["shadow_rays"], st["paths"]))
    for s in sums[1:]:
        assert np.array_equal(_bits(s[0]), _bits(sums[0][0]))
        assert s[1:] == sums[0][1:]
    assert sums[0][3] == w * h * 7


def test_ray_counts_equal_the_counting_variant(built):
    """Ray counts come from the queues' lengths; the counting variant counts
    the rays it walked."""
    from xenon_amd import HipRenderer
    for name, w, h in (("cornell", 33, 17), ("mesh", 130, 70)):
        scene = built[name]
        with HipRenderer(w, h, 6, 2) as r:
            r.upload_scene(scene)
            got = []
            for work in (False, True):
                r.set_profiling(work=work)
                r.reset()
                r.render(scene.camera(w, h), 1, 5, want_image=False)
                st = r.stats()
                got.append((st["closest_rays"], st["shadow_rays"], st["paths"], _bits(r.read_accum()[0]).sum()))
            assert got[0] == got[1]


def test_many_small_jobs_in_one_batch(built):
    """Seventy jobs (more than a batch's chunks) of every scene at odd sizes
    against each rendered alone."""
    from xenon_amd import GpuScene, HipRenderer
    rng = np.random.default_rng(3)
    with HipRenderer(128, 128, 6, 2, spp_per_launch=16) as r:
        gpu = {k: GpuScene(r, s) for k, s in built.items()}
        jobs = []
        for k in range(70):
            name = list(gpu)[k % 4]
            w, h = int(rng.integers(1, 90)), int(rng.integers(1, 90))
            jobs.append(dict(scene=gpu[name], camera=built[name].camera(w, h), width=w, height=h, spp_first=1 + k,
                             spp_count=int(rng.integers(1, 9)), max_bounces=int(rng.integers(1, 7)), min_bounces=2))
        print("[small launches] 70 jobs", flush=True)
        together = r.render_jobs(jobs)
        for k in range(0, 70, 7):
            alone = r.render_jobs([jobs[k]])[0]
            assert np.array_equal(_bits(alone), _bits(together[k])), k
        for g in gpu.values():
            g.release()
