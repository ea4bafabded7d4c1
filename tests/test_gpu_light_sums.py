"""Per-slot light sums that are kept only for the lights a job has: scenes with
area lights, with suns, with both and with neither, jobs of odd sizes (sums
that begin off a 16-byte boundary) and of no bounces, in one batch and after
renders that left other values in the slots. Every job has, bit for bit, the
sums that it has alone in a new context."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _scenes():
    from xenon_amd import scenes
    area, sun, both = scenes.cornell(8, 8), scenes.big_mesh(level=2), scenes.prim_shapes()
    none = scenes.big_mesh(level=2)
    none.suns = []
    return [area, sun, both, none]


def _sums(r, gs, hs, order, sizes):
    jobs = [dict(scene=gs[k], camera=hs[k].camera(w, h), width=w, height=h, spp_first=1 + n, spp_count=n,
                 max_bounces=b, min_bounces=2) for k, (w, h, n, b) in zip(order, sizes)]
    return [np.asarray(s).view(np.uint32).copy() for s in r.render_jobs(jobs, want_sums=True)[1]]


@pytest.mark.parametrize("order,sizes", [
    ((0, 1, 2, 3), ((9, 7, 3, 5), (13, 5, 2, 4), (7, 11, 3, 6), (5, 5, 1, 3))),
    ((1, 0), ((3, 1, 1, 4), (17, 3, 5, 0))),
    ((3, 2, 1, 0, 1), ((1, 1, 1, 4), (3, 3, 3, 0), (31, 9, 4, 8), (33, 2, 7, 8), (8, 8, 8, 2))),
])
def test_jobs_with_other_lights(order, sizes):
    from xenon_amd import GpuScene, HipRenderer, HipScene
    hs = [HipScene(d) for d in _scenes()]
    with HipRenderer(32, 32, 8, 3, spp_per_launch=3) as r:
        gs = [GpuScene(r, h) for h in hs]
        print(f"[lights] jobs {order}", flush=True)
        _sums(r, gs, hs, (2, 0, 1), ((40, 30, 3, 8), (30, 40, 3, 8), (20, 20, 2, 8)))   # leaves sums of every kind
        got = _sums(r, gs, hs, order, sizes)
        for g in gs:
            g.release()
    for k, (o, size) in enumerate(zip(order, sizes)):
        with HipRenderer(8, 8, 8, 3) as one:
            g = GpuScene(one, hs[o])
            alone = _sums(one, {o: g}, hs, (o,), (size,))[0]
            g.release()
        assert np.array_equal(got[k], alone), k
        assert size[3] == 0 or o != 0 or np.any(got[k])
