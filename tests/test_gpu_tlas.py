"""The TLAS walk of the rendering kernels, which tests both children of a node
when the node is popped and a popped node only where a direction component is
zero or not finite, against the counting variant, which tests every node it
pops as the reference does (and whose hits and counts the trace tests compare
with the oracle): the same bits, on many instances and on TLAS forms that the
builder does not make (leaves of several instances, an instance in two leaves,
a root that is such a leaf)."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _sums(r, upload, cam, spp):
    out = []
    for work in (False, True):
        upload()
        r.set_profiling(work=work)
        r.reset()
        r.render(cam, 3, spp, want_image=False)
        st = r.stats()
        out.append((r.read_accum()[0].view(np.uint32).copy(), st["closest_rays"], st["shadow_rays"]))
    return out


@pytest.mark.parametrize("n_inst,w,h,spp", [(1, 40, 30, 8), (2, 40, 30, 8), (63, 64, 48, 8), (64, 65, 47, 8),
                                            (700, 97, 61, 16), (4096, 160, 90, 8)])
def test_render_equals_counting_variant(n_inst, w, h, spp):
    from xenon_amd import HipRenderer, HipScene, scenes
    hs = HipScene(scenes.instancing(width=w, height=h, n_inst=n_inst, tri_range=(500, 3000), n_emit=8))
    print(f"[tlas] {n_inst} instances {w}x{h}", flush=True)
    with HipRenderer(w, h, 8, 3) as r:
        a, b = _sums(r, lambda: r.upload_scene(hs), hs.camera(w, h), spp)
    assert np.array_equal(a[0], b[0]) and a[1:] == b[1:]
    assert np.any(a[0] != 0)


def _forms(nodes, order, N):
    """(name, nodes, order) of other TLAS forms over the same leaves."""
    n = len(order)
    lo = np.min([x.lo[:] for x in nodes], 0)
    hi = np.max([x.hi[:] for x in nodes], 0)

    def node(child, count, a=lo, b=hi):
        x = N.BvhNode()
        x.lo[:], x.hi[:] = [float(v) for v in a], [float(v) for v in b]
        x.child, x.count = child, count
        return x

    flat = list(range(n))
    yield "root list", [node(0, n)], flat
    yield "two lists", [node(1, 0), node(0, n // 2), node(n // 2, n - n // 2)], flat
    yield "list and one", [node(1, 0), node(0, n - 1), node(n - 1, 1)], flat
    # an instance in two leaves (the order array names it twice, another not at all)
    twice = list(flat)
    twice[0] = twice[-1]
    yield "named twice", [node(1, 0), node(0, 1), node(1, n - 1)], twice


def test_other_tlas_forms():
    from xenon_amd import HipRenderer, HipScene, native as N, scenes
    hs = HipScene(scenes.instancing(width=48, height=36, n_inst=9, tri_range=(500, 1500), n_emit=4, box=12.0))
    src = hs.flat
    nodes = [src.tlas_nodes[k] for k in range(src.num_tlas_nodes)]
    order = [src.tlas_inst_indices[k] for k in range(src.num_instances)]
    cam = hs.camera(48, 36)
    with HipRenderer(48, 36, 6, 2) as r:
        for name, ns, od in _forms(nodes, order, N):
            arr = (N.BvhNode * len(ns))(*ns)
            o = np.array(od, np.uint32)
            flat = N.FlatScene()
            C.memmove(C.byref(flat), C.byref(src), C.sizeof(N.FlatScene))
            flat.num_tlas_nodes = len(ns)
            flat.tlas_nodes = C.cast(arr, type(src.tlas_nodes))
            flat.tlas_inst_indices = o.ctypes.data_as(C.POINTER(C.c_uint32))
            print(f"[tlas] {name}", flush=True)
            a, b = _sums(r, lambda: r._chk(N.lib().xnh_upload_scene(r.h, C.byref(flat))), cam, 8)
            assert np.array_equal(a[0], b[0]) and a[1:] == b[1:], name
            assert np.any(a[0] != 0), name
