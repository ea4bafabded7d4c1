"""The plain form of the TLAS box test (hardware min and max, for 16 and more
nodes with ordered finite boxes) against the counting variant, which orders the
planes by the direction's signs for every box: the same bits just below, at and
above the rule's node count, and with a box that is turned over or infinite,
which takes the general form."""
import ctypes as C

import numpy as np
import pytest

from test_gpu_tlas import _sums

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_inst,spoil", [(7, None), (8, None), (9, None), (40, None), (40, "turned"), (40, "infinite"),
                                          (40, "nan")])
def test_plain_boxes_equal_signed_ones(n_inst, spoil):
    from xenon_amd import HipRenderer, HipScene, native as N, scenes
    hs = HipScene(scenes.instancing(width=56, height=40, n_inst=n_inst, tri_range=(500, 1500), n_emit=4, box=10.0))
    flat = N.FlatScene()
    C.memmove(C.byref(flat), C.byref(hs.flat), C.sizeof(N.FlatScene))
    nodes = (N.BvhNode * flat.num_tlas_nodes)()
    C.memmove(nodes, hs.flat.tlas_nodes, C.sizeof(nodes))
    flat.tlas_nodes = C.cast(nodes, type(hs.flat.tlas_nodes))
    leaf = next(x for x in nodes if x.count > 0)
    if spoil == "turned":
        leaf.lo[1], leaf.hi[1] = leaf.hi[1], leaf.lo[1]
    elif spoil == "infinite":
        leaf.hi[0] = float("inf")
    elif spoil == "nan":
        leaf.lo[2] = float("nan")
    print(f"[tlas] {n_inst} instances, {flat.num_tlas_nodes} nodes, {spoil}", flush=True)
    with HipRenderer(56, 40, 6, 2) as r:
        a, b = _sums(r, lambda: r._chk(N.lib().xnh_upload_scene(r.h, C.byref(flat))), hs.camera(56, 40), 8)
    assert np.array_equal(a[0], b[0]) and a[1:] == b[1:]
    assert np.any(a[0] != 0)
