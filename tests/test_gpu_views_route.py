"""The multi-view passes A and C take the route that is faster: many small views, views over small trees
and views without rays as one persistent launch, larger ones queued view after view. The sizes lie on
both sides of the rule; each result is the inline schedule's, bit for bit."""
import pytest

import test_gpu_views_queued
from restir_amd import abi, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scene,sizes,rays,queued_a,queued_c", [
    ("terrain", [(48, 27)] * 12, True, False, False),
    ("terrain", [(33, 21)], True, True, True),
    ("terrain", [(213, 121)] * 3, True, False, True),
    ("terrain", [(961, 541), (960, 540)], True, True, True),
    ("room", [(213, 121)], True, True, True),
    ("room", [(213, 121)] * 4, True, False, False),
    ("room", [(1280, 720)], True, False, False),
    ("terrain", [(320, 180)], False, True, True),
    ("terrain", [(320, 180)] * 2, False, False, False),
])
def test_the_faster_route_is_taken(monkeypatch, scene, sizes, rays, queued_a, queued_c):
    import torch
    sc = scenes.cornell_box(1) if scene == "room" else scenes.terrain(11, grid=48, n_boxes=60, n_point_lights=2000,
                                                                      extent=16.0)
    monkeypatch.setattr(test_gpu_views_queued, "_views", lambda sizes: [(sc, w, h) for w, h in sizes])
    p = test_gpu_views_queued._Passes(torch, sizes)
    for u in p.us:
        u.flags = abi.VISIBILITY_REUSE_FLAG if rays else 0
    p.run(abi.Launch(0, 0, abi.SCHEDULE_INLINE))
    ref = p.out(torch)
    for buf in p.bufs:
        for t in buf:
            t.zero_()
    ctx = p.b.ctx
    ctx.profile_read()
    ctx.profile_enable(True)
    p.run()
    rows = ctx.profile_read()
    ctx.profile_enable(False)
    assert all(torch.equal(a, b) for a, b in zip(p.out(torch), ref))
    assert ("k_pass_a_finish" in rows, "k_pass_c_merge" in rows) == (queued_a, queued_c)
