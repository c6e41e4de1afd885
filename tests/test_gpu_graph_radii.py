"""Tunnel radii of a captured batch (ckd_graph_update): a graph captured with a
largest radius above 32 takes any later one, whose window may be far wider than
the captured; up to 32 the captured radius is the limit.  Replays bit for bit
against the oracle."""
import numpy as np
import pytest

from cookiedough_amd import workloads as wl
from cookiedough_amd._lib import CKD_EINVAL, CKD_FX_TUNNEL, CKD_SHADE_FP32
from oracles import P

pytestmark = pytest.mark.gpu
SHAPES = [(300, 261), (264, 256)]


class Batch:
    def __init__(self, ctx):
        self.ctx, self.total = ctx, sum(w * h for w, h in SHAPES)
        self.tex = wl.noise_texture(0, 9)
        self.grids = [wl.tunnel_grid(w, h, 2.0 + w) for w, h in SHAPES]
        self.held = [ctx.upload(g) for g in self.grids]
        self.d_tex = ctx.upload(self.tex)
        self.out, self.tmp = ctx.empty(self.total), ctx.empty(self.total)

    def requests(self, radii):
        at, reqs = 0, []
        for (w, h), g, r in zip(SHAPES, self.held, radii):
            reqs.append(wl.make_request(wl.BatchItem(CKD_FX_TUNNEL, w, h, 0.0, r), self.out.ptr + 4 * at, None, None,
                                        g.ptr))
            at += w * h
        return self.ctx.request_array(reqs)

    def want(self, orc, radii):
        frames = []
        for (w, h), g, r in zip(SHAPES, self.grids, radii):
            ref, o0, o1 = (np.zeros(w * h, np.uint32) for _ in range(3))
            orc.orc_tunnel_frame(P(ref), P(o0), P(o1), w, h, P(g), P(self.tex), 9, r, 8)
            frames.append(ref)
        return np.concatenate(frames)


@pytest.mark.parametrize("seg", [8, 32, 64])
@pytest.mark.parametrize("captured,updates", [
    ((40, 3), [(60, 60), (111, 112), (127, 127), (33, 1), (5, 32)]),
    ((33, 33), [(127, 34), (8, 8)]),
    ((1, 111), [(112, 127), (95, 96)]),
    ((127, 2), [(126, 127), (2, 2)]),
    ((32, 7), [(7, 32), (1, 1)])])
def test_radii_after_capture(ctx, orc, captured, updates, seg):
    saved, t = ctx.get_tuning(), ctx.get_tuning()
    t.tunnelVSeg = seg
    ctx.set_tuning(t)
    try:
        b = Batch(ctx)
        graph = ctx.batch_graph(b.requests(captured), None, CKD_SHADE_FP32, b.d_tex, 9, b.tmp, b.total)
    finally:
        ctx.set_tuning(saved)
    try:
        for radii in [captured] + updates:
            print("graph radii", captured, "->", radii, "segment", seg, flush=True)
            graph.update(b.requests(radii))
            ctx.memset32(b.out, 0x12345678, b.total)
            graph.launch()
            ctx.sync()
            assert np.array_equal(b.out.numpy(), b.want(orc, radii)), radii
        if max(captured) <= 32:
            arr = b.requests((max(captured) + 1, 1))
            assert ctx.lib.ckd_graph_update(graph.h, arr, len(arr)) == CKD_EINVAL
    finally:
        graph.close()
