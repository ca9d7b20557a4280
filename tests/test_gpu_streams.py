"""Calls on one context from several streams and threads.  The context's
scratch is shared: a call's kernels must run after the previous call's, on
whatever stream that was, also when buffers grow in between and when a call is
refused after it has enqueued kernels; and values the kernels publish to the
host belong to their own call.  Every plane equals its render alone.  Bin starts
and the order of the tiles are checked by planes at the edges of their kernels."""
import threading

import numpy as np
import pytest

from film_grain_amd import capi, synth
from tests import fgcases

pytestmark = pytest.mark.gpu


def _jobs(oracle):
    import torch
    specs = [("pixel", 96, 64, 0.1, 0.0, 1.0, 32), ("grain", 120, 90, 0.1, 0.04, 1.0, 64),
             ("pixel", 200, 150, 0.12, 0.05, 2.0, 100), ("pixel", 33, 21, 0.3, 0.0, 1.0, 16),
             ("grain", 64, 64, 0.06, 0.0, 2.0, 128), ("pixel", 260, 240, 0.08, 0.0, 1.0, 64)]
    jobs = []
    for i, (algo, w, h, r, sd, z, n) in enumerate(specs):
        c = fgcases.build_case(oracle, f"s{i}", synth.sinusoid_field(w, h, i, n_waves=3), r, sd,
                               "lognorm" if sd else "const", zoom=z, n_samples=n, seed=100 + i)
        offs = c.offsets_input if algo == "pixel" else c.offsets
        jobs.append((algo, c.desc, torch.from_numpy(c.lam).to("cuda:0"),
                     torch.from_numpy(np.ascontiguousarray(offs)).to("cuda:0")))
    return jobs


def _alone(jobs):
    import torch
    want = []
    for algo, desc, lam, offs in jobs:
        ctx = capi.Context(0)
        out = torch.empty((desc.out_h, desc.out_w), device="cuda:0")
        ctx.render_device(algo, desc, lam, offs, out)
        ctx.stream_status()
        want.append(out.cpu().numpy())
        ctx.close()
    return want


def test_streams_in_turn(oracle):
    import torch
    jobs = _jobs(oracle)
    want = _alone(jobs)
    ctx = capi.Context(0)
    streams = [torch.cuda.Stream() for _ in range(3)]
    outs = []
    torch.cuda.synchronize()
    for rep in range(4):
        for j, (algo, desc, lam, offs) in enumerate(jobs):
            s = streams[(j + rep) % 3]
            out = torch.empty((desc.out_h, desc.out_w), device="cuda:0")
            s.wait_stream(torch.cuda.current_stream())
            ctx.render_device(algo, desc, lam, offs, out, stream=s)
            outs.append((j, out))
    torch.cuda.synchronize()
    ctx.stream_status()
    for j, out in outs:
        assert np.array_equal(out.cpu().numpy(), want[j]), j
    ctx.close()


def test_threads_share_a_context(oracle):
    import torch
    jobs = _jobs(oracle)
    want = _alone(jobs)
    ctx = capi.Context(0)
    torch.cuda.synchronize()
    bad = []

    def work(t):
        s = torch.cuda.Stream()
        for rep in range(3):
            for j in range(t, len(jobs), 2):
                algo, desc, lam, offs = jobs[j]
                with torch.cuda.stream(s):
                    out = torch.empty((desc.out_h, desc.out_w), device="cuda:0")
                    ctx.render_device(algo, desc, lam, offs, out, stream=s)
                    s.synchronize()
                    if not np.array_equal(out.cpu().numpy(), want[j]):
                        bad.append(j)
    threads = [threading.Thread(target=work, args=(t,)) for t in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert bad == []
    ctx.stream_status()
    ctx.close()


def test_call_after_a_refused_one(oracle):
    """A plane of more grains than one render addresses is refused after its
    count has run; the next calls, on another stream, are unaffected."""
    import torch
    jobs = _jobs(oracle)
    want = _alone(jobs)
    ctx = capi.Context(0)
    lam = np.full((8, 8), 1.0e6, dtype=np.float32)
    d = oracle.derive(0.05, 0.0, "const", 1.0, 0.8, 4, cell_delta=64.0, seed=3, in_w=8, in_h=8)
    desc = capi.make_desc(d.in_w, d.in_h, d.out_w, d.out_h, 4, 0, 3, 1.0, d.delta, d.rm, 0.05, d.log_mu, d.log_sigma)
    offs = torch.from_numpy(oracle.make_offsets(3, 4, 0.8)).to("cuda:0")
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    for j in (2, 5):
        with pytest.raises(capi.FilmGrainError) as err:
            ctx.render_device("pixel", desc, torch.from_numpy(lam).to("cuda:0"), offs,
                              torch.empty((d.out_h, d.out_w), device="cuda:0"), stream=a)
        assert err.value.code == capi.FG_ECAPACITY
        algo, jd, jl, jo = jobs[j]
        out = torch.empty((jd.out_h, jd.out_w), device="cuda:0")
        ctx.render_device(algo, jd, jl, jo, out, stream=b)
        torch.cuda.synchronize()
        assert np.array_equal(out.cpu().numpy(), want[j])
    ctx.close()


@pytest.mark.parametrize("w,h,radius,grey", [
    (96, 96, 0.1, None),       # below 4096 bins: the scan's first round
    (104, 104, 0.1, None),     # just above
    (200, 200, 0.1, None),     # either side of 16384 bins: one workgroup, three launches
    (212, 212, 0.1, None),
    (64, 48, 0.1, 0.0),        # no grain at all
    (2200, 2000, 1.0, 0.02),   # 8625 tiles and more: ordered by the radix sort
    (3000, 2900, 1.0, 0.02),
])
def test_bin_starts_and_tile_order(oracle, w, h, radius, grey):
    plane = (np.full((h, w), grey, dtype=np.float32) if grey is not None
             else synth.sinusoid_field(w, h, w, n_waves=3))
    c = fgcases.build_case(oracle, "scan", plane, radius, 0.0, "const", zoom=1.0, n_samples=4, seed=w)
    want = oracle.render_pixelwise(c.plane, c.lam, c.offsets_input)
    ctx = capi.Context(0)
    got = ctx.render_host("pixel", c.desc, c.lam, c.offsets_input)
    ctx.close()
    assert np.array_equal(got, want)


@pytest.mark.parametrize("tiles,w,h", [
    (2048, 1024, 1024),  # the most that one launch weighs and orders
    (2080, 1024, 1033),  # weights in their own launch, then the counting sort
    (8192, 2048, 2048),  # the most that it orders
    (8256, 2048, 2049),  # ordered by the radix sort
])
@pytest.mark.parametrize("algo", ["pixel", "grain"])
def test_tile_order(oracle, algo, tiles, w, h):
    """Planes at the limits of the tile orders: every tile is in the order."""
    c = fgcases.build_case(oracle, "order", np.full((h, w), 0.02, dtype=np.float32), 1.0, 0.0, "const", zoom=1.0,
                           n_samples=4, seed=w + h)
    ctx = capi.Context(0)
    ctx.set_launch_config(pix_tile_w=32, pix_tile_h=16, grain_tile_w=32, grain_tile_h=16)
    cfg = ctx.launch_config(c.desc, algo)
    tw, th = (cfg[f"{'pix' if algo == 'pixel' else 'grain'}_tile_{s}"] for s in "wh")
    assert -(-w // tw) * -(-h // th) == tiles
    offs = c.offsets_input if algo == "pixel" else c.offsets
    got = ctx.render_host(algo, c.desc, c.lam, offs)
    ctx.close()
    render = oracle.render_pixelwise if algo == "pixel" else oracle.render_grainwise
    assert np.array_equal(got, render(c.plane, c.lam, offs))


def test_captured_grainwise_render(oracle):
    """A grain-wise render recorded into the caller's graph (after eager renders
    of every plane here, so that the scratch grows no more): every replay, with
    eager renders between, and the eager calls after it equal the plane alone."""
    import torch
    jobs = _jobs(oracle)
    want = _alone(jobs)
    ctx = capi.Context(0)
    for algo, desc, lam, offs in jobs:
        ctx.render_device(algo, desc, lam, offs, torch.empty((desc.out_h, desc.out_w), device="cuda:0"))
    torch.cuda.synchronize()
    for j in (1, 4):
        algo, desc, lam, offs = jobs[j]
        out = torch.zeros((desc.out_h, desc.out_w), device="cuda:0")
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            ctx.render_device(algo, desc, lam, offs, out, stream=torch.cuda.current_stream())
        for k in (j, 0, 2):
            graph.replay()
            torch.cuda.synchronize()
            assert np.array_equal(out.cpu().numpy(), want[j]), (j, k)
            out.zero_()
            a, d, l, o = jobs[k]
            eager = torch.empty((d.out_h, d.out_w), device="cuda:0")
            ctx.render_device(a, d, l, o, eager)
            torch.cuda.synchronize()
            assert np.array_equal(eager.cpu().numpy(), want[k]), (j, k)
        del graph
    ctx.stream_status()
    ctx.close()


def test_graph_outlives_the_buffers_it_recorded(oracle):
    """Grain-wise renders recorded while the context's buffers are small: later
    calls outgrow every one of them, and the graphs, whose kernels still work in
    the old ones, give their planes."""
    import torch
    jobs = _jobs(oracle)
    want = _alone(jobs)
    ctx = capi.Context(0)
    recorded = []
    for j in (1, 4):
        algo, desc, lam, offs = jobs[j]
        out = torch.zeros((desc.out_h, desc.out_w), device="cuda:0")
        ctx.render_device(algo, desc, lam, offs, out)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            ctx.render_device(algo, desc, lam, offs, out, stream=torch.cuda.current_stream())
        recorded.append((j, graph, out))
    for size, n in ((300, 256), (700, 700)):
        # more samples, pixels, tiles and classes than any plane before
        c = fgcases.build_case(oracle, "large", synth.sinusoid_field(size, size - 40, size, n_waves=3), 0.25, 0.1,
                               "lognorm", zoom=2.0, n_samples=n, seed=size)
        lam, offs = torch.from_numpy(c.lam).to("cuda:0"), torch.from_numpy(c.offsets).to("cuda:0")
        large = torch.empty((c.desc.out_h, c.desc.out_w), device="cuda:0")
        ctx.render_device("grain", c.desc, lam, offs, large)
        torch.cuda.synchronize()
        before = large.clone()
        for j, graph, out in recorded:
            out.zero_()
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            assert np.array_equal(out.cpu().numpy(), want[j]), (size, j)
        ctx.render_device("grain", c.desc, lam, offs, large)
        torch.cuda.synchronize()
        assert torch.equal(large, before)
    del recorded
    ctx.stream_status()
    ctx.close()


def test_captured_pixelwise_render_is_refused(oracle):
    """A pixel-wise render waits for its grain total: while its stream captures
    it is refused before it enqueues anything, and the capture goes on."""
    import torch
    jobs = _jobs(oracle)
    want = _alone(jobs)
    ctx = capi.Context(0)
    algo, desc, lam, offs = jobs[0]
    out = torch.zeros((desc.out_h, desc.out_w), device="cuda:0")
    ctx.render_device(algo, desc, lam, offs, out)
    torch.cuda.synchronize()
    x = torch.zeros(8, device="cuda:0")
    graph = torch.cuda.CUDAGraph()
    refused = []
    with torch.cuda.graph(graph):
        s = torch.cuda.current_stream()
        for call in (lambda: ctx.render_device(algo, desc, lam, offs, out, stream=s),
                     lambda: ctx.render_planes_device(desc, [lam, lam], offs, [out, out], stream=s),
                     lambda: ctx.render_device_noalloc(desc, lam, offs, out, stream=s)):
            try:
                call()
            except capi.FilmGrainError as err:
                refused.append(err.code)
        x += 1
    assert refused == [capi.FG_EHIP] * 3
    out.zero_()
    for k in (1, 2):
        graph.replay()
        torch.cuda.synchronize()
        assert torch.all(x == k) and torch.all(out == 0)
    for j in (0, 1):
        a, d, l, o = jobs[j]
        out = torch.zeros((d.out_h, d.out_w), device="cuda:0")
        ctx.render_device(a, d, l, o, out)
        torch.cuda.synchronize()
        assert np.array_equal(out.cpu().numpy(), want[j])
    ctx.close()
