"""One scenario of test_gpu_memory.py in a process of its own: `gpu_memory_worker.py SHIM SCENARIO`."""
import ctypes as C
import os
import sys

shim = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)  # before libhrt.so, whose calls then find it
sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))

import numpy as np  # noqa: E402

import heavyrt_amd as H  # noqa: E402
from heavyrt_amd import workloads as W  # noqa: E402

MB = 1 << 20
for fn in (shim.shim_used, shim.shim_calls, shim.shim_refused):
    fn.restype = C.c_uint64
shim.shim_limit.argtypes = [C.c_size_t]
shim.shim_names.restype = C.c_char_p


def kernels():
    """Names launched since the last call."""
    n = shim.shim_names().decode().split()
    shim.shim_clear_names()
    return n


def limited(room):
    """From here on the device has `room` bytes more than are allocated."""
    shim.shim_limit(shim.shim_used() + room)


def unlimited():
    shim.shim_limit(C.c_size_t(-1).value)


def committed(ctx, v, f, layout=H.LAYOUT_BVH2):
    s = H.Scene(ctx)
    s.add_instance(s.add_triangles(v, f))
    s.commit(layout=layout)
    return s


def leave_idle(ctx):
    """Memory that the engine keeps for its next trees: more than 200 MB."""
    unlimited()
    v, f = W.soup(600_000, stream=W.STREAM_TEST)
    s = committed(ctx, v, f, H.LAYOUT_AUTO_FP16)
    before = shim.shim_used()
    s.close()
    assert before > 300 * MB and shim.shim_used() > 200 * MB, (before, shim.shim_used())


def refused(fn):
    try:
        fn()
    except H.HrtError as e:
        assert e.status == 3, e.status  # out of memory
        return True
    return False


def idle_memory():
    """What a call of the engine needs beside its trees, it takes from their idle memory."""
    ctx = H.Context(0)
    v, f = W.soup(100_000, stream=W.STREAM_TEST)
    rays = W.incoherent_rays(700_000, stream=W.STREAM_TEST)

    def batch():
        b = H.Batch(ctx, [v.shape[0]], [f.shape[0]], [1000])
        b.upload([(v, f, rays[:1000])])
        b.run()
        b.hits()
        b.close()

    def server():
        H.Server(ctx, 20 * MB).close()

    def trace(layout, any_hit=False):
        s = committed(ctx, v, f, layout)
        run = s.trace_any_host if any_hit else s.trace_nearest_host
        want = run(rays)  # (and the staging of the next call: that one needs stacks alone)

        def call():
            assert np.asarray(run(rays)).tobytes() == np.asarray(want).tobytes()
            s.close()
        return call

    calls = [("batch", lambda: batch), ("server", lambda: server)]
    calls += [(f"trace {lay}", lambda lay=lay: trace(lay)) for lay in (H.LAYOUT_BVH2, H.LAYOUT_BVH4)]
    calls += [("any", lambda: trace(H.LAYOUT_AUTO_FP16, True))]
    for name, make in calls:
        call = make()
        print("idle memory for", name, flush=True)
        leave_idle(ctx)
        limited(MB)
        n = shim.shim_refused()
        call()
        assert shim.shim_refused() > n, "the device was not full"
    unlimited()
    ctx.close()


def smaller_launches():
    """BVH4 nearest hits without memory for every lane's stack: several launches, the same records."""
    ctx = H.Context(0)
    v, f = W.soup(50_000, stream=W.STREAM_TEST)
    s = committed(ctx, v, f, H.LAYOUT_BVH4)
    rays = W.incoherent_rays(300_001, stream=W.STREAM_TEST)
    rays[::3, 7] = -1.0
    kernels()
    want = s.trace_nearest_host(rays)
    assert len([k for k in kernels() if "k_trace4_simple" in k]) == 1
    limited(0)
    assert refused(lambda: s.trace_nearest_host(rays))  # (nothing is idle after that)
    kernels()
    for share, launches in ((75_000, 5), (65_536, 5)):  # a quarter of the rays, and the least
        lanes = (share + 63) // 64 * 64
        limited(156 * lanes)
        got = s.trace_nearest_host(rays)
        assert len([k for k in kernels() if "k_trace4_simple" in k]) == launches
        assert np.asarray(got).tobytes() == np.asarray(want).tobytes()
    limited(156 * 65_536 - 1)
    assert refused(lambda: s.trace_nearest_host(rays))
    unlimited()
    assert np.asarray(s.trace_nearest_host(rays)).tobytes() == np.asarray(want).tobytes()
    s.close()
    ctx.close()


def refused_refit():
    """A refit that could not upload its vertices leaves the geometry as it was, its vertex count too."""
    ctx = H.Context(0)
    v, f = W.soup(200_000, stream=W.STREAM_TEST)
    v = np.concatenate([v, v[:1]])  # a vertex that no triangle uses
    rays = W.incoherent_rays(1000, stream=W.STREAM_TEST)
    s = committed(ctx, v, f)
    want = s.trace_nearest_host(rays)
    other = H.Scene(ctx)
    limited(0)
    assert refused(lambda: other.add_triangles(*W.soup(500_000)))  # nothing is idle after that
    limited(0)
    assert refused(lambda: s.update_triangles(0, v[:-1], quality=3))
    unlimited()
    s.commit()
    assert s.trace_nearest_host(rays).tobytes() == want.tobytes()
    s.update_triangles(0, 2 * v, quality=3)
    s.update_triangles(0, v, quality=3)
    s.commit()
    assert s.trace_nearest_host(rays).tobytes() == want.tobytes()
    s.close()
    ctx.close()


def wide_nodes():
    """The nodes of two levels are made for the scenes that walk them, by the commit and then by each refit."""
    ctx = H.Context(0)
    v, f = W.soup(50_000, stream=W.STREAM_TEST)
    rays = W.incoherent_rays(1000, stream=W.STREAM_TEST)
    s = H.Scene(ctx)
    g = s.add_triangles(v, f)

    def instanced():
        s.clear_instances()
        for k in range(2):
            s.add_instance(g, np.array([1, 0, 0, 0, 0, 1, 0, 0, 0, 0, 1, 0, 2 * k, 0, 0, 1], np.float32))
        return H.LAYOUT_BVH2

    def alone(layout):
        s.clear_instances()
        s.add_instance(g)
        return layout

    def made():
        return len([k for k in kernels() if "k_wide_nodes" in k])

    want = {}
    walked = False  # by the layout committed last
    kernels()
    for name in ("two", "bvh2", "two", "bvh4", "auto", "auto", "ploc", "bvh2"):
        layout = instanced() if name == "two" else alone(getattr(H, "LAYOUT_" + name.upper()))
        s.update_triangles(g, 2 * v, quality=3)
        s.update_triangles(g, v, quality=3)
        assert made() == (2 if walked else 0), f"refits before {name}"
        s.commit(layout=layout)
        s.commit(layout=layout)
        walks = name in ("bvh2", "auto")
        assert made() == (1 if walks and not walked else 0), f"commit of {name}"
        walked = walks
        hits = s.trace_nearest_host(rays)
        assert len([k for k in kernels() if "k_trace_quad" in k]) == int(walks), name
        assert hits.tobytes() == want.setdefault(name, hits).tobytes()
        assert name == "two" or hits[:, 0].tobytes() == want.setdefault("t", hits[:, 0]).tobytes()
    s.close()
    ctx.close()


def candidates():
    """The candidate that was set runs, in plain launches and in the graph; an untuned or tuned batch may keep the
    four-lane kernel."""
    ctx = H.Context(0)
    for sizes, rays in (([500, 3000], 700), ([500, 5000], 700)):
        scenes = [(*W.soup(n, stream=2200 + n), W.incoherent_rays(rays, stream=3200 + n)) for n in sizes]
        b = H.Batch(ctx, [x[0].shape[0] for x in scenes], [x[1].shape[0] for x in scenes], [rays] * len(sizes))
        b.upload(scenes)
        four = sizes[1] <= 4096

        def trace(run):
            kernels()
            run()
            hits = b.hits().tobytes()
            return [k for k in kernels() if "k_b_trace" in k], hits

        default, hits = trace(b.run)
        assert len(default) == 1 and ("k_b_trace_quad" in default[0]) == four, default
        for i, c in enumerate(H.batch_candidates()):
            b.set_candidate(i)
            assert b.candidate == i
            for run in (b.run, b.trace):
                names, h = trace(run)
                assert len(names) == 1 and h == hits
                want = f"k_b_trace_simpleILi{64 * c[0]}E" if c[1] == 0 else f"k_b_traceILi{c[0]}ELi{c[1]}ELi{c[2]}ELj{c[3]}E"
                assert want in names[0], (want, names)
            assert trace(b.run)[0] == [], "the graph is recorded once"
        chosen, ms = b.autotune(2)
        assert b.candidate == chosen == int(np.argmin(ms))
        kept, h = trace(b.run)
        assert len(kept) == 1 and h == hits
        last = kept[0]
        assert ("k_b_trace_quad" in last and four) or f"ELj{H.batch_candidates()[chosen][3]}E" in last or "simple" in last
        b.set_candidate(chosen)
        names, h = trace(b.trace)
        assert "k_b_trace_quad" not in names[0] and h == hits
        b.close()
    ctx.close()


if __name__ == "__main__":
    globals()[sys.argv[2]]()
    assert shim.shim_calls() > 0, "the engine's calls did not reach the shim"
    print("done", sys.argv[2], flush=True)
