"""What a loaded mesh goes through before and while its tree is built, at the sizes where the path changes: the index
check, vertex strides, and one-workgroup builds with many triangles in one Morton cell."""
import numpy as np
import pytest

import heavyrt_amd as H
from gpu_util import make_scene, say, trace
from heavyrt_amd import workloads as W
from oracle import oracle as O
from test_gpu_parity import check_build, rays_for

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ntris", [16383, 16384, 16385, 16386, 16387, 200_001])
def test_index_out_of_range_is_refused(gpu_ctx, ntris):
    """On the host below 16,384 triangles, on the device from there on, its last one to three words too."""
    v, f = W.soup(ntris, stream=W.STREAM_TEST)
    s = H.Scene(gpu_ctx)
    flat = f.reshape(-1)
    for at in (0, flat.size // 2, flat.size - 4, flat.size - 3, flat.size - 2, flat.size - 1):
        for bad in (len(v), 0xFFFFFFFF):
            say(f"index check {ntris}: word {at} = {bad}")
            g = flat.copy()
            g[at] = bad
            with pytest.raises(H.HrtError) as e:
                s.add_triangles(v, g.reshape(-1, 3))
            assert e.value.status == 1 and s.geom_count == 0
    s.add_instance(s.add_triangles(v, f))  # its largest index is the last vertex
    s.commit()
    rays = rays_for(v, 500, 9100)
    t, prim = O.OracleBVH(v, f).trace(rays)[:2]
    g = trace(s, rays, "full")
    np.testing.assert_array_equal(g["t"].view(np.uint32), t.view(np.uint32))
    np.testing.assert_array_equal(g["prim"], prim)
    s.close()


@pytest.mark.parametrize("n", [200, 20_000])
@pytest.mark.parametrize("floats", [4, 5, 8, 9, 10, 33])
def test_vertex_strides(gpu_ctx, n, floats):
    """Up to 32 bytes the records go up as they are, wider ones are packed first: the same trees as packed vertices."""
    v, f = W.soup(n, stream=W.STREAM_TEST)
    say(f"stride {4 * floats}, {n} triangles")

    def wide(x):
        w = np.full((len(x), floats), np.nan, np.float32)  # what is between the positions is not read
        w[:, :3] = x
        return w

    a, b = make_scene(gpu_ctx, v, f), make_scene(gpu_ctx, wide(v), f)

    def same():
        for what in (H.DUMP_SIZES, H.DUMP_PAIRS, H.DUMP_PERM):
            np.testing.assert_array_equal(a.dump(0, what), b.dump(0, what))
        rays = rays_for(v, 500, 9200)
        for s in (a, b):
            s.commit()
        x, y = trace(a, rays, "full"), trace(b, rays, "full")
        for k in ("t", "prim", "u", "v"):
            np.testing.assert_array_equal(x[k].view(np.uint32), y[k].view(np.uint32))

    same()
    moved = (v[::-1] * np.float32(1.5)).astype(np.float32)
    for quality in (3, 1):  # a refit, a rebuild
        a.update_triangles(0, moved, quality=quality)
        b.update_triangles(0, wide(moved), quality=quality)
        same()
    a.close()
    b.close()


def with_runs(n, seed, longest=9):
    """A soup where triangles share Morton cells: copies in runs of 1 to `longest` everywhere, one run of 127 and one of
    64 in cells of their own, the copies scattered over the ids."""
    v, f = W.soup(n, stream=seed)
    rng = np.random.default_rng(seed)
    src, at = np.zeros(n, np.int64), 0
    for size in [127, 64] + list(rng.integers(1, longest + 1, n)):
        if at < n:
            src[at:at + size] = at
            at += size
    return v, f[rng.permutation(src)]


@pytest.mark.parametrize("longest", [2, 9])  # more leaves than threads, and fewer
@pytest.mark.parametrize("n", [256, 511, 512, 513, 1023, 1024, 1025, 2047, 2048, 3000, 4095, 4096, 4097])
def test_small_build_with_shared_codes(gpu_ctx, n, longest):
    v, f = with_runs(n, 9300 + n, longest)
    say(f"small build with runs {n} {longest}")
    ob = O.OracleBVH(v, f)
    s = make_scene(gpu_ctx, v, f)
    check_build(s, ob)
    sizes, pairs = s.dump(0, H.DUMP_SIZES), s.dump(0, H.DUMP_PAIRS)
    assert sizes[2] == 127 and sizes[1] < 3 * n // 4, sizes
    rays = rays_for(v, 1000, 9400)
    t, prim = ob.trace(rays)[:2]
    g = trace(s, rays, "full")
    np.testing.assert_array_equal(g["t"].view(np.uint32), t.view(np.uint32))
    np.testing.assert_array_equal(g["prim"], prim)
    s.update_triangles(0, (v * np.float32(2)).astype(np.float32), quality=3)
    s.update_triangles(0, v, quality=3)
    np.testing.assert_array_equal(s.dump(0, H.DUMP_PAIRS), pairs)
    s.close()


def test_small_batch_with_shared_codes(gpu_ctx):
    import torch
    from test_gpu_batch import make_batch
    scenes = [(*with_runs(n, 9500 + n, 2 if n > 1024 else 9), W.incoherent_rays(300, stream=9600 + n)) for n in (256, 1025, 2048, 4096)]
    b = make_batch(gpu_ctx, scenes)
    b.run(torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    b.status()
    hits = b.hits()
    for k, (v, f, r) in enumerate(scenes):
        s = make_scene(gpu_ctx, v, f, keep=False)
        for what in (H.DUMP_PAIRS, H.DUMP_PERM):
            np.testing.assert_array_equal(b.dump(k, what), s.dump(0, what))
        c = trace(s, r, "compact")
        np.testing.assert_array_equal(hits[b.ray_off[k]:b.ray_off[k + 1], 0], c["t"].view(np.uint32))
        np.testing.assert_array_equal(hits[b.ray_off[k]:b.ray_off[k + 1], 1], c["prim"])
        s.close()
    b.close()


@pytest.mark.parametrize("nverts", [16383, 16384, 16385, 40_000])
def test_few_triangles_of_many_vertices(gpu_ctx, nverts):
    """The scene box goes over every vertex, used or not; past 16,384 of them one workgroup no longer reads them all."""
    import torch
    from test_gpu_batch import make_batch
    v, f = W.soup(300, stream=W.STREAM_TEST)
    spread = (4.0 * W.uniform01(W.pcg32(nverts - len(v), 3, 9700)) - 2.0).astype(np.float32)
    v = np.concatenate([v, spread])
    say(f"300 triangles, {nverts} vertices")
    ob = O.OracleBVH(v, f)
    s = make_scene(gpu_ctx, v, f)
    check_build(s, ob)
    rays = rays_for(v, 500, 9800)
    b = make_batch(gpu_ctx, [(v, f, rays)])
    b.run(torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(b.dump(0, H.DUMP_PAIRS), s.dump(0, H.DUMP_PAIRS))
    t, prim = ob.trace(rays)[:2]
    np.testing.assert_array_equal(b.hits(), np.stack([t.view(np.uint32), prim], 1))
    b.close()
    s.close()
