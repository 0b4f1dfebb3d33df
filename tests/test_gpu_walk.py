"""The two forms of the BVH2 nearest-hit walk (four lanes per ray for small launches, one for large ones): bit for
bit the oracle's hits, and the counting variant's, at the sizes where the form or the last workgroup changes."""
import numpy as np
import pytest

import heavyrt_amd as H
from gpu_util import make_scene, say, trace
from heavyrt_amd import workloads as W
from oracle import oracle as O
from test_gpu_bvh4 import oracle_any_tree
from test_gpu_parity import check_build, rays_for

pytestmark = pytest.mark.gpu


def stacked(n=100, copies=2):
    """A small soup with n nested triangles in one Morton cell (one leaf), and every triangle twice (equal t)."""
    v, f = W.soup(500, stream=W.STREAM_TEST)
    tri = np.array([[0.0, 0.0, 0.0], [1.0, 0.0, 0.2], [0.0, 1.0, 0.1]]) - np.array([1.0, 1.0, 0.3]) / 3.0
    k = np.arange(1, n + 1)[:, None, None]
    nest = (np.array([0.5, 0.5, 0.5]) + 1e-3 * tri[None] * k + np.array([0, 0, 1e-6]) * k).reshape(-1, 3)
    v = np.concatenate([v, nest.astype(np.float32)])
    f = np.concatenate([f, 1500 + np.arange(3 * n, dtype=np.uint32).reshape(-1, 3)])
    return v, np.concatenate([f] * copies)


MESHES = {
    "one_triangle": lambda: (np.array([[0, 0, 0], [1, 0, 0], [0, 1, 0]], np.float32), np.array([[0, 1, 2]], np.uint32)),
    "two_leaves": lambda: W.soup(2, stream=W.STREAM_TEST),
    "three_leaves": lambda: W.soup(3, stream=W.STREAM_TEST),
    "stacked": lambda: stacked(50),
    "soup_20k": lambda: W.soup(20_000, stream=W.STREAM_TEST),
}


def same(a, b):
    for k in ("t", "prim", "u", "v"):
        np.testing.assert_array_equal(a[k].view(np.uint32), b[k].view(np.uint32))


@pytest.mark.parametrize("mesh", sorted(MESHES))
@pytest.mark.parametrize("n", [1, 3, 63, 65, 5000])
def test_small_launches_match_the_oracle(gpu_ctx, mesh, n):
    v, f = MESHES[mesh]()
    say(f"walk {mesh} {n}")
    s = make_scene(gpu_ctx, v, f, keep=False)
    rays = rays_for(v, n, 8100)
    rays[1::3, 7] = -2.0 * W.scene_diagonal(v)  # any-hit queries among them
    rays[2::7, 4:7] = [0.0, 0.0, -1.0]          # axis-parallel directions
    g = trace(s, rays, "full")
    t, prim = O.OracleBVH(v, f).trace(rays)[:2]
    np.testing.assert_array_equal(g["t"].view(np.uint32), t.view(np.uint32))
    np.testing.assert_array_equal(g["prim"], prim)
    same(g, trace(s, rays, "full", stats=True))  # counted on the node pairs
    s.close()


@pytest.mark.parametrize("test", [H.TRI_MT, H.TRI_WATERTIGHT], ids=["mt", "wt"])
def test_forms_agree_across_sizes(gpu_ctx, test):
    v, f = W.merge(W.icosphere(4), W.ground_quad())
    s = H.Scene(gpu_ctx)
    s.add_instance(s.add_triangles(v, f))
    s.set_triangle_test(test)
    s.commit()
    rays = rays_for(v, 140_000, 8200)
    whole = trace(s, rays, "full")  # a ray per lane
    for n in (1, 64, 32_768, 65_535, 65_536, 65_537, 131_073):
        say(f"walk size {n}")
        part = trace(s, rays[:n], "full")
        for k in ("t", "prim", "u", "v"):
            np.testing.assert_array_equal(part[k].view(np.uint32), whole[k][:n].view(np.uint32))
    s.close()


@pytest.mark.parametrize("layout", [H.LAYOUT_BVH4, H.LAYOUT_PLOC_FP16], ids=["bvh4", "ploc_fp16"])
@pytest.mark.parametrize("test", [H.TRI_MT, H.TRI_WATERTIGHT], ids=["mt", "wt"])
def test_bvh4_forms_agree_across_sizes(gpu_ctx, layout, test):
    v, f = W.merge(stacked(50), W.icosphere(3))
    s = H.Scene(gpu_ctx)
    s.add_instance(s.add_triangles(v, f))
    s.set_triangle_test(test)
    s.commit(layout=layout)
    rays = rays_for(v, 600_000, 8500)
    rays[1::5, 7] = -0.7 * W.scene_diagonal(v)  # any-hit queries among the nearest ones
    whole, hit = trace(s, rays[:200_000], "full"), trace(s, rays, "any")["hit"]  # a ray per lane
    say(f"bvh4 walk layout {layout}: {int(hit.sum())} of {hit.size} hit")
    for n in (1, 17, 64, 4097, 65_536, 65_537, 131_073):
        part = trace(s, rays[:n], "full")
        for k in ("t", "prim", "u", "v"):
            np.testing.assert_array_equal(part[k].view(np.uint32), whole[k][:n].view(np.uint32))
    for n in (1, 63, 65_537, 524_288, 524_289):
        np.testing.assert_array_equal(trace(s, rays[:n], "any")["hit"], hit[:n])
    s.close()


def test_nan_vertices_walk_the_pairs(gpu_ctx):
    """A leaf without finite corners has an inverted box, which a union of boxes drops: such trees keep their pairs."""
    v, f = W.soup(3000, stream=W.STREAM_TEST)
    v = v.copy()
    v[f[::97].reshape(-1)] = np.nan
    s = make_scene(gpu_ctx, v, f, keep=False)
    rays = rays_for(np.nan_to_num(v), 4000, 8300)
    same(trace(s, rays, "full"), trace(s, rays, "full", stats=True))
    s.close()


def test_refit_moves_the_walked_boxes(gpu_ctx):
    v, f = W.soup(20_000, stream=W.STREAM_TEST)
    s = make_scene(gpu_ctx, v, f, keep=False)
    s.update_triangles(0, (v * np.float32(1.5) + np.float32(0.25)).astype(np.float32), quality=3)
    s.commit()
    rays = rays_for(v * 1.5 + 0.25, 4000, 8400)
    same(trace(s, rays, "full"), trace(s, rays, "full", stats=True))
    s.close()


@pytest.mark.parametrize("test", [H.TRI_MT, H.TRI_WATERTIGHT], ids=["mt", "wt"])
@pytest.mark.parametrize("w,h", [(16, 8), (256, 256), (264, 256), (1032, 520)])
def test_frame_in_one_launch_equals_its_parts(gpu_ctx, test, w, h):
    import torch

    v, f = W.eye_scene()
    s = H.Scene(gpu_ctx)
    s.add_instance(s.add_triangles(v, f))
    s.set_triangle_test(test)
    s.commit()
    say(f"eye frame {w}x{h}")
    cam, stream = W.eye_camera(w, h), torch.cuda.current_stream().cuda_stream
    rays = torch.zeros((w * h, 8), dtype=torch.float32, device="cuda")
    xy = torch.zeros(w * h, dtype=torch.int32, device="cuda")
    image = torch.zeros((h, w), dtype=torch.int32, device="cuda")
    gpu_ctx.eye_make_rays(*cam, w, h, rays, xy, stream=stream)
    s.eye_render(*cam, w, h, W.EYE_PALETTE, image, stream=stream)
    torch.cuda.synchronize()
    prim = trace(s, rays.cpu().numpy(), "compact")["prim"]
    px = xy.cpu().numpy().view(np.uint32)
    want = np.zeros((h, w), np.uint32)
    hit = prim != 0xFFFFFFFF
    want[(px >> 16)[hit], (px & 0xFFFF)[hit]] = W.EYE_PALETTE[prim[hit] % W.EYE_PALETTE.size]
    np.testing.assert_array_equal(image.cpu().numpy().view(np.uint32), want)
    s.close()


@pytest.mark.parametrize("layout", [H.LAYOUT_BVH4, H.LAYOUT_BVH4_FP16], ids=["fp32", "fp16"])
def test_sorted_batch_equals_its_parts(gpu_ctx, layout):
    """2^20 rays or more on a tree of 128 MB or more are traced in sorted order, under either triangle test."""
    rng = np.random.default_rng(7)
    n = 2_200_000
    v = (rng.random((n, 1, 3)) + 0.02 * (rng.random((n, 3, 3)) - 0.5)).reshape(-1, 3).astype(np.float32)
    f = np.arange(3 * n, dtype=np.uint32).reshape(-1, 3)
    s = H.Scene(gpu_ctx)
    s.add_instance(s.add_triangles(v, f))
    rays = W.incoherent_rays((1 << 20) + 3, stream=W.STREAM_TEST)
    rays[5::1001, 7] = -0.5
    rays[6::1003, 4] = np.nan
    for test in (H.TRI_MT, H.TRI_WATERTIGHT):
        s.set_triangle_test(test)
        s.commit(layout=layout)
        say(f"sorted batch layout {layout} test {test}")
        whole = trace(s, rays, "full")
        for lo, hi in ((0, 1000), (600_000, (1 << 20) + 3)):
            part = trace(s, rays[lo:hi], "full")
            for k in ("t", "prim", "u", "v"):
                np.testing.assert_array_equal(part[k].view(np.uint32), whole[k][lo:hi].view(np.uint32))
    s.close()


@pytest.mark.parametrize("ntris", [3, 255, 4096, 4097, 5000, 70_000])
def test_clustered_hierarchy_at_round_edges(gpu_ctx, ntris):
    """The clustering's two forms (a workgroup up to 4,096 clusters, tiles of 256 above) build the oracle's nodes."""
    v, f = W.soup(ntris, stream=W.STREAM_TEST + 1)
    s = H.Scene(gpu_ctx, keep_build_arrays=True)
    s.add_instance(s.add_triangles(v, f))
    s.commit(layout=H.LAYOUT_PLOC)
    say(f"clustering {ntris}")
    ob, clustered = oracle_any_tree(v, f)
    sizes = s.dump(0, H.DUMP_ANY_TREE | H.DUMP_SIZES)
    assert (int(sizes[1]), int(sizes[5])) == (ob.leaves, int(clustered))
    np.testing.assert_array_equal(s.dump(0, H.DUMP_ANY_TREE | H.DUMP_LR_NODES), ob.lr_nodes())
    s.close()


@pytest.mark.parametrize("layout", [H.LAYOUT_BVH2, H.LAYOUT_AUTO_FP16], ids=["bvh2", "auto_fp16"])
def test_commit_is_whole_for_a_trace_on_another_stream(gpu_ctx, layout):
    """The rays wait on the device and the stream is idle: the trace starts as soon as the commit has returned."""
    import torch
    v, f = W.soup(400_000, stream=W.STREAM_TEST)
    rays = torch.from_numpy(rays_for(v, 4000, 8500)).cuda()
    out = [torch.zeros((4000, 8), dtype=torch.int32, device="cuda") for _ in range(2)]
    other = torch.cuda.Stream()
    torch.cuda.synchronize()
    s = H.Scene(gpu_ctx)
    s.add_instance(s.add_triangles(v, f))
    for scale in (1.0, 1.25):
        if scale != 1.0:
            s.update_triangles(0, (v * np.float32(scale)).astype(np.float32), quality=3)
        s.commit(layout=layout)
        s.trace_nearest(rays, 4000, out[0], H.HIT_FULL, stream=other.cuda_stream)
        torch.cuda.synchronize()
        s.trace_nearest(rays, 4000, out[1], H.HIT_FULL, stream=other.cuda_stream)
        torch.cuda.synchronize()
        np.testing.assert_array_equal(out[0].cpu().numpy(), out[1].cpu().numpy())
    s.close()


SMALL = [1, 2, 3, 64, 65, 255, 256, 512, 1023, 1024, 1025, 4095, 4096, 4097]


@pytest.mark.parametrize("n", SMALL)
def test_small_build_equals_the_oracle(gpu_ctx, n):
    """Trees of one workgroup, up to and past the last size, with triangles that share a code; then their refit."""
    v, f = W.soup(n, stream=W.STREAM_TEST)
    if n >= 256:
        f = f.copy()
        f[5::7] = f[5]  # one code many times over
        f[6::64] = f[6]
        f = np.concatenate([f[:n - n // 8], f[:n // 8]]) if n // 7 < 127 else W.soup(n, stream=W.STREAM_TEST)[1]
    say(f"small build {n}")
    ob = O.OracleBVH(v, f)
    s = make_scene(gpu_ctx, v, f)
    check_build(s, ob)
    rays = rays_for(v, 500, 8600)
    g = trace(s, rays, "full")
    t, prim = ob.trace(rays)[:2]
    np.testing.assert_array_equal(g["t"].view(np.uint32), t.view(np.uint32))
    np.testing.assert_array_equal(g["prim"], prim)
    pairs = s.dump(0, H.DUMP_PAIRS)
    s.update_triangles(0, (v * np.float32(2)).astype(np.float32), quality=3)
    s.update_triangles(0, v, quality=3)
    np.testing.assert_array_equal(s.dump(0, H.DUMP_PAIRS), pairs)  # through the parents and ranges
    s.close()


@pytest.mark.parametrize("sizes,rays", [([1, 2, 3, 256, 1000, 1024], 37), (SMALL[:-1], 700), (SMALL[:-1], 9000),
                                        (SMALL, 37)],
                         ids=["1024", "4096", "4096_many_rays", "4097"])
def test_small_batch_equals_solo_scenes(gpu_ctx, sizes, rays):
    import torch
    from test_gpu_batch import make_batch
    scenes = []
    for k, n in enumerate(sizes):
        v, f = W.soup(n, stream=2000 + k)
        scenes.append((v, f, W.incoherent_rays(0 if k == 1 else rays + k, stream=3000 + k)))
    scenes[2][0][scenes[2][1][0]] = np.nan  # one scene is walked on its pairs
    b = make_batch(gpu_ctx, scenes)
    stream = torch.cuda.current_stream().cuda_stream
    for run in (b.run, b.run, b.trace):
        run(stream)
        torch.cuda.synchronize()
        hits = b.hits()
        for k, (v, f, r) in enumerate(scenes):
            s = make_scene(gpu_ctx, v, f, keep=False)
            np.testing.assert_array_equal(b.dump(k, H.DUMP_SIZES)[:4], s.dump(0, H.DUMP_SIZES)[:4])
            np.testing.assert_array_equal(b.dump(k, H.DUMP_PAIRS), s.dump(0, H.DUMP_PAIRS))
            np.testing.assert_array_equal(b.dump(k, H.DUMP_PERM), s.dump(0, H.DUMP_PERM))
            if r.shape[0]:
                c = trace(s, r, "compact")
                np.testing.assert_array_equal(hits[b.ray_off[k]:b.ray_off[k + 1], 0], c["t"].view(np.uint32))
                np.testing.assert_array_equal(hits[b.ray_off[k]:b.ray_off[k + 1], 1], c["prim"])
            s.close()
    b.close()


@pytest.mark.parametrize("sizes,rays", [([700, 3000], 40_000), ([700, 5000], 40_000), ([700, 5000], 600_000)],
                         ids=["small", "lane", "stream"])
def test_batch_default_kernel_equals_the_candidates(gpu_ctx, sizes, rays):
    import torch
    from test_gpu_batch import make_batch
    scenes = [(*W.soup(n, stream=2100 + k), W.incoherent_rays(rays + k, stream=3100 + k)) for k, n in enumerate(sizes)]
    for _, _, r in scenes:
        r[1::3, 7] = -0.5  # any-hit queries among them
    b = make_batch(gpu_ctx, scenes)
    stream = torch.cuda.current_stream().cuda_stream
    b.run(stream)
    torch.cuda.synchronize()
    ref = b.hits()
    assert b.candidate == 1
    for c in (1, 11, 12, 14):
        b.set_candidate(c)
        b.run(stream)
        torch.cuda.synchronize()
        np.testing.assert_array_equal(b.hits(), ref)
    b.close()


@pytest.mark.parametrize("n,dup", [(4097, 1), (16384, 1), (16385, 130), (33_000, 200), (70_000, 1)])
def test_leaf_pass_and_refit_at_group_edges(gpu_ctx, n, dup):
    """Trees over one or several of the refit's groups, with runs longer than the leaf pass stages."""
    v, f = W.soup(n, stream=W.STREAM_TEST)
    f = f.copy()
    for k in range(0, dup - 1):  # a run of up to 127 and many of two and three
        f[(k * 71) % n if k < 100 else (k * 37) % n] = f[n // 2 if k < 100 else n // 3]
    ob = O.OracleBVH(v, f)
    s = make_scene(gpu_ctx, v, f)
    check_build(s, ob)
    pairs, perm = s.dump(0, H.DUMP_PAIRS), s.dump(0, H.DUMP_PERM)
    rays = rays_for(v, 2000, 8700)
    g = trace(s, rays, "full")
    t, prim = ob.trace(rays)[:2]
    np.testing.assert_array_equal(g["t"].view(np.uint32), t.view(np.uint32))
    np.testing.assert_array_equal(g["prim"], prim)
    s.update_triangles(0, (v * np.float32(2)).astype(np.float32), quality=3)
    assert (s.dump(0, H.DUMP_PAIRS) != pairs).any()
    s.update_triangles(0, v, quality=3)
    np.testing.assert_array_equal(s.dump(0, H.DUMP_PAIRS), pairs)
    np.testing.assert_array_equal(s.dump(0, H.DUMP_PERM), perm)
    s.close()


@pytest.mark.parametrize("full", [False, True], ids=["compact", "full"])
def test_bvh4_launches_of_a_large_batch_join(gpu_ctx, full):
    """More rays than one launch takes: the seam's records are those of the same rays traced by themselves."""
    import torch
    v, f = W.soup(3000, stream=W.STREAM_TEST)
    s = H.Scene(gpu_ctx)
    s.add_instance(s.add_triangles(v, f))
    s.commit(layout=H.LAYOUT_BVH4_FP16)
    n, seam = (1 << 22) + 65, 1 << 22
    rays = torch.from_numpy(np.tile(rays_for(v, 4096, 8800), (n // 4096 + 1, 1))[:n]).cuda()
    rays[:, 0] += torch.arange(n, device="cuda") * 1e-8
    words, fmt = (8, H.HIT_FULL) if full else (2, H.HIT_COMPACT)
    out = torch.full((n, words), -7, dtype=torch.int32, device="cuda")
    part = torch.zeros((300_000, words), dtype=torch.int32, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    s.trace_nearest(rays, n, out, fmt, stream=stream)
    lo = n - 300_000
    s.trace_nearest(rays[lo:].contiguous(), 300_000, part, fmt, stream=stream)
    torch.cuda.synchronize()
    assert lo < seam < n and torch.equal(out[lo:], part)
    s.trace_nearest(rays[:300_000].contiguous(), 300_000, part, fmt, stream=stream)
    torch.cuda.synchronize()
    assert torch.equal(out[:300_000], part)
    s.close()


@pytest.mark.parametrize("n", [700, 70_000], ids=["four_lanes", "one_lane"])
def test_fp16_planes_picked_by_direction(gpu_ctx, n):
    """Zero, negative-zero and signed direction components, origins on box planes, triangles without finite corners:
    the hits of the FP16 walk are the counting variant's, which takes minimum and maximum."""
    v, f = W.soup(5000, stream=W.STREAM_TEST)
    v = v.copy()
    v[f[::61].reshape(-1)] = np.nan
    s = H.Scene(gpu_ctx)
    s.add_instance(s.add_triangles(v, f))
    s.commit(layout=H.LAYOUT_BVH4_FP16)
    rays = rays_for(np.nan_to_num(v), n, 8900)
    rays[1::5, 4] = 0.0
    rays[2::5, 5] = -0.0
    rays[3::5, 4:7] = [0.0, 0.0, -1.0]
    rays[4::5, 0:3] = v[f[1 + (np.arange(len(rays[4::5])) % 60), 0]].astype(np.float16)  # on FP16 planes
    same(trace(s, rays, "full"), trace(s, rays, "full", stats=True))
    s.close()
