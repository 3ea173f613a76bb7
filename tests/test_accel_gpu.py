"""GPU parity of the wide-BVH traversal kernel against the CPU oracle.

Bar: hit triangle index, t and barycentrics bit-exact against the oracle's
brute force under the same triangle test and the canonical tie rule
(smallest id among equal t), for both the reference-compatible TriAccel test
and the watertight test.  At the benchmark's full size (1,310,720 triangles,
2048^2 coherent + 2048^2 incoherent rays) the kernel is compared bit-exactly
with the host walker over the same BVH on every ray and with the oracle's
brute force on a seeded sample of rays (watertight mode), and in TriAccel
mode with the oracle's restatement of the reference's QBVH on every ray.
"""
import numpy as np
import pytest

import orc
from lmx import accel, scenes

pytestmark = pytest.mark.gpu


def _gpu_hits(a, rays, dev):
    import torch
    r = torch.from_numpy(rays).to(dev)
    h = a.intersect(r)
    torch.cuda.synchronize()
    return h.cpu().numpy()


@pytest.mark.parametrize("mode", [accel.ISECT_TRIACCEL, accel.ISECT_WATERTIGHT])
def test_small_mesh_bitexact_vs_bruteforce(gpu, mode):
    v, f = scenes.displaced_icosphere(4, seed=3)
    coh, inc = scenes.traversal_rays(v, res=64, n_incoherent=8192)
    rays = np.concatenate([coh, inc])
    a = accel.Accel(v, f, isect=mode)
    hg = _gpu_hits(a, rays, gpu)
    ho = orc.closest_hit_naive(v, f, rays, test=mode, tie=orc.TIE_MIN_ID)
    assert (orc.hit_ids(ho) != orc.MISS).sum() > 1000
    np.testing.assert_array_equal(hg.view(np.uint32), ho.view(np.uint32))


@pytest.mark.parametrize("n", [0, 1, 5, 63, 64, 65, 1000])
def test_ragged_ray_counts(gpu, n):
    v, f = scenes.displaced_icosphere(3, seed=5)
    _, inc = scenes.traversal_rays(v, res=4, n_incoherent=max(n, 1), seed=9)
    rays = inc[:n]
    a = accel.Accel(v, f)
    if n == 0:
        import torch
        h = a.intersect(torch.zeros((0, 8), dtype=torch.float32, device=gpu))
        assert h.shape == (0, 4)
        return
    hg = _gpu_hits(a, rays, gpu)
    ho = orc.closest_hit_naive(v, f, rays, test=orc.TEST_WATERTIGHT, tie=orc.TIE_MIN_ID)
    np.testing.assert_array_equal(hg.view(np.uint32), ho.view(np.uint32))


@pytest.mark.parametrize("scale,shift", [(1e-12, 0.0), (1e12, 0.0), (1.0, 1e6), (1e-6, 1.0)])
def test_extreme_scales_bitexact_vs_bruteforce(gpu, scale, shift):
    """Scene sizes from 1e-12 to 1e12 and far from the origin (ray origins
    and tmin scaled with the scene): the kernel's byte-grid box test, with
    its binary16 subnormal operands, still finds exactly the brute force's
    hits."""
    v, f = scenes.displaced_icosphere(4, seed=3)
    coh, inc = scenes.traversal_rays(v, res=48, n_incoherent=4096)
    rays = np.concatenate([coh, inc]).copy()
    v = (v.astype(np.float64) * scale + shift).astype(np.float32)
    rays[:, 0:3] = (rays[:, 0:3].astype(np.float64) * scale + shift).astype(np.float32)
    rays[:, 3] = np.float32(rays[0, 3] * scale)
    a = accel.Accel(v, f)
    hg = _gpu_hits(a, rays, gpu)
    ho = orc.closest_hit_naive(v, f, rays, test=orc.TEST_WATERTIGHT, tie=orc.TIE_MIN_ID)
    assert (orc.hit_ids(ho) != orc.MISS).sum() > 1000
    np.testing.assert_array_equal(hg.view(np.uint32), ho.view(np.uint32))


@pytest.mark.parametrize("n", [327679, 327680, 327681, 400003])
def test_fixed_and_claimed_chunks(gpu, n):
    """Ray counts around 5,120 waves x 64 rays, where the waves' fixed first
    chunks stop covering the batch and the rest is claimed through the
    region cursors: every ray is traced exactly once (bit-exact against the
    host walker over the same BVH)."""
    v, f = scenes.displaced_icosphere(4, seed=6)
    _, rays = scenes.traversal_rays(v, res=4, n_incoherent=n, seed=10)
    a = accel.Accel(v, f)
    hg = _gpu_hits(a, rays, gpu)
    hh = a.intersect_host(rays)
    assert (accel.hit_ids(hh) != accel.MISS).sum() > n // 10
    np.testing.assert_array_equal(hg.view(np.uint32), hh.view(np.uint32))


def test_full_size_traversal_benchmark(gpu):
    v, f = scenes.traversal_scene()
    assert f.shape[0] == 1310720
    coh, inc = scenes.traversal_rays(v)
    rays = np.concatenate([coh, inc])
    assert rays.shape[0] == 8388608
    a = accel.Accel(v, f)
    hg = _gpu_hits(a, rays, gpu)
    hh = a.intersect_host(rays)
    np.testing.assert_array_equal(hg.view(np.uint32), hh.view(np.uint32))
    # seeded sample against brute force over all 1.3M triangles
    idx = np.random.default_rng(0).choice(rays.shape[0], 512, replace=False)
    ho = orc.closest_hit_naive(v, f, rays[idx], test=orc.TEST_WATERTIGHT, tie=orc.TIE_MIN_ID, nthreads=8)
    np.testing.assert_array_equal(hg[idx].view(np.uint32), ho.view(np.uint32))
    # every coherent ray aimed at the sphere's silhouette interior hits it
    ids = accel.hit_ids(hg)
    assert (ids[: coh.shape[0]] != accel.MISS).mean() > 0.2
    assert (ids[coh.shape[0]:] != accel.MISS).mean() > 0.3


def test_full_size_triaccel_vs_reference_qbvh_every_ray(gpu):
    """The benchmark's full size in the reference's TriAccel mode
    (triaccel.h:93-151) against the oracle's restatement of the reference's
    own accel, the 4-wide QBVH (accel_qbvh.cpp:392-481, a later equal-t hit
    replaces an earlier one), on all 8,388,608 rays: the same triangle on
    every ray except exact t ties (two triangles hit at the same t, where the
    kernel keeps the smallest id and the QBVH its traversal order), and where
    the triangle agrees t and barycentrics bit for bit (the same FP32
    operations in the same order).  Ties are checked with the FP64 solve:
    both triangles are hit at that t."""
    from test_oracle import _fp64_solve
    v, f = scenes.traversal_scene()
    coh, inc = scenes.traversal_rays(v)
    rays = np.concatenate([coh, inc])
    a = accel.Accel(v, f, isect=accel.ISECT_TRIACCEL)
    hg = _gpu_hits(a, rays, gpu)
    ho = orc.QBVH(v, f).intersect(rays, nthreads=16)
    ig, io = accel.hit_ids(hg), orc.hit_ids(ho)
    same = ig == io
    assert (ig != accel.MISS).mean() > 0.5
    np.testing.assert_array_equal(hg[same].view(np.uint32), ho[same].view(np.uint32))
    bad = np.nonzero(~same)[0]
    print(f"TriAccel mode, {rays.shape[0]} rays: {len(bad)} with another triangle")
    assert len(bad) <= 1e-5 * rays.shape[0]
    for k in bad:
        assert ig[k] != accel.MISS and io[k] != accel.MISS, (k, ig[k], io[k])
        assert hg[k, 0] == ho[k, 0], (k, hg[k, 0], ho[k, 0])          # an exact t tie
        for tri in (ig[k], io[k]):
            t, b0, b1 = _fp64_solve(v, f, rays[k:k + 1], np.array([tri]))
            assert abs(t[0] - hg[k, 0]) <= 1e-5 * abs(t[0])
            assert min(b0[0], b1[0], 1.0 - b0[0] - b1[0]) > -1e-5
    assert a.info()["stack_overflow"] == 0


@pytest.mark.parametrize("simple2", [False, True])
@pytest.mark.parametrize("mode", [accel.ISECT_TRIACCEL, accel.ISECT_WATERTIGHT])
def test_accel3_analytic_quads_on_gpu(gpu, simple2, mode):
    """src/lightmetrica-test/test_accel3.cpp:272-345 through the HIP kernel:
    p, gn and uv within EpsLarge = 1e-3 of the analytic answer."""
    from test_oracle import (SIMPLE_F, SIMPLE_UV, SIMPLE_V, SIMPLE2_F, SIMPLE2_UV, SIMPLE2_V,
                             hit_geometry, quad_rays)
    v, f, uv = (SIMPLE2_V, SIMPLE2_F, SIMPLE2_UV) if simple2 else (SIMPLE_V, SIMPLE_F, SIMPLE_UV)
    rays, expect = quad_rays(simple2)
    a = accel.Accel(v, f, isect=mode)
    hg = _gpu_hits(a, rays, gpu)
    assert (accel.hit_ids(hg) != accel.MISS).all()
    p, gn, tuv = hit_geometry(v, f, uv, rays, hg)
    np.testing.assert_allclose(p, expect, atol=1e-3)
    n_exp = np.array([0, 0, 1], np.float32) if not simple2 else np.array([1, 0, 1], np.float32) / np.sqrt(2)
    np.testing.assert_allclose(gn, np.broadcast_to(n_exp, gn.shape), atol=1e-3)
    np.testing.assert_allclose(tuv, expect[:, 0:2], atol=1e-3)
    ho = orc.closest_hit_naive(v, f, rays, test=mode, tie=orc.TIE_MIN_ID)
    np.testing.assert_array_equal(hg.view(np.uint32), ho.view(np.uint32))


@pytest.mark.parametrize("tmax_scale", [0.5, 1.0, 2.0])
def test_occlusion_matches_closest_hit(gpu, tmax_scale):
    """Any-hit traversal: a ray is occluded on [tmin, tmax] exactly when the
    closest hit lies in that range, and the reported triangle really is hit
    there.  Mixed lengths exercise lanes that finish early and are refilled."""
    import torch
    v, f = scenes.displaced_icosphere(5, seed=13)
    coh, inc = scenes.traversal_rays(v, res=96, n_incoherent=40000, seed=21)
    rays = np.concatenate([coh, inc]).copy()
    hc = orc.closest_hit_naive(v, f, rays, test=orc.TEST_WATERTIGHT, tie=orc.TIE_MIN_ID)
    ids = orc.hit_ids(hc)
    rng = np.random.default_rng(4)
    # finite tmax around the closest hit distance (and beyond for misses)
    t_ref = np.where(ids != orc.MISS, hc[:, 0], 3.0)
    rays[:, 7] = (t_ref * tmax_scale * rng.uniform(0.7, 1.3, rays.shape[0])).astype(np.float32)
    a = accel.Accel(v, f)
    hg = a.occluded(torch.from_numpy(rays).to(gpu))
    torch.cuda.synchronize()
    hg = hg.cpu().numpy()
    occ_expect = (ids != orc.MISS) & (hc[:, 0] <= rays[:, 7])
    occ = accel.hit_ids(hg) != accel.MISS
    np.testing.assert_array_equal(occ, occ_expect)
    # the reported triangle is hit by that ray within range
    k = np.nonzero(occ)[0][:2000]
    for i in k[:200]:
        tri = int(accel.hit_ids(hg)[i])
        one = orc.closest_hit_naive(v, f[tri:tri + 1], rays[i:i + 1], test=orc.TEST_WATERTIGHT)
        assert orc.hit_ids(one)[0] == 0


@pytest.mark.parametrize("mode", [accel.ISECT_TRIACCEL, accel.ISECT_WATERTIGHT])
@pytest.mark.parametrize("subdiv", [0, 2, 5])
@pytest.mark.parametrize("n", [1, 7, 9, 63, 4097, 8 * 5120, 8 * 5120 + 1, 12 * 4096 + 5, 13 * 5120 + 1])
def test_last_rays_of_a_wave(gpu, n, subdiv, mode):
    """The part of the kernel that traces a wave's last rays with all its
    lanes: alone (one ray per wave, up to 8), and after the one-ray-per-lane
    loop (64 a wave); trees of one level and of many; tmin below 0, finite
    tmax, zero direction components and rays that cannot hit.  Bit-exact
    against the host walker over the same BVH, which visits one ray at a
    time; an occlusion query agrees with the closest hit."""
    import torch
    v, f = scenes.displaced_icosphere(subdiv, seed=17)
    _, rays = scenes.traversal_rays(v, res=2, n_incoherent=n, seed=n)
    rays = rays.copy()
    rays[::5, 4 + np.arange(3)[n % 3]] = 0.0
    rays[1::7, 3] = -2.0
    rays[2::3, 7] = 0.7
    rays[3::11, 7] = -1.0
    a = accel.Accel(v, f, isect=mode)
    d = torch.from_numpy(rays).to(gpu)
    hg, ho = a.intersect(d), a.occluded(d)
    torch.cuda.synchronize()
    hh = a.intersect_host(rays)
    np.testing.assert_array_equal(hg.cpu().numpy().view(np.uint32), hh.view(np.uint32))
    np.testing.assert_array_equal(accel.hit_ids(ho.cpu().numpy()) != accel.MISS, accel.hit_ids(hh) != accel.MISS)
    assert a.info()["stack_overflow"] == 0


@pytest.mark.parametrize("mode", [accel.ISECT_TRIACCEL, accel.ISECT_WATERTIGHT])
@pytest.mark.parametrize("n", [9, 2001, 200003])
def test_unusual_ranges(gpu, n, mode):
    """tmin and tmax of NaN (either sign), infinity, -0 and crossed, and
    origins and directions that are not finite: the same hits as the host
    walker's, bit for bit, whichever part of the kernel traces the ray."""
    import torch
    v, f = scenes.displaced_icosphere(3, seed=5)
    _, rays = scenes.traversal_rays(v, res=2, n_incoherent=n, seed=n)
    rays = rays.copy()
    odd = np.array([0x7fc00000, 0xffc00000, 0x7f800000, 0xff800000, 0x80000000, 0x3f000000], np.uint32).view(np.float32)
    k = np.arange(len(rays))
    rays[:, 7] = np.where(k % 8 < 6, odd[k % 8 % 6], rays[:, 7])
    rays[:, 3] = np.where(k % 11 < 6, odd[k % 11 % 6], rays[:, 3])
    rays[5::37, 0], rays[7::41, 5], rays[11::43, 6], rays[3::47, 1] = np.inf, np.nan, -np.inf, np.nan
    a = accel.Accel(v, f, isect=mode)
    d = torch.from_numpy(rays).to(gpu)
    hg, ho = a.intersect(d).cpu().numpy(), a.occluded(d).cpu().numpy()
    hh = a.intersect_host(rays)
    np.testing.assert_array_equal(hg.view(np.uint32), hh.view(np.uint32))
    np.testing.assert_array_equal(accel.hit_ids(ho) != accel.MISS, accel.hit_ids(hh) != accel.MISS)
    assert n < 100 or (accel.hit_ids(hh) != accel.MISS).any()


@pytest.mark.parametrize("mode", [accel.ISECT_TRIACCEL, accel.ISECT_WATERTIGHT])
def test_long_batches(gpu, mode):
    """Batches long enough for the launch shapes of a tree beyond an XCD's L2
    (81,920 triangles): 16 or 20 waves per CU, and the loop without the part
    that finishes a wave's last rays (occlusion from 256 rays a wave on,
    closest hits from 2,048).  The same rays in batches below all of those
    lines: the same hits bit for bit, the same rays occluded."""
    import torch
    v, f = scenes.displaced_icosphere(6, seed=17)
    _, rays = scenes.traversal_rays(v, res=2, n_incoherent=1 << 20, seed=4)
    a = accel.Accel(v, f, isect=mode)
    one = torch.from_numpy(rays).to(gpu)
    waves = 20 * torch.cuda.get_device_properties(gpu).multi_processor_count
    for n in (256 * waves - 1, 256 * waves, 400 * waves, 2048 * waves + 77):
        k = torch.arange(n, device=gpu) % one.shape[0]
        d = one[k].contiguous()
        d[:, 7] = torch.where(k % 3 == 0, 0.9 + 1e-7 * torch.arange(n, device=gpu), d[:, 7])
        hit, occ = a.intersect(d).view(torch.int32), a.occluded(d).view(torch.int32)[:, 3]
        for b in range(0, n, 1 << 20):
            part = d[b:b + (1 << 20)]
            assert torch.equal(hit[b:b + (1 << 20)], a.intersect(part).view(torch.int32)), (n, b)
            assert torch.equal(occ[b:b + (1 << 20)] == -1, a.occluded(part).view(torch.int32)[:, 3] == -1), (n, b)
        assert torch.equal(occ == -1, hit[:, 3] == -1)
    assert a.info()["stack_overflow"] == 0
    np.testing.assert_array_equal(hit[-100003:].cpu().numpy().view(np.uint32),
                                  a.intersect_host(d[-100003:].cpu().numpy()).view(np.uint32))


def _slivers(n, rng):
    """Thin triangles along the diagonal of the unit cube: nearly every box
    of the tree spans the cube."""
    a, d = 0.02 * rng.random((n, 3)), 0.02 * rng.random((n, 3))
    return np.stack([a, 1.0 - d, a + 0.004 * rng.random((n, 3))], axis=1)


def _shells(n, rng):
    """Rings of small triangles around the x axis, in clusters of geometric
    spacing: a tree of many levels whose nodes' boxes all hold the axis."""
    c, s, i = np.meshgrid(np.arange(n), np.arange(8), np.arange(8), indexing="ij")
    x = 0.7 ** c
    a = 2.0 * np.pi * (i + 0.5) / 8
    x0, r = x - 0.27 * x * (s + 1) / 8, 0.3 * x
    def ring(dx, da):
        return np.stack([x0 + dx * x, r * np.cos(a + da), r * np.sin(a + da)], axis=-1)
    return np.stack([ring(0, 0), ring(0.006, 0), ring(0, 0.05)], axis=-2).reshape(-1, 3, 3)


@pytest.mark.parametrize("mode", [accel.ISECT_TRIACCEL, accel.ISECT_WATERTIGHT])
@pytest.mark.parametrize("make,size", [(_slivers, 70), (_slivers, 3000), (_slivers, 6000), (_shells, 9), (_shells, 90)])
def test_last_rays_in_deep_trees(gpu, make, size, mode):
    """The last rays of a wave in trees whose boxes overlap or nest over many
    levels, so that a ray has many nodes waiting at every level when all lanes
    take it over and most nodes it visits have several children hit.  Waves of
    8 rays, and of 64 of which 12 go through everything and the rest end early;
    bit-exact against the host walker."""
    import torch
    rng = np.random.default_rng(size)
    t = make(size, rng).astype(np.float32)
    v, f = t.reshape(-1, 3), np.arange(3 * len(t), dtype=np.uint32).reshape(-1, 3)
    a = accel.Accel(v, f, isect=mode)
    waves = 20 * torch.cuda.get_device_properties(gpu).multi_processor_count
    for per in (8, 64):
        n = per * waves
        rays = np.empty((n, 8), np.float32)
        if make is _slivers:
            m = rng.random((n, 1))
            rays[:, 0:3] = np.where(rng.random((n, 1)) < 0.5, m + 0.05 * (rng.random((n, 3)) - 0.5), rng.random((n, 3)))
            rays[:, 4:7] = 2.0 * rng.random((n, 3)) - 1.0
        else:
            rays[:, 0:3] = 0.0
            rays[:, 4] = 1.0
            rays[:, 5:7] = 0.3 * (rng.random((n, 2)) - 0.5)
        rays[:, 3] = 0.0
        rays[:, 7] = np.where(np.arange(n) % per < 12, 1e30, 0.3 * rng.random(n) ** 6)
        d = torch.from_numpy(rays).to(gpu)
        hg, ho, hh = a.intersect(d).cpu().numpy(), a.occluded(d).cpu().numpy(), a.intersect_host(rays)
        np.testing.assert_array_equal(hg.view(np.uint32), hh.view(np.uint32))
        np.testing.assert_array_equal(accel.hit_ids(ho) != accel.MISS, accel.hit_ids(hh) != accel.MISS)
    assert a.info()["stack_overflow"] == 0
