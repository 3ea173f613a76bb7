"""GPU parity of the wavefront renderer::pt against the CPU oracle.

* per-sample contributions from identical uniform tables: the same splat
  raster position, the same number of splats and C within 1e-4 relative for
  at least 99.99 % of the samples, and no sample beyond 1e-3 among those
  with the same splats (kernels and oracle share the FP32 sine, cosine and
  power of lmx_fmath.h and both round every operation as written, so the
  records agree bit for bit in practice);
* the same with Philox-generated uniforms (the generator itself is pinned
  in the CPU tests by the published Random123 known-answer vectors);
* a closed form: radiance inside an emitting, reflecting closed sphere;
* converged images: GPU and oracle renders of the Cornell box agree per
  pixel within 3 sigma.
"""
import numpy as np
import pytest

import orc
from lmx import render, scenes

pytestmark = pytest.mark.gpu


def _table(n, width, seed):
    rng = np.random.default_rng(seed)
    return rng.random((n, width), dtype=np.float32)


def _compare(gpu_s, cpu_s, rtol=1e-4, worst=1e-3):
    """per-sample records: raster x, y, C rgb, #splats.  Returns the mask of
    samples that agree within rtol; asserts the worst case among samples
    with the same splats."""
    g = gpu_s[:, :6]
    c = cpu_s
    same = (g[:, 5] == c[:, 5]) & np.all(g[:, 0:2] == c[:, 0:2], axis=1)
    rel = (np.abs(g[:, 2:5] - c[:, 2:5]) / np.maximum(np.abs(c[:, 2:5]), 1e-3)).max(axis=1)
    if same.any():
        assert rel[same].max() <= worst, f"worst relative error {rel[same].max():.3e}"
    return same & (rel <= rtol)


@pytest.mark.parametrize("raster_mode", [render.RASTER_STRATIFIED, render.RASTER_RANDOM])
def test_pt_per_sample_parity_uniform_table(gpu, raster_mode):
    import torch
    sc = scenes.cornell_box(64, 64)
    n = 64 * 64 * 16
    maxv = 9
    tab = _table(n, render.table_width(maxv), 7)
    rs = render.Scene(sc)
    film, stats, so = rs.render_pt(n, max_num_vertices=maxv, raster_mode=raster_mode,
                                   table=torch.from_numpy(tab).to(gpu), sample_out=True)
    g = so.cpu().numpy()
    c = orc.Scene(sc).pt_samples(0, n, max_num_vertices=maxv, raster_mode=raster_mode, table=tab)
    ok = _compare(g, c)
    assert (c[:, 5] > 0).sum() > 200                     # paths that reach the light
    assert ok.mean() >= 0.9999, f"{(~ok).sum()} of {n} samples differ"
    # the film is the sum of the per-sample splats, rescaled by W H / N
    f_cpu = orc.Scene(sc).film(c) * (64 * 64 / n)
    np.testing.assert_allclose(film.cpu().numpy(), f_cpu, rtol=2e-3, atol=2e-3)


@pytest.mark.parametrize("exponent", [20.0, 400.0])
def test_pt_per_sample_parity_phong(gpu, exponent):
    """Cornell box with normalized-Phong boxes, and the displaced-sphere mesh
    with smooth vertex normals (shading-normal correction in play)."""
    sc = scenes.cornell_box(64, 64, phong_boxes=exponent)
    n = 64 * 64 * 16
    _, _, so = render.Scene(sc).render_pt(n, max_num_vertices=9, seed=77, sample_out=True)
    c = orc.Scene(sc).pt_samples(0, n, max_num_vertices=9, seed=77)
    ok = _compare(so.cpu().numpy(), c)
    assert ok.mean() >= 0.9999, f"{(~ok).sum()} of {n} samples differ"


def test_pt_per_sample_parity_sphere_grid_small(gpu):
    sc = scenes.sphere_grid(96, 96, grid=3, subdiv=3, seed=3)
    n = 96 * 96 * 8
    _, _, so = render.Scene(sc).render_pt(n, max_num_vertices=17, rr_depth=3, seed=5, sample_out=True)
    c = orc.Scene(sc).pt_samples(0, n, max_num_vertices=17, rr_depth=3, seed=5)
    ok = _compare(so.cpu().numpy(), c)
    assert (c[:, 5] > 0).sum() > 100
    assert ok.mean() >= 0.9999, f"{(~ok).sum()} of {n} samples differ"


@pytest.mark.parametrize("rr_mode", [render.RR_FIXED, render.RR_THROUGHPUT])
def test_pt_per_sample_parity_philox(gpu, rr_mode):
    sc = scenes.cornell_box(64, 64)
    n = 64 * 64 * 16
    rs = render.Scene(sc)
    _, _, so = rs.render_pt(n, max_num_vertices=9, seed=1234, sample_out=True, rr_mode=rr_mode, rr_depth=2)
    c = orc.Scene(sc).pt_samples(0, n, max_num_vertices=9, seed=1234, rr_mode=rr_mode, rr_depth=2)
    ok = _compare(so.cpu().numpy(), c)
    assert ok.mean() >= 0.9999, f"{(~ok).sum()} of {n} samples differ"


@pytest.mark.parametrize("maxv,rr_depth", [(4, 1), (7, 3), (-1, 2)])
def test_pt_furnace_closed_form(gpu, maxv, rr_depth):
    rho, Le = 0.5, 1.0
    sc = scenes.furnace_sphere(albedo=rho, Le=Le, width=32, height=32)
    spp = 512
    n = 32 * 32 * spp
    rs = render.Scene(sc)
    film, stats, _ = rs.render_pt(n, max_num_vertices=maxv, rr_depth=rr_depth, seed=5)
    img = film.cpu().numpy()
    if maxv == -1:
        expect = Le / (1 - rho)
    else:
        expect = Le * sum(rho ** j for j in range(maxv - 1))
    # the pixel mean over 1024 pixels x 512 spp is within 1% of the closed form
    assert abs(img.mean() - expect) < 0.01 * expect, (img.mean(), expect)
    assert stats["rays"] > n


def test_pt_cornell_image_within_3_sigma(gpu):
    sc = scenes.cornell_box(32, 32)
    spp = 1024
    n = 32 * 32 * spp
    rs = render.Scene(sc)
    _, _, so = rs.render_pt(n, max_num_vertices=9, seed=99, sample_out=True)
    g = so.cpu().numpy()[:, 2:5].reshape(spp, 32 * 32, 3)       # stratified: sample i -> pixel i mod WH
    c = orc.Scene(sc).pt_samples(0, n, max_num_vertices=9, seed=4242)[:, 2:5].reshape(spp, 32 * 32, 3)
    mg, mc = g.mean(axis=0), c.mean(axis=0)
    sg, sc_ = g.var(axis=0, ddof=1) / spp, c.var(axis=0, ddof=1) / spp
    z = np.abs(mg - mc) / np.sqrt(sg + sc_ + 1e-12)
    lit = (mg + mc) > 0
    assert lit.mean() > 0.5
    assert (z[lit] <= 3.0).mean() > 0.99, (z[lit] > 3).mean()


def _compare_nee(g, c, rtol=1e-4):
    """(n, 16) records of renderer::ptdirect / ptmis: the pixel part (0-5)
    and the camera-vertex connection (8-13) must agree like _compare's."""
    ok = _compare(g[:, 0:8], c[:, 0:8], rtol)
    cam_g, cam_c = g[:, 13] > 0, c[:, 13] > 0
    same = cam_g == cam_c
    close = np.all(np.abs(g[:, 10:13] - c[:, 10:13]) <= rtol * np.maximum(np.abs(c[:, 10:13]), 1e-6), axis=1)
    ras = np.all(~cam_c[:, None] | (np.abs(g[:, 8:10] - c[:, 8:10]) <= 1e-5), axis=1)
    return ok & same & close & ras


@pytest.mark.parametrize("entry,mode", [("ptdirect", 1), ("ptmis", 2)])
@pytest.mark.parametrize("raster_mode", [render.RASTER_STRATIFIED, render.RASTER_RANDOM])
def test_nee_per_sample_parity_uniform_table(gpu, entry, mode, raster_mode):
    import torch
    sc = scenes.cornell_box(32, 32, phong_boxes=20.0)
    n, m = 32 * 32 * 16, 9
    tab = np.random.default_rng(21).random((n, render.table_width(m, nee=True)), dtype=np.float32)
    rs = render.Scene(sc)
    _, _, so = getattr(rs, "render_" + entry)(n, max_num_vertices=m, raster_mode=raster_mode,
                                              table=torch.from_numpy(tab).to(gpu), sample_out=True)
    c = orc.Scene(sc).nee_samples(0, n, mode, max_num_vertices=m, raster_mode=raster_mode, table=tab)
    assert (c[:, 5] > 0).sum() > 1000 and (c[:, 13] > 0).sum() > 10
    ok = _compare_nee(so.cpu().numpy(), c)
    assert ok.mean() > 0.998, f"{(~ok).sum()} of {n} samples differ"


@pytest.mark.parametrize("entry,mode", [("ptdirect", 1), ("ptmis", 2)])
def test_nee_per_sample_parity_philox(gpu, entry, mode):
    sc = scenes.cornell_box(64, 64)
    n = 64 * 64 * 8
    _, _, so = getattr(render.Scene(sc), "render_" + entry)(n, max_num_vertices=9, seed=77, sample_out=True,
                                                            rr_depth=2)
    c = orc.Scene(sc).nee_samples(0, n, mode, max_num_vertices=9, seed=77, rr_depth=2)
    ok = _compare_nee(so.cpu().numpy(), c)
    assert ok.mean() > 0.998, f"{(~ok).sum()} of {n} samples differ"


@pytest.mark.parametrize("entry", ["ptdirect", "ptmis"])
def test_nee_furnace_closed_form(gpu, entry):
    rho, Le, maxv = 0.5, 1.0, 6
    sc = scenes.furnace_sphere(albedo=rho, Le=Le, width=32, height=32)
    film, _, _ = getattr(render.Scene(sc), "render_" + entry)(32 * 32 * 256, max_num_vertices=maxv, rr_depth=2,
                                                              seed=9)
    expect = Le * sum(rho ** j for j in range(maxv - 1))
    assert abs(float(film.mean()) - expect) < 0.01 * expect


def test_nee_images_agree_with_pt(gpu):
    sc = scenes.cornell_box(32, 32)
    rs = render.Scene(sc)
    def batches(fn, k):
        a = np.stack([fn(s).cpu().numpy().astype(np.float64) for s in range(k)])
        return a.mean(0), a.std(0, ddof=1) / np.sqrt(k)
    mp, sp = batches(lambda s: rs.render_pt(32 * 32 * 4096, max_num_vertices=9, seed=50 + s)[0], 16)
    for entry in ("ptdirect", "ptmis"):
        mn, sn = batches(lambda s: getattr(rs, "render_" + entry)(32 * 32 * 256, max_num_vertices=9, seed=90 + s)[0], 16)
        z = np.abs(mn - mp) / np.sqrt(sn ** 2 + sp ** 2 + 1e-12)
        lit = (mn + mp) > 1e-3
        assert (z[lit] <= 3.0).mean() > 0.97, (entry, (z[lit] > 3).mean())
        assert abs(mn.mean() - mp.mean()) < 0.01 * mp.mean(), entry


@pytest.mark.parametrize("entry,mode", [("pt", 0), ("ptmis", 2)])
def test_ggx_per_sample_parity(gpu, entry, mode):
    """bsdf::cooktorrance (GGX) boxes: GPU and oracle per sample."""
    import torch
    sc = scenes.cornell_box(32, 32, ggx_boxes=0.3)
    n, m = 32 * 32 * 16, 9
    rs = render.Scene(sc)
    tab = np.random.default_rng(31).random((n, render.table_width(m, nee=mode > 0)), dtype=np.float32)
    _, _, so = getattr(rs, "render_" + entry)(n, max_num_vertices=m, table=torch.from_numpy(tab).to(gpu),
                                              sample_out=True)
    if mode == 0:
        c = orc.Scene(sc).pt_samples(0, n, max_num_vertices=m, table=tab)
        ok = _compare(so.cpu().numpy(), c)
    else:
        c = orc.Scene(sc).nee_samples(0, n, mode, max_num_vertices=m, table=tab)
        ok = _compare_nee(so.cpu().numpy(), c)
    assert ok.mean() >= 0.9999, f"{(~ok).sum()} of {n} samples differ"


@pytest.mark.parametrize("n,cap", [(1, 64), (63, 64), (1000, 64), (70001, 4096), (200000, 1 << 20)])
def test_ray_and_sample_counts(gpu, n, cap):
    """Queue counts kept on the device between iterations, at odd queue sizes
    and refills: inside a closed, scattering, emitting sphere without
    roulette every path has max_num_vertices - 1 segments (but the few that
    leave through an edge of the tessellation), every sample is started once,
    and the film holds each segment's emission."""
    sc = scenes.furnace_sphere(albedo=0.5, Le=1.0, subdiv=2, width=9, height=7)
    rs = render.Scene(sc)
    for seed in (1, 2):                       # the second render reuses the queues and the recorded graph
        film, st, _ = rs.render_pt(n, max_num_vertices=5, rr_depth=100, seed=seed, queue_capacity=cap)
        assert st["samples"] == n
        assert 4 * n * (1 - 1e-4) - 4 <= st["rays"] <= 4 * n
        got = float(film.double().mean())
        assert abs(got - (1 + 0.5 + 0.25 + 0.125)) <= 1e-4 + 4.0 / n * (st["rays"] < 4 * n)


def _split_cornell(ntri, **kw):
    """The Cornell box with its walls and boxes split at edge midpoints into ntri triangles."""
    sc = scenes.cornell_box(33, 21, **kw)
    tris, mat, verts = sc["tris"][:-2].tolist(), sc["tri_mat"][:-2].tolist(), sc["verts"].tolist()
    while len(tris) + 2 < ntri:
        (a, b, c), m = tris.pop(0), mat.pop(0)
        verts.append([(x + y) / 2 for x, y in zip(verts[b], verts[c])])
        k = len(verts) - 1
        tris += [[k, a, b], [k, c, a]]
        mat += [m, m]
    assert len(tris) + 2 == ntri
    return dict(sc, verts=np.array(verts, np.float32), lights=[(len(tris), 2)],
                tris=np.array(tris + sc["tris"][-2:].tolist(), np.uint32),
                tri_mat=np.array(mat + sc["tri_mat"][-2:].tolist(), np.uint32))


@pytest.mark.gpu
@pytest.mark.parametrize("ntri,n,cap,kw", [
    (36, 1, 0, {}), (36, 63, 0, {}), (36, 255, 64, dict(phong_boxes=20.0)), (36, 257, 0, dict(ggx_boxes=0.2)),
    (47, 100003, 0, {}), (48, 20001, 1000, dict(ggx_boxes=0.5)), (48, 700001, 0, {}), (49, 5000, 0, {})])
@pytest.mark.parametrize("entry", ["pt", "ptmis", "ptdirect"])
def test_few_triangles(gpu, entry, ntri, n, cap, kw):
    """Scenes small enough for one kernel per frame (48 triangles, and one
    more) against the queues, which a render binned by material always takes:
    the same rays and the same record of every sample, bit for bit."""
    rs = render.Scene(_split_cornell(ntri, **kw))
    for opts in (dict(max_num_vertices=-1, rr_depth=2), dict(max_num_vertices=-1, rr_prob=0.95), dict(max_num_vertices=2), dict(max_num_vertices=6, min_num_vertices=3),
                 dict(max_num_vertices=9, rr_depth=1, rr_mode=render.RR_THROUGHPUT, raster_mode=render.RASTER_STRATIFIED)):
        got = [getattr(rs, "render_" + entry)(n, seed=n + 1, sample_out=True, queue_capacity=cap, shade_order=order, **opts)
               for order in (render.SHADE_QUEUE, render.SHADE_BY_MATERIAL)]
        (fa, sa, ra), (fb, sb, rb) = got
        assert sa["rays"] == sb["rays"] and sa["samples"] == sb["samples"] == n
        assert np.array_equal(np.asarray(ra.cpu()).view(np.uint32), np.asarray(rb.cpu()).view(np.uint32))
        # the additions of a pixel in another order: FP32 sums of at most c terms of one sign
        c = 8.0 * (n / (33 * 21) + 30.0)
        assert float((fa - fb).abs().max()) <= c * 2.0 ** -24 * 2 * float(fb.abs().max())


@pytest.mark.gpu
@pytest.mark.parametrize("ntri", [1, 2, 4])
@pytest.mark.parametrize("entry", ["pt", "ptmis", "ptdirect"])
def test_fewest_triangles(gpu, entry, ntri):
    """A light of one triangle or two facing the camera, and one over a
    floor, against the queues: the same rays and records, bit for bit."""
    sc = scenes.cornell_box(31, 17)
    quad = [[-1, -0.4, 0], [1, -0.4, 0], [1, 0.9, 0.1], [-1, 0.9, 0.1]]
    floor = [[-2, -0.5, 2], [2, -0.5, 2], [2, -0.5, -2], [-2, -0.5, -2]]
    tris, mat = [[0, 1, 2], [0, 2, 3], [4, 5, 6], [4, 6, 7]], [3, 3, 0, 0]
    rs = render.Scene(dict(sc, verts=np.array(quad + floor, np.float32), tris=np.array(tris[:ntri], np.uint32),
                           tri_mat=np.array(mat[:ntri], np.uint32), lights=[(0, min(ntri, 2))]))
    n = 20011
    for opts in (dict(max_num_vertices=-1, rr_depth=1), dict(max_num_vertices=2), dict(max_num_vertices=5)):
        (fa, sa, ra), (fb, sb, rb) = [
            getattr(rs, "render_" + entry)(n, seed=7, sample_out=True, shade_order=order, **opts)
            for order in (render.SHADE_QUEUE, render.SHADE_BY_MATERIAL)]
        assert sa["rays"] == sb["rays"] >= n and sa["samples"] == n
        assert entry == "ptdirect" or float(fa.max()) > 1.0
        assert np.array_equal(np.asarray(ra.cpu()).view(np.uint32), np.asarray(rb.cpu()).view(np.uint32))
        # FP32 sums of a pixel's terms of one sign in another order
        assert float((fa - fb).abs().max()) <= 8.0 * (n / (31 * 17) + 30.0) * 2.0 ** -24 * 2 * float(fb.abs().max())


@pytest.mark.gpu
def test_few_triangles_beyond_one_launch(gpu):
    """More samples than a path tracer's frame usually has (2^26): every one is counted and splat once."""
    rs = render.Scene(_split_cornell(36))
    n = (1 << 26) + 7
    (fa, sa, _), (fb, sb, _) = [rs.render_pt(n, seed=3, max_num_vertices=2, shade_order=order)
                                for order in (render.SHADE_QUEUE, render.SHADE_BY_MATERIAL)]
    assert sa["rays"] == sb["rays"] == n and sa["samples"] == sb["samples"] == n
    # FP32 sums of n / (33 21) terms of one sign in another order, both rounded
    assert float((fa - fb).abs().max()) <= 2 * 1.1 * n / (33 * 21) * 2.0 ** -24 * float(fb.abs().max())


@pytest.mark.gpu
@pytest.mark.parametrize("cap,n", [(64, 5000), (256, 1200), (600, 20000)])
@pytest.mark.parametrize("entry", ["pt", "ptmis", "ptdirect"])
def test_few_triangles_long_paths(gpu, entry, cap, n):
    """Paths of 1,023 segments in a closed scene of few triangles, more of
    them than a launch may start (4,096 segments a wave, four waves to each
    256 paths in flight): several launches, the samples of each workgroup
    continued where the last one stopped, and the frame of the queues."""
    rs = render.Scene(scenes.furnace_sphere(albedo=0.9, Le=1.0, subdiv=0, width=16, height=12))
    opts = dict(max_num_vertices=1024, rr_depth=2000, seed=9, sample_out=True)
    fa, sa, ra = getattr(rs, "render_" + entry)(n, queue_capacity=cap, **opts)
    fb, sb, rb = getattr(rs, "render_" + entry)(n, queue_capacity=1 << 15, shade_order=render.SHADE_BY_MATERIAL, **opts)
    lanes = (cap + 255) // 256 * 256
    steps = n * 1023.0 / lanes                 # of a wave, if its lanes never idle
    assert steps / (4096 + 1023) * 0.9 <= sa["iterations"] <= steps / 4096 * 1.5 + 2
    assert sa["rays"] == sb["rays"] > 1000 * n and sa["samples"] == sb["samples"] == n
    assert np.array_equal(np.asarray(ra.cpu()).view(np.uint32), np.asarray(rb.cpu()).view(np.uint32))
    # FP32 sums of at most 1,023 segments and as many connections of every sample of a pixel, in another order
    c = 2 * 1024.0 * (n / (16 * 12) + 1)
    assert float((fa - fb).abs().max()) <= c * 2.0 ** -24 * float(fb.abs().max())
