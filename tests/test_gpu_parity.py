"""GPU parity tests: librgx (through the C ABI / the autograd op) against the CPU oracle.

Gates: per-segment hit sets bit-exact; first-hit t bit-exact; forward image <= 1e-4 max abs;
gradients cosine >= 0.9999 and relative L2 <= 1e-3 per parameter tensor; integer work
(Morton codes, permutations) bit-exact.
"""
import numpy as np
import pytest
import torch

from raygaussx_amd import scenes

pytestmark = pytest.mark.gpu

IMG_TOL = 1e-4
COS_MIN = 0.9999
REL_MAX = 1e-3


@pytest.fixture(scope="module")
def gx():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import gpu_common
    from raygaussx_amd import _lib
    _lib.lib()          # a missing librgx.so is an error, not a skip
    return gpu_common


@pytest.fixture(scope="module")
def c0():
    return scenes.scene_to_numpy(scenes.make_scene(0)), scenes.make_camera(0), scenes.CONFIGS[0]


def _step(msg):
    print(f"[gpu-step] {msg}", flush=True)


def test_aabb_and_scene_bbox_bit_exact(gx, orc, c0):
    from raygaussx_amd import optix_utils as u_ox
    sc, _, _ = c0
    _step("aabb n=4096")
    d = gx.to_dev(sc)
    boxes, bmin, bmax = u_ox.ellipsoids_bbox_from_quat(d["quaternions"], d["positions"], d["scales"], d["densities"])
    oboxes, obmin, obmax = orc.aabb(sc["positions"], sc["scales"], sc["quaternions"], sc["densities"])
    np.testing.assert_array_equal(boxes.cpu().numpy(), oboxes)
    np.testing.assert_array_equal(bmin.cpu().numpy(), obmin)
    np.testing.assert_array_equal(bmax.cpu().numpy(), obmax)


def test_sh_colour_and_gradient(gx, orc):
    from raygaussx_amd.render_optix import compute_rgb, compute_sh_grad
    rng = np.random.default_rng(0)
    for degree, G in ((0, 0), (1, 2), (2, 0), (3, 7), (3, 0)):
        _step(f"sh degree={degree} G={G}")
        n, K = 1000, (degree + 1) ** 2
        pos = rng.normal(size=(n, 3)).astype(np.float32)
        eye = np.array([0.5, 3.0, -1.0], np.float32)
        sh = rng.normal(size=(n, 3, K)).astype(np.float32)
        sg = rng.normal(size=(n, 3, G)).astype(np.float32)
        sharp = rng.uniform(0.5, 4, size=(n, G)).astype(np.float32)
        axis = rng.normal(size=(n, G, 3)).astype(np.float32)
        drgb = rng.normal(size=(n, 3)).astype(np.float32)
        drgb[11] = 0
        t = [torch.from_numpy(a).to(gx.DEV) for a in (pos, sh, sg, sharp, axis, drgb)]
        rgb = compute_rgb(eye, t[0], t[1], t[2], t[3], t[4], G, degree).cpu().numpy()
        kw = dict(sg=sg, sharp=sharp, axis=axis) if G else {}
        np.testing.assert_allclose(rgb, orc.sh_forward(eye, pos, sh, **kw), atol=2e-5, rtol=2e-5)
        dsh, dpos, dsg, dsharp, daxis = compute_sh_grad(eye, t[0], t[1], t[2], t[3], t[4], G, degree, t[5])
        o = orc.sh_backward(eye, pos, sh, drgb, **kw)
        np.testing.assert_allclose(dsh.cpu().numpy().reshape(n, 3, K), o[0], atol=2e-5, rtol=2e-5)
        np.testing.assert_allclose(dpos.cpu().numpy(), o[1], atol=2e-5, rtol=1e-4)
        if G:
            np.testing.assert_allclose(dsg.cpu().numpy().reshape(n, 3, G), o[2], atol=2e-5, rtol=1e-4)
            np.testing.assert_allclose(dsharp.cpu().numpy().reshape(n, G), o[3], atol=2e-5, rtol=1e-4)
            np.testing.assert_allclose(daxis.cpu().numpy().reshape(n, G, 3), o[4], atol=2e-5, rtol=1e-4)
        if degree == 3 and G == 0:
            # coefficients that do not start on a 16-byte boundary take the kernels without the staged rows: same values
            off = torch.empty(n * 3 * K + 1, device=gx.DEV)[1:].view(n, 3, K)
            off.copy_(t[1])
            assert off.data_ptr() % 16 == 4 and off.is_contiguous()
            np.testing.assert_array_equal(compute_rgb(eye, t[0], off, t[2], t[3], t[4], G, degree).cpu().numpy(), rgb)
            dsh2, dpos2 = compute_sh_grad(eye, t[0], off, t[2], t[3], t[4], G, degree, t[5])[:2]
            np.testing.assert_array_equal(dsh2.cpu().numpy(), dsh.cpu().numpy())
            np.testing.assert_array_equal(dpos2.cpu().numpy(), dpos.cpu().numpy())


def _built(gx, sc, eye, rgb=None):
    from raygaussx_amd import optix_utils as u_ox
    d = gx.to_dev(sc)
    n = d["positions"].shape[0]
    gas = u_ox.AccelerationStructure(n, gx.DEV).build_from_gaussians(d["positions"], d["scales"], d["quaternions"],
                                                                      d["densities"])
    rgb_t = torch.zeros(n, 3, device=gx.DEV) if rgb is None else torch.from_numpy(rgb).to(gx.DEV)
    prims_sorted = u_ox.pack_prims(gas, eye, d["positions"], d["scales"], d["quaternions"], d["densities"], rgb_t)
    prims_input = u_ox.pack_prims(None, eye, d["positions"], d["scales"], d["quaternions"], d["densities"], rgb_t)
    return gas, prims_sorted, prims_input


def test_build_permutation_bbox_and_packing_bit_exact(gx, orc, c0):
    sc, cam, _ = c0
    eye = cam.camera_center.numpy()
    rgb = np.random.default_rng(1).random((4096, 3), dtype=np.float32)
    _step("build + pack n=4096")
    gas, ps, pi = _built(gx, sc, eye, rgb)
    order = gas.order().cpu().numpy()
    assert sorted(order.tolist()) == list(range(4096))
    _, obmin, obmax = orc.aabb(sc["positions"], sc["scales"], sc["quaternions"], sc["densities"])
    bmin, bmax = gas.scene_bbox()
    np.testing.assert_array_equal(np.array(bmin, np.float32), obmin)
    np.testing.assert_array_equal(np.array(bmax, np.float32), obmax)
    oprims = orc.pack_prims(eye, sc["positions"], sc["scales"], sc["quaternions"], sc["densities"], rgb)
    got = pi.cpu().numpy()
    np.testing.assert_array_equal(got.view(np.uint32), oprims.view(np.uint32))      # bit-exact incl. NaN k
    np.testing.assert_array_equal(ps.cpu().numpy().view(np.uint32), oprims[order].view(np.uint32))
    for n in (1, 2, 3, 65, 2049):       # ragged sizes around the sort tile and wave sizes
        _step(f"build n={n}")
        sub = {k: v[:n] for k, v in sc.items()}
        gas_n, _, _ = _built(gx, sub, eye)
        assert sorted(gas_n.order().cpu().numpy().tolist()) == list(range(n))


def test_queries_on_given_segments_bit_exact(gx, orc, c0):
    """first-hit t and collect hit sets on identical primitives and segments: exact equality."""
    from raygaussx_amd import optix_utils as u_ox
    sc, cam, _ = c0
    sc = dict(sc)
    sc["scales"] = sc["scales"] * 2.0
    eye = cam.camera_center.numpy()
    gas, ps, pi = _built(gx, sc, eye)
    cs = orc.camera_struct(cam)
    rng = np.random.default_rng(3)
    rays = rng.choice(128 * 128, 3000, replace=False)
    dirs = orc.ray_dirs(cs, rays)
    tlo = rng.uniform(2.0, 5.0, 3000).astype(np.float32)
    thi = (tlo + rng.uniform(0.01, 1.5, 3000)).astype(np.float32)
    oprims = pi.cpu().numpy()
    _step("first_hit 3000 segments")
    t_gpu = u_ox.first_hit(gas, ps, eye, *[torch.from_numpy(a).to(gx.DEV) for a in (dirs, tlo, thi)]).cpu().numpy()
    t_cpu = orc.first_hit(oprims, dirs, tlo, thi)
    np.testing.assert_array_equal(t_gpu, t_cpu)
    assert (t_cpu >= 0).sum() > 500
    _step("trace_segments 3000 segments")
    cap = 256
    c_gpu, i_gpu = u_ox.trace_segments(gas, ps, eye, *[torch.from_numpy(a).to(gx.DEV) for a in (dirs, tlo, thi)], cap)
    c_gpu, i_gpu = c_gpu.cpu().numpy(), i_gpu.cpu().numpy()
    c_cpu, i_cpu = orc.trace_segments(oprims, dirs, tlo, thi, cap)
    np.testing.assert_array_equal(c_gpu, c_cpu)
    assert c_cpu.max() > 32          # some lists overflow the LDS part into the spill area
    for r in range(3000):
        assert sorted(i_gpu[r, :c_gpu[r]].tolist()) == i_cpu[r, :c_cpu[r]].tolist(), r
    # truncation at cap is reported the same way
    c_small, _ = u_ox.trace_segments(gas, ps, eye, *[torch.from_numpy(a).to(gx.DEV) for a in (dirs, tlo, thi)], 4)
    c_small_cpu, _ = orc.trace_segments(oprims, dirs, tlo, thi, 4)
    np.testing.assert_array_equal(c_small.cpu().numpy(), c_small_cpu)


def test_forward_config0_image_and_hit_sets(gx, orc, c0):
    sc, cam, cfg = c0
    _step("forward config0")
    out = gx.gpu_render(sc, cam, cfg)
    img, st, ctx = orc.render_forward(sc, cam, cfg["dt_step"], cfg["dynamic_sampling"], cfg["max_prim_slice"])
    assert np.abs(out["image"] - img).max() <= IMG_TOL
    for k in ("hit_pairs", "slabs", "empty_slabs", "overflow_rays", "rays_hit"):
        assert out["stats_fwd"][k] == st[k], k
    # slab-by-slab hit sets of a ray subset, on the slabs the oracle marched
    from raygaussx_amd import optix_utils as u_ox
    settings = out["settings"]
    rays = np.arange(0, 128 * 128, 61)
    dirs_all, tlo, thi, want = [], [], [], []
    for r in rays:
        slabs, _ = orc.march_trace(ctx["cs"], ctx["ms"], ctx["bmin"], ctx["bmax"], ctx["prims"], int(r))
        d = orc.ray_dirs(ctx["cs"], [r])[0]
        for tb, dt, lo, hi, ids in slabs:
            dirs_all.append(d); tlo.append(lo); thi.append(hi); want.append(sorted(ids.tolist()))
    dirs_all = np.asarray(dirs_all, np.float32)
    d = gx.to_dev(sc)
    rgb = torch.from_numpy(ctx["rgb"]).to(gx.DEV)
    ps = u_ox.pack_prims(settings.gas, ctx["eye"], d["positions"], d["scales"], d["quaternions"], d["densities"], rgb)
    _step(f"hit sets of {len(want)} slabs")
    cnt, ids = u_ox.trace_segments(settings.gas, ps, ctx["eye"], torch.from_numpy(dirs_all).to(gx.DEV),
                                   torch.tensor(tlo, dtype=torch.float32, device=gx.DEV),
                                   torch.tensor(thi, dtype=torch.float32, device=gx.DEV), 64)
    cnt, ids = cnt.cpu().numpy(), ids.cpu().numpy()
    assert len(want) > 1000
    for s in range(len(want)):
        assert sorted(ids[s, :cnt[s]].tolist()) == want[s], s


def test_config0_against_committed_golden_vectors(gx, orc, c0):
    """The same configuration-0 results the oracle produced when tests/golden/config0.npz was
    written: image, march counters, gradients, per-slab hit sets and first-hit distances."""
    import os
    import sys
    from raygaussx_amd import optix_utils as u_ox
    from raygaussx_amd.render_optix import compute_rgb
    here = os.path.dirname(os.path.abspath(__file__))
    sys.path.insert(0, os.path.join(here, "golden"))
    import make_golden
    g = np.load(os.path.join(here, "golden", "config0.npz"))
    _, cam, cfg = c0
    sc = make_golden.scene_of(g)
    _step("golden: forward + backward config0")
    out = gx.gpu_render(sc, cam, cfg, want_grad=make_golden.mse_dloss(g["image"]))
    assert np.abs(out["image"] - g["image"]).max() <= IMG_TOL
    for k in ("hit_pairs", "slabs", "empty_slabs", "rays_hit"):
        assert out["stats_fwd"][k] == int(g["stats_" + k]), k
    _check_grads(gx, out["grads"], {k[2:]: g[k] for k in g.files if k.startswith("d_")})
    # the two ray queries on the stored segments
    d = gx.to_dev(sc)
    eye = cam.camera_center.numpy()
    gas = out["settings"].gas
    rgb = compute_rgb(cam.camera_center, d["positions"], d["color_features"], None, None, None, 0, 3)
    ps = u_ox.pack_prims(gas, eye, d["positions"], d["scales"], d["quaternions"], d["densities"], rgb)

    def dirs_of(rays):   # computeRay on the host (fp32, no contraction), as the kernels evaluate it
        return orc.ray_dirs(orc.camera_struct(cam), rays)
    _step("golden: hit sets")
    dv = lambda a, t=torch.float32: torch.from_numpy(np.ascontiguousarray(a)).to(gx.DEV, t)
    cnt, ids = u_ox.trace_segments(gas, ps, eye, dv(dirs_of(g["seg_ray"])), dv(g["seg_lo"]), dv(g["seg_hi"]), 64)
    cnt, ids = cnt.cpu().numpy(), ids.cpu().numpy()
    off = g["seg_off"]
    np.testing.assert_array_equal(cnt, np.diff(off))
    for s in range(len(cnt)):
        assert sorted(ids[s, :cnt[s]].tolist()) == g["seg_ids"][off[s]:off[s + 1]].tolist(), s
    _step("golden: first hits")
    t = u_ox.first_hit(gas, ps, eye, dv(dirs_of(g["fh_ray"])), dv(g["fh_lo"]), dv(g["fh_hi"])).cpu().numpy()
    np.testing.assert_array_equal(t, g["fh_t"])


def test_tile_cooperative_collect_hit_sets_bit_exact(gx, orc, c0):
    """The collect query as the march kernels run it (one 8x8 tile per wavefront, shared candidate
    gather, per-ray exact predicate) on the oracle's own slab intervals: identical hit sets."""
    from raygaussx_amd import optix_utils as u_ox
    sc, cam, cfg = c0
    img, st, ctx = orc.render_forward(sc, cam, cfg["dt_step"], cfg["dynamic_sampling"], cfg["max_prim_slice"])
    d = gx.to_dev(sc)
    gas = u_ox.AccelerationStructure(4096, gx.DEV).build_from_gaussians(d["positions"], d["scales"], d["quaternions"],
                                                                         d["densities"])
    ps = u_ox.pack_prims(gas, ctx["eye"], d["positions"], d["scales"], d["quaternions"], d["densities"],
                         torch.from_numpy(ctx["rgb"]).to(gx.DEV))
    R = 128 * 128
    traces = [orc.march_trace(ctx["cs"], ctx["ms"], ctx["bmin"], ctx["bmax"], ctx["prims"], r)[0] for r in range(R)]
    cams = u_ox.camera_struct(cam)
    checked = 0
    # uncounted: the filter without counters, as in the kernels launched without a statistics block
    for rank, uncounted in ((0, False), (0, True), (1, True), (4, False), (4, True), (9, True)):
        tlo = np.ones(R, np.float32)
        thi = np.zeros(R, np.float32)          # thi < tlo: pixel idle
        for r in range(R):
            if len(traces[r]) > rank:
                tlo[r], thi[r] = traces[r][rank][2], traces[r][rank][3]
        _step(f"collect_tiles slab rank {rank}, uncounted {uncounted}")
        cnt, ids = u_ox.collect_tiles(gas, cams, ps, torch.from_numpy(tlo).to(gx.DEV), torch.from_numpy(thi).to(gx.DEV), 64,
                                      uncounted=uncounted)
        cnt, ids = cnt.cpu().numpy(), ids.cpu().numpy()
        for r in range(R):
            want = sorted(traces[r][rank][4].tolist()) if len(traces[r]) > rank else []
            assert sorted(ids[r, :cnt[r]].tolist()) == want, (rank, r)
            checked += len(want)
    assert checked > 30000
    # the max_prim_slice cut is reported per ray
    tlo = np.full(R, 3.0, np.float32)
    thi = np.full(R, 5.0, np.float32)
    dirs = orc.ray_dirs(ctx["cs"])
    c_cpu, _ = orc.trace_segments(ctx["prims"], dirs, tlo, thi, 3)
    for uncounted in (False, True):
        cnt, _ = u_ox.collect_tiles(gas, cams, ps, torch.from_numpy(tlo).to(gx.DEV), torch.from_numpy(thi).to(gx.DEV), 3,
                                    uncounted=uncounted)
        np.testing.assert_array_equal(cnt.cpu().numpy(), c_cpu)


@pytest.mark.parametrize("thin,spread", [(0.02, 0.5), (1e-3, 0.5), (2e-5, 0.5), (2e-8, 0.5), (0.3, 1.0)])
def test_hit_sets_of_segments_that_end_at_a_surface(gx, orc, thin, spread):
    """Segments that end exactly at a Gaussian's entry, one ulp before it and one after: the filter's shortcut must leave
    these to the exact roots.  Gaussians as thin as ``thin`` along one axis, some 10 to 10^8 of their radii away (from
    2e-5 on beyond the range of the shortcut, at 2e-8 of the plain division too), and around the eye."""
    from raygaussx_amd import optix_utils as u_ox
    cam = scenes.make_camera(0, 0, width=40, height=24)
    sc = scenes.scene_to_numpy(scenes.make_scene(0, n=500, seed=77))
    rng = np.random.default_rng(5)
    eye = cam.camera_center.numpy()
    if spread == 1.0:      # the eye among them
        sc["positions"] = (eye + rng.normal(size=(500, 3))).astype(np.float32)
    else:
        sc["positions"] = (sc["positions"] * spread).astype(np.float32)
    sc["scales"] = rng.uniform(0.05, 0.2, (500, 3)).astype(np.float32)
    sc["scales"][:, 1] = thin * rng.uniform(0.5, 1.5, 500).astype(np.float32)
    rgb = np.ones((500, 3), np.float32)
    d = gx.to_dev(sc)
    prims = orc.pack_prims(eye, sc["positions"], sc["scales"], sc["quaternions"], sc["densities"], rgb)
    gas = u_ox.AccelerationStructure(500, gx.DEV).build_from_gaussians(d["positions"], d["scales"], d["quaternions"], d["densities"])
    ps = u_ox.pack_prims(gas, eye, d["positions"], d["scales"], d["quaternions"], d["densities"], torch.from_numpy(rgb).to(gx.DEV))
    dirs = orc.ray_dirs(orc.camera_struct(cam))
    R = len(dirs)
    start = rng.uniform(0, 4, R).astype(np.float32) if spread == 1.0 else rng.uniform(0, 2, R).astype(np.float32)
    t = orc.first_hit(prims, dirs, start, np.full(R, 100.0, np.float32))
    hit = t > start      # (a ray that starts inside reports its start)
    assert hit.sum() > (R // 20 if spread == 1.0 else R // 4)
    t = np.where(hit, t, start + np.float32(1.0)).astype(np.float32)
    dv = lambda a: torch.from_numpy(np.ascontiguousarray(a, np.float32)).to(gx.DEV)
    for cap in (512, 2):
        for thi in (t, np.nextafter(t, np.float32(0)), np.nextafter(t, np.float32(1e9))):
            tlo = np.maximum(start, thi - np.float32(0.3)).astype(np.float32)
            want_n, want = orc.trace_segments(prims, dirs, tlo, thi, cap)
            for uncounted in (False, True):
                _step(f"segments ending at a surface, thin {thin}, cap {cap}, uncounted {uncounted}")
                n, ids = u_ox.collect_tiles(gas, u_ox.camera_struct(cam), ps, dv(tlo), dv(thi), cap, uncounted=uncounted)
                n, ids = n.cpu().numpy(), ids.cpu().numpy()
                np.testing.assert_array_equal(n, want_n)
                if cap == 512:
                    np.testing.assert_array_equal(np.sort(np.where(ids < 0, 1 << 30, ids), 1), np.sort(np.where(want < 0, 1 << 30, want), 1))


def _check_grads(gx, got, want, keys=("positions", "scales", "quaternions", "densities", "color_features")):
    for k in keys:
        cos, rel = gx.cos_rel(got[k], want[k])
        assert cos >= COS_MIN and rel <= REL_MAX, (k, cos, rel)


def test_backward_config0_gradients(gx, orc, c0):
    sc, cam, cfg = c0
    img, st, ctx = orc.render_forward(sc, cam, cfg["dt_step"], cfg["dynamic_sampling"], cfg["max_prim_slice"])
    target = np.random.default_rng(7).random(img.shape, dtype=np.float32)
    dloss = (2.0 * (img - target) / img.size).astype(np.float32)      # d MSE / d image
    og, ost = orc.render_backward(sc, ctx, img, dloss)
    _step("forward+backward config0")
    out = gx.gpu_render(sc, cam, cfg, want_grad=dloss)
    _check_grads(gx, out["grads"], og)
    assert out["stats_bwd"]["hit_pairs"] == ost["hit_pairs"]
    for k in ("sph_gauss_features", "bandwidth_sharpness", "lobe_axis"):
        assert out["grads"][k] is None
    # the kernels a training loop runs (no statistics block: no counters), with each kind of record
    for label, kw in (("default record", {}), ("hit lists only", dict(rec_tile_words=16384)), ("no record", dict(record_hits=False))):
        _step("forward+backward config0, uncounted kernels, " + label)
        out = gx.gpu_render(sc, cam, cfg, want_grad=dloss, stats=False, **kw)
        assert np.abs(out["image"] - img).max() <= IMG_TOL
        _check_grads(gx, out["grads"], og)


def test_backward_replay_of_recorded_hit_lists_equals_recomputation(gx, orc):
    """The backward fed with the forward's record (hit lists, and the per-sample density and colour
    sums when the record has room for them) must give what the backward that searches the tree
    again gives (same hits, same order; only summation orders may differ), also when some tiles'
    records overflow and fall back to recomputation, when the pool of sample sums runs out, and
    with the adaptive step and candidate sets that need several table batches."""
    for label, config, scale, dyn, words in (("fixed step", 0, 3.0, False, None), ("adaptive step", 2, 3.0, True, None),
                                             ("hit lists only, no sample sums", 0, 3.0, False, 16384),
                                             ("sample-sum pool runs out: some tiles with sums, some without", 0, 3.0, False, 16384 + 3 * 8192),
                                             ("fat Gaussians, small records", 0, 8.0, False, 1024)):
        sc = scenes.scene_to_numpy(scenes.make_scene(config, n=5000, sh_degree=1, seed=21))
        sc["scales"] = sc["scales"] * scale
        cam = scenes.make_camera(config, 1, width=52, height=44)
        cfg = dict(dt_step=0.004, dynamic_sampling=dyn, max_prim_slice=4096)
        dloss = np.random.default_rng(3).normal(size=(52 * 44, 3)).astype(np.float32)
        _step("replay vs recompute: " + label)
        a = gx.gpu_render(sc, cam, cfg, want_grad=dloss, record_hits=False)
        b = gx.gpu_render(sc, cam, cfg, want_grad=dloss, record_hits=True, rec_tile_words=words)
        # the recording forward and the plain one may add a ray's Gaussians in different orders
        assert np.abs(a["image"] - b["image"]).max() <= 2e-6
        for k in ("slabs", "empty_slabs", "overflow_rays", "rays_hit"):
            assert a["stats_fwd"][k] == b["stats_fwd"][k], k
        assert a["stats_fwd"]["hit_pairs"] == b["stats_fwd"]["hit_pairs"]
        assert a["stats_bwd"]["hit_pairs"] == b["stats_bwd"]["hit_pairs"] > 10000
        assert a["stats_bwd"]["slabs"] == b["stats_bwd"]["slabs"]
        # gradient scatter: 14 adds per Gaussian and window when replaying, per Gaussian, slab and pixel row otherwise
        assert a["stats_fwd"]["grad_atomics"] == b["stats_fwd"]["grad_atomics"] == 0
        assert 0 < b["stats_bwd"]["grad_atomics"] <= a["stats_bwd"]["grad_atomics"]
        assert a["stats_bwd"]["grad_atomics"] % 14 == b["stats_bwd"]["grad_atomics"] % 14 == 0
        if words is None or words >= 16384:   # everything replayed: the backward fetched no tree node
            assert b["stats_bwd"]["nodes_visited"] == 0
        else:               # some tiles replayed, some recomputed
            print("nodes", b["stats_bwd"]["nodes_visited"], a["stats_bwd"]["nodes_visited"], flush=True)
            assert 0 < b["stats_bwd"]["nodes_visited"] <= a["stats_bwd"]["nodes_visited"]
        for k in ("positions", "scales", "quaternions", "densities", "color_features"):
            cos, rel = gx.cos_rel(b["grads"][k], a["grads"][k])
            assert cos >= 1 - 1e-9 and rel <= 2e-5, (label, k, cos, rel)


def test_backward_ignores_a_record_of_another_launch(gx):
    """A record names the launch it belongs to; handed the record of another scene (or step), the
    backward searches the tree for every tile, as without a record, instead of replaying it."""
    from raygaussx_amd import optix_utils as u_ox
    from raygaussx_amd.render_optix import compute_rgb
    cam = scenes.make_camera(0, 0, width=40, height=32)
    cs = u_ox.camera_struct(cam)
    dloss = torch.from_numpy(np.random.default_rng(1).normal(size=(40 * 32, 3)).astype(np.float32)).to(gx.DEV)

    def launch(n, seed, dt, records_from=None):
        sc = gx.to_dev(scenes.scene_to_numpy(scenes.make_scene(0, n=n, sh_degree=0, seed=seed)))
        gas = u_ox.AccelerationStructure(n, gx.DEV).build_from_gaussians(sc["positions"], sc["scales"] * 1.5,
                                                                          sc["quaternions"], sc["densities"])
        rgb = compute_rgb(cam.camera_center, sc["positions"], sc["color_features"], None, None, None, 0, 0)
        ps = u_ox.pack_prims(gas, cs, sc["positions"], sc["scales"] * 1.5, sc["quaternions"], sc["densities"], rgb)
        rec = u_ox.new_records(cs, gx.DEV)
        img = u_ox.march_forward(gas, cs, ps, dt, False, 512, True, records=rec)
        stats = u_ox.new_stats(gx.DEV)
        grads = u_ox.march_backward(gas, cs, ps, img, dloss, dt, False, 512, True, stats=stats,
                                    records=rec if records_from is None else records_from)
        return rec, [g.cpu().numpy() for g in grads], u_ox.read_stats(stats)

    _step("backward with its own record")
    rec_a, own, st_own = launch(3000, 5, 0.004)
    assert st_own["nodes_visited"] == 0 and st_own["hit_pairs"] > 10000
    for label, n, seed, dt in (("another scene", 2500, 6, 0.004), ("another step", 3000, 5, 0.005)):
        _step("backward with the record of " + label)
        _, ref, st_ref = launch(n, seed, dt)                       # its own record: the expected gradients
        _, got, st = launch(n, seed, dt, records_from=rec_a)       # the foreign one
        assert st["nodes_visited"] > 0 and st["replay_lost"] == 0 and st["hit_pairs"] == st_ref["hit_pairs"]
        for g, r in zip(got, ref):
            cos, rel = gx.cos_rel(g, r)
            assert cos >= 1 - 1e-6 and rel <= 1e-4


def test_dynamic_sampling_lobes_supersampling_black_background(gx, orc):
    """The unbounded-scene settings (adaptive step, camera inside the cloud) with spherical-Gaussian
    lobes, a non-multiple-of-8 image, 2x1 supersampling and a black background."""
    rng = np.random.default_rng(5)
    sc = scenes.scene_to_numpy(scenes.make_scene(2, n=6000, sh_degree=2, seed=77))
    n, G = 6000, 3
    sc["sph_gauss_features"] = rng.normal(size=(n, 3, G)).astype(np.float32) * 0.1
    sc["bandwidth_sharpness"] = rng.uniform(0.5, 3, size=(n, G)).astype(np.float32)
    ax = rng.normal(size=(n, G, 3)).astype(np.float32)
    sc["lobe_axis"] = ax / np.linalg.norm(ax, axis=2, keepdims=True)
    sc["scales"] = sc["scales"] * 3.0
    cam = scenes.make_camera(2, 5, width=45, height=31)
    cfg = dict(dt_step=0.005, dynamic_sampling=True, max_prim_slice=512, t_eps=1e-3)
    img, st, ctx = orc.render_forward(sc, cam, 0.005, True, 512, white_background=False, supersampling=(2, 1))
    dloss = rng.normal(size=img.shape).astype(np.float32)
    _step("dynamic sampling + lobes + supersampling")
    out = gx.gpu_render(sc, cam, cfg, white=False, supersampling=(2, 1), want_grad=dloss)
    assert out["image"].shape == (90 * 31, 3)
    assert st["hit_pairs"] > 50000
    # The adaptive step feeds exp / cbrt roundings back into sample positions.  Ray by ray (see
    # gpu_common.comparable_rays): rays that blended other slabs than on the CPU, or on which the
    # oracle itself jumps when its step moves by a few ulp, are set aside, counted and bounded; every
    # other ray must meet the image gate, and the gradient of a loss restricted to them the gradient gates.
    _, counts = gx.gpu_forward_counts(sc, cam, cfg, white=False, supersampling=(2, 1))
    same, n_rephased, n_edge = gx.comparable_rays(orc, ctx, img, counts)
    err = np.abs(out["image"] - img).max(1)
    print(f"of {same.size} rays: {n_rephased} re-phased, {n_edge} on a cut-off edge; image max err on the others {err[same].max():.2e}, "
          f"on them {err[~same].max() if (~same).any() else 0.0:.2e}", flush=True)
    assert err[same].max() <= IMG_TOL                     # every comparable ray meets the gate
    assert (err > IMG_TOL).sum() <= 0.005 * same.size     # the rays that miss it (all explained) are few: 1 of 2 790 measured
    assert n_rephased + n_edge <= 0.03 * same.size        # measured: 0 re-phased + 31 on an edge of 2 790 (1.1 %)
    assert err.max() < 5e-3                               # and no ray, set aside or not, is far off
    dl = dloss * same[:, None]
    og, _ = orc.render_backward(sc, ctx, img, dl)
    out = gx.gpu_render(sc, cam, cfg, white=False, supersampling=(2, 1), want_grad=dl)
    _check_grads(gx, out["grads"], og, keys=("positions", "scales", "quaternions", "densities", "color_features",
                                             "sph_gauss_features", "bandwidth_sharpness", "lobe_axis"))


@pytest.mark.parametrize("n,scale", [(1, 12.0), (2, 12.0), (112, 8.0), (113, 8.0), (600, 2.0), (3000, 0.5)])
@pytest.mark.parametrize("words", [None, 16384])
def test_window_sums_of_groups_at_one_slot_and_at_many(gx, n, scale, words):
    """A replay's groups of lanes add to a window's sums at the same table slot in one trip (one Gaussian that
    covers the image: all eight of them) or at eight different ones (small Gaussians), with tables around their size
    of 112: the gradients of the backward that adds every row's share to memory.  Sums of at most some 10^5
    terms in another order: 2e-5, as for the other replays."""
    sc = scenes.scene_to_numpy(scenes.make_scene(0, n=n, sh_degree=0, seed=31))
    sc["scales"] = sc["scales"] * scale
    sc["positions"] = sc["positions"] * 0.4
    sc["densities"] = sc["densities"] + 0.2
    cam = scenes.make_camera(0, 1, width=44, height=36)
    cfg = dict(dt_step=0.004, dynamic_sampling=False, max_prim_slice=4096)
    dloss = np.random.default_rng(5).normal(size=(44 * 36, 3)).astype(np.float32)
    _step(f"window sums n={n} scale={scale} words={words}")
    a = gx.gpu_render(sc, cam, cfg, want_grad=dloss, record_hits=False)
    b = gx.gpu_render(sc, cam, cfg, want_grad=dloss, rec_tile_words=words, stats=False)
    assert a["stats_bwd"]["hit_pairs"] > 500
    for k in ("positions", "scales", "quaternions", "densities", "color_features"):
        cos, rel = gx.cos_rel(b["grads"][k], a["grads"][k])
        assert cos >= 1 - 1e-9 and rel <= 2e-5, (k, cos, rel)


@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
@pytest.mark.parametrize("words", [None, 16384])
def test_a_loss_gradient_that_is_no_number_stays_with_the_gaussians_its_ray_hits(gx, bad, words):
    """dL/dC of one ray is not a number: the Gaussians that this ray does not hit keep their gradients."""
    sc = scenes.scene_to_numpy(scenes.make_scene(0, n=4096, sh_degree=0, seed=31))
    cam = scenes.make_camera(0, 1, width=64, height=64)
    cfg = dict(dt_step=0.004, dynamic_sampling=False, max_prim_slice=4096)
    dloss = np.random.default_rng(5).normal(size=(64 * 64, 3)).astype(np.float32)
    ray = 30 * 64 + 33
    only = np.zeros_like(dloss)
    only[ray] = 1.0
    _step(f"odd loss {bad} words={words}")
    hit = np.abs(gx.gpu_render(sc, cam, cfg, want_grad=only, record_hits=False)["grads"]["color_features"]).sum((1, 2)) > 0
    dloss[ray] = 0.0
    a = gx.gpu_render(sc, cam, cfg, want_grad=dloss, record_hits=False)
    dloss[ray] = bad
    b = gx.gpu_render(sc, cam, cfg, want_grad=dloss, rec_tile_words=words, stats=False)
    assert 1 <= hit.sum() < 400
    for k in ("positions", "scales", "quaternions", "densities", "color_features"):
        assert np.isfinite(b["grads"][k][~hit]).all(), k
        cos, rel = gx.cos_rel(b["grads"][k][~hit], a["grads"][k][~hit])
        assert cos >= 1 - 1e-9 and rel <= 2e-5, (k, cos, rel)


def test_rays_beside_the_scene_leave_its_gradients_alone(gx):
    """Rays along an axis that pass the scene's box stand at no finite place; they share lane groups with rays that hit."""
    sc = scenes.scene_to_numpy(scenes.make_scene(0, n=300, sh_degree=0, seed=31))
    sc["positions"] = sc["positions"] * np.array([0.3, 0.03, 0.3], np.float32) + np.array([0.0, 0.12, 0.0], np.float32)
    sc["scales"] = sc["scales"] * 0.3
    cam = scenes.look_at_camera((3.0, 0.0, 0.0), fov_x_deg=30, width=33, height=33)      # the middle column: y = 0 throughout
    cfg = dict(dt_step=0.004, dynamic_sampling=False, max_prim_slice=4096)
    dloss = np.random.default_rng(5).normal(size=(33 * 33, 3)).astype(np.float32)
    _step("rays beside the scene")
    a = gx.gpu_render(sc, cam, cfg, want_grad=dloss, record_hits=False)
    b = gx.gpu_render(sc, cam, cfg, want_grad=dloss, stats=False)
    for k in ("positions", "scales", "quaternions", "densities", "color_features"):
        assert np.isfinite(b["grads"][k]).all() and np.abs(b["grads"][k]).sum() > 0, k
        cos, rel = gx.cos_rel(b["grads"][k], a["grads"][k])
        assert cos >= 1 - 1e-9 and rel <= 2e-5, (k, cos, rel)


@pytest.mark.parametrize("w,h,half", [(52, 44, True), (321, 307, False), (321, 307, True)])
def test_backward_in_pieces_equals_recomputation(gx, w, h, half):
    """The record of a tile cut into pieces that are replayed side by side, each from the rays' state that the
    forward kept: few tiles (up to 16 pieces; 11 with half-precision sums, whose slots hold fewer states) and
    between half a round and two rounds of tiles (up to 8, the XCDs at different pieces)."""
    sc = scenes.scene_to_numpy(scenes.make_scene(2, n=5000, sh_degree=1, seed=21))
    sc["scales"] = sc["scales"] * 3.0
    cam = scenes.make_camera(2, 1, width=w, height=h)
    cfg = dict(dt_step=0.004, dynamic_sampling=True, max_prim_slice=4096)
    dloss = np.random.default_rng(3).normal(size=(w * h, 3)).astype(np.float32)
    _step(f"pieces {w}x{h} half={half}")
    a = gx.gpu_render(sc, cam, cfg, want_grad=dloss, record_hits=False)
    b = gx.gpu_render(sc, cam, cfg, want_grad=dloss, half_sums=half)
    assert b["stats_bwd"]["nodes_visited"] == 0 and a["stats_bwd"]["hit_pairs"] == b["stats_bwd"]["hit_pairs"] > 10000
    for k in ("positions", "scales", "quaternions", "densities", "color_features"):
        cos, rel = gx.cos_rel(b["grads"][k], a["grads"][k])
        assert cos >= 1 - 1e-6 and rel <= (1e-3 if half else 1e-4), (k, cos, rel)


@pytest.mark.parametrize("w,h", [(1, 1), (9, 7), (216, 224), (224, 224)])
@pytest.mark.parametrize("config,scale,dyn", [(0, 1.0, False), (2, 4.0, True)])
def test_forward_with_one_and_with_four_wavefronts_per_tile(gx, orc, w, h, config, scale, dyn):
    """The smallest images and both sides of the number of tiles (756, 784) at which the forward goes over from four
    wavefronts per tile to one; sparse slabs, and slabs whose candidates fill several tables.  With and without a
    record, counting and not."""
    sc = scenes.scene_to_numpy(scenes.make_scene(config, n=6000, sh_degree=1, seed=31))
    sc["scales"] = sc["scales"] * scale
    cam = scenes.make_camera(config, 1, width=w, height=h)
    cfg = dict(dt_step=0.004, dynamic_sampling=dyn, max_prim_slice=4096)
    ids = np.unique(np.random.default_rng(6).integers(0, w * h, 300))
    img, st, ctx = orc.render_forward(sc, cam, cfg["dt_step"], dyn, 4096, ray_ids=ids)
    dloss = np.zeros((w * h, 3), np.float32)
    dloss[ids] = np.random.default_rng(7).normal(size=(len(ids), 3)).astype(np.float32)
    _step(f"wavefronts per tile {w}x{h} config {config}")
    _, counts = gx.gpu_forward_counts(sc, cam, cfg)
    same, rephased, edge = gx.comparable_rays(orc, ctx, img, counts, ids)
    assert rephased + edge <= (0.05 * len(ids) if dyn else 0)
    dloss[ids[~same]] = 0
    og, _ = orc.render_backward(sc, ctx, img, dloss)
    plain = gx.gpu_render(sc, cam, cfg)["image"]
    for stats in (True, False):
        out = gx.gpu_render(sc, cam, cfg, want_grad=dloss, stats=stats)
        for image in (out["image"], plain):
            assert np.abs(image[ids] - img[ids])[same].max() <= IMG_TOL
        assert np.abs(out["image"] - plain).max() <= (5e-3 if dyn else 1e-5)      # (adaptive: a ray may be re-phased)
        if w > 1:
            _check_grads(gx, out["grads"], og)


@pytest.mark.parametrize("dyn,cap,scale", [(True, 4096, 1.0), (True, 4096, 4.0), (False, 4096, 1.0), (False, 8, 4.0)])
def test_forward_without_a_record_is_the_march_that_its_backward_repeats(gx, dyn, cap, scale):
    """A backward without a record searches the tree again, with one wavefront per tile: its forward has to add up and
    to cut off the hits of a ray as that does, whatever the number of tiles.  The same rays as the first rows of an
    image eight times as high (a power of two: the same directions in every bit), whose 1040 tiles always have one
    wavefront each, come out the same in every bit.  An image that no backward follows only has to be near."""
    from raygaussx_amd import optix_utils as u_ox
    from raygaussx_amd.render_optix import compute_rgb
    w, h = 100, 80          # (whole tiles downwards: the same rays take part in each)
    sc = gx.to_dev(scenes.scene_to_numpy(scenes.make_scene(2, n=6000, sh_degree=0, seed=31)))
    cam = scenes.make_camera(2, 1, width=w, height=h)
    cs, tall = u_ox.camera_struct(cam), u_ox.camera_struct(cam)
    tall.height, tall.tan_half_fov_y, tall.principal_y = 8 * h, 8 * cs.tan_half_fov_y, cs.principal_y / 8
    params = sc["positions"], sc["scales"] * scale, sc["quaternions"], sc["densities"]
    gas = u_ox.AccelerationStructure(6000, gx.DEV).build_from_gaussians(*params)
    rgb = compute_rgb(cam.camera_center, sc["positions"], sc["color_features"], None, None, None, 0, 0)
    prims = u_ox.pack_prims(gas, cs, *params, rgb)
    _step(f"forward without a record, adaptive {dyn}, cut at {cap}")
    image = u_ox.march_forward(gas, cs, prims, 0.004, dyn, cap, True)
    assert torch.equal(image, u_ox.march_forward(gas, tall, prims, 0.004, dyn, cap, True)[:w * h])
    assert (image - 1.0).abs().max() > 0.1                                    # (not the background)
    only = u_ox.launch_pipeline_test(None, None, gas, None, None, 0.004, dyn, cam, params[3], rgb, *params[:3], cap)
    if cap > 8:
        assert (only - image).abs().max() <= (5e-3 if dyn else 1e-5)          # (adaptive: a ray may be re-phased)
    # the same through the autograd function: with a backward to come, and without
    np_scene = {k: v.cpu().numpy() for k, v in sc.items()}
    np_scene["scales"] = np_scene["scales"] * np.float32(scale)
    cfg = dict(dt_step=0.004, dynamic_sampling=dyn, max_prim_slice=cap)
    out = gx.gpu_render(np_scene, cam, cfg, want_grad=np.ones((w * h, 3), np.float32), stats=False, record_hits=False)
    assert np.array_equal(out["image"], image.cpu().numpy())
    assert np.array_equal(gx.gpu_render(np_scene, cam, cfg, stats=False)["image"], only.cpu().numpy())


@pytest.mark.parametrize("n", [1, 2, 3, 64, 65, 129, 6000])
# 812, 1 296 and 1 332 tiles, by 4x4 blocks (adaptive: halves); 3 249 whole tiles, by pairs; 18 496 and 18 632, by nodes: six rounds are 18 432
@pytest.mark.parametrize("w,h", [(225, 224), (285, 281), (289, 288), (456, 456), (1088, 1083), (1096, 1084)])
@pytest.mark.parametrize("dyn", [False, True])
def test_sweeps_by_pairs_of_nodes_and_by_nodes_find_the_same(gx, n, w, h, dyn):
    """Trees from a single leaf up, either side of the number of tiles up to which an image that no backward follows
    sweeps the tree by pairs of nodes: image and counters of the forward that goes by nodes.  Dense scenes fill several
    tables.  (Sums in another order: 1e-5; adaptive: a ray may be re-phased.)"""
    from raygaussx_amd import optix_utils as u_ox
    from raygaussx_amd.render_optix import compute_rgb
    sc = gx.to_dev(scenes.scene_to_numpy(scenes.make_scene(2 if dyn else 0, n=n, sh_degree=0, seed=33)))
    cam = scenes.make_camera(0, 1, width=w, height=h)
    params = sc["positions"], sc["scales"] * 4.0, sc["quaternions"], sc["densities"]
    gas = u_ox.AccelerationStructure(n, gx.DEV).build_from_gaussians(*params)
    cs = u_ox.camera_struct(cam)
    rgb = compute_rgb(cam.camera_center, sc["positions"], sc["color_features"], None, None, None, 0, 0)
    prims = u_ox.pack_prims(gas, cs, *params, rgb)
    a_st, b_st = u_ox.new_stats(gx.DEV), u_ox.new_stats(gx.DEV)
    _step(f"pairs n={n} {w}x{h} adaptive {dyn}")
    a = u_ox.march_forward(gas, cs, prims, 0.01, dyn, 4096, True, stats=a_st)
    b = u_ox.launch_pipeline_test(None, None, gas, None, None, 0.01, dyn, cam, params[3], rgb, *params[:3], 4096, stats=b_st)
    plain = u_ox.launch_pipeline_test(None, None, gas, None, None, 0.01, dyn, cam, params[3], rgb, *params[:3], 4096)
    assert torch.equal(b, plain)
    assert (a - b).abs().max() <= (5e-3 if dyn else 1e-5)
    sa, sb = u_ox.read_stats(a_st), u_ox.read_stats(b_st)
    assert (sa["hit_pairs"] > 0 or n < 64) and sa["rays_hit"] == sb["rays_hit"]
    if not dyn:
        # (A ray whose transmittance is within rounding of its end: it ends a slab earlier or later, some hundred hits.)
        assert abs(sa["slabs"] - sb["slabs"]) <= 1
        assert abs(sb["hit_pairs"] - sa["hit_pairs"]) <= (0 if n < 6000 else 100)


# fixed step: 768 and 784 tiles, 2 048 and 2 064, 3 200 and 3 240; adaptive: 256 and 272, 800 and 825, 1 600 and 1 640.  Odd sizes: parts without a ray
@pytest.mark.parametrize("dyn,w,h", [(False, 5, 3), (False, 256, 190), (False, 219, 219), (False, 507, 256), (False, 509, 257), (False, 512, 395),
                                     (False, 479, 427), (True, 5, 3), (True, 125, 126), (True, 131, 126), (True, 200, 251), (True, 195, 259),
                                     (True, 313, 318), (True, 328, 313)])
@pytest.mark.parametrize("scale,n", [(1.0, 6000), (5.0, 6000), (1.0, 3)])
def test_images_by_parts_of_tiles(gx, dyn, w, h, scale, n):
    """Either side of the numbers of tiles at which an image goes over from 4x2 pixels a wavefront to 4x4, to half a tile and to a tile: the image and
    the counters of the forward that leaves a record.  Sparse slabs, and slabs whose candidates fill several tables; with lists that
    max_prim_slice could cut but does not (the filter then goes entry by entry).  (Sums in another order: 1e-5; adaptive: a ray may be re-phased.)"""
    from raygaussx_amd import optix_utils as u_ox
    from raygaussx_amd.render_optix import compute_rgb
    sc = gx.to_dev(scenes.scene_to_numpy(scenes.make_scene(2 if dyn else 0, n=n, sh_degree=0, seed=33)))
    cam = scenes.make_camera(2 if dyn else 0, 1, width=w, height=h)
    params = sc["positions"], sc["scales"] * scale, sc["quaternions"], sc["densities"]
    gas = u_ox.AccelerationStructure(n, gx.DEV).build_from_gaussians(*params)
    cs = u_ox.camera_struct(cam)
    rgb = compute_rgb(cam.camera_center, sc["positions"], sc["color_features"], None, None, None, 0, 0)
    prims = u_ox.pack_prims(gas, cs, *params, rgb)
    tol = 5e-3 if dyn else 1e-5
    _step(f"parts {w}x{h} n={n} scale {scale} adaptive {dyn}")
    st = [u_ox.new_stats(gx.DEV) for _ in range(3)]
    rec = torch.empty(u_ox.records_bytes(cs, 16384 * 4), dtype=torch.uint8, device=gx.DEV)
    whole = u_ox.march_forward(gas, cs, prims, 0.01, dyn, 4096, True, records=rec, stats=st[0])
    test = lambda cap, **kw: u_ox.launch_pipeline_test(None, None, gas, None, None, 0.01, dyn, cam, params[3], rgb, *params[:3], cap, **kw)
    image = test(4096, stats=st[1])
    assert torch.equal(image, test(4096)) and (image - whole).abs().max() <= tol
    a, b = u_ox.read_stats(st[0]), u_ox.read_stats(st[1])
    assert a["rays_hit"] == b["rays_hit"] and a["overflow_rays"] == b["overflow_rays"] == 0
    if not dyn:
        assert abs(a["slabs"] - b["slabs"]) <= 1 and abs(a["hit_pairs"] - b["hit_pairs"]) <= 100 * abs(a["slabs"] - b["slabs"]), (a, b)
    cut = test(60, stats=st[2])
    if u_ox.read_stats(st[2])["overflow_rays"] == 0:
        assert (cut - whole).abs().max() <= tol
    frame, depth = u_ox.march_viewer(gas, cs, prims, 0.01, dyn, 4096)
    black = u_ox.march_forward(gas, cs, prims, 0.01, dyn, 4096, False, records=rec)
    assert (frame.reshape(-1, 4)[:, :3].float() - (black.clamp(0, 1) * 256).floor().clamp(max=255)).abs().max() <= (1 if not dyn else 2)
    hit = (whole - black).amax(1) < 1 - 1e-6                                   # (some of the background is gone: something was met)
    assert torch.equal(depth.reshape(-1)[hit] > 0, torch.ones_like(hit[hit]))


@pytest.mark.parametrize("w,h", [(45, 64), (225, 224), (393, 400), (457, 456)])    # 4x2 pixels, 4x4 blocks, halves, whole tiles
@pytest.mark.parametrize("axis", [0, 1])
def test_viewer_depth_of_rays_that_are_nowhere(gx, axis, w, h):
    """A ray whose direction has a component of exactly zero, with the eye beside the box on that axis, enters the box at no finite distance: its depth is
    zero, whatever the rays marched together with it meet."""
    from raygaussx_amd import _lib as L
    from raygaussx_amd import optix_utils as u_ox
    w, h = (w, h) if axis == 0 else (h, w)
    n = 4000
    rng = np.random.default_rng(2)
    pos = rng.uniform(0.0, 0.5, size=(n, 3)).astype(np.float32)
    pos[:, 1 - axis] -= 0.25
    pos[:, 2] += 4.0
    d = gx.to_dev(dict(positions=pos, scales=np.full((n, 3), 0.02, np.float32), quaternions=np.float32([[1, 0, 0, 0]]).repeat(n, 0),
                       densities=np.full(n, 2.0, np.float32), rgb=np.full((n, 3), 0.5, np.float32)))
    params = d["positions"], d["scales"], d["quaternions"], d["densities"]
    gas = u_ox.AccelerationStructure(n, gx.DEV).build_from_gaussians(*params)
    cs = L.RgxCamera()
    cs.u[0] = cs.v[1] = cs.w[2] = 1.0
    cs.tan_half_fov_x = cs.tan_half_fov_y = 0.1
    cs.principal_x = cs.principal_y = 0.5
    cs.width, cs.height = w, h
    cs.eye[axis] = float(u_ox.ellipsoids_bbox_from_quat(params[2], params[0], params[1], params[3])[1][axis]) - 1e-3
    prims = u_ox.pack_prims(gas, cs, *params, d["rgb"])
    _step(f"viewer depth, {w}x{h}")
    _, depth = u_ox.march_viewer(gas, cs, prims, 0.01, False, 4096)
    depth = depth if axis == 0 else depth.T
    mid = depth.shape[1] // 2
    assert torch.isfinite(depth).all() and (depth[:, : mid + 1] == 0).all() and (depth[:, mid + 1:] > 3.0).sum() > 100


# an image by 4x2 pixels (756 tiles; a strip of 760), 4x4 blocks (1 225), halves (2 500) and whole tiles (3 249); its record by 4x4 blocks, halves, whole tiles
@pytest.mark.parametrize("fov,w,h", [(5.0, 216, 224), (40.0, 760, 64), (5.0, 276, 276), (5.0, 312, 304), (5.0, 400, 400), (5.0, 456, 456), (1.0, 216, 224), (1.0, 456, 456)])
def test_narrow_pixels_lose_no_hit(gx, orc, fov, w, h):
    """Where neighbouring rays are a ten-thousandth apart a part's frustum still holds all that its rays meet: as many slabs and hits as the oracle counts
    ray by ray (small spheres, of which many are only grazed, and too thin for any ray to end), in the image, in the forward that leaves a record, in the forward by
    whole tiles, and in a search of the tree in the place of a replay."""
    from raygaussx_amd import optix_utils as u_ox
    from raygaussx_amd.render_optix import compute_rgb
    n = 6000
    sc = scenes.scene_to_numpy(scenes.make_scene(0, n=n, sh_degree=0, seed=5))
    sc["scales"] = np.repeat(np.exp(np.random.default_rng(1).normal(size=(n, 1)) * 0.4 - 3.5).astype(np.float32), 3, 1)
    sc["densities"][:] = 0.2
    at = np.float32([13.0, 14.0, 12.0]) * (5.0 / fov if fov < 40.0 else 0.18)
    cam = scenes.look_at_camera(tuple(float(x) for x in at), fov_x_deg=fov, width=w, height=h)
    _, want, ctx = orc.render_forward(sc, cam, 0.01, False, 4096, cull=True)
    orc.cull_free()
    d = gx.to_dev(sc)
    params = d["positions"], d["scales"], d["quaternions"], d["densities"]
    gas = u_ox.AccelerationStructure(n, gx.DEV).build_from_gaussians(*params)
    cs = u_ox.camera_struct(cam)
    rgb = compute_rgb(cam.camera_center, d["positions"], d["color_features"], None, None, None, 0, 0)
    prims = u_ox.pack_prims(gas, cs, *params, rgb)
    _step(f"narrow pixels, {w}x{h} over {fov} degrees")
    st = [u_ox.new_stats(gx.DEV) for _ in range(4)]
    u_ox.launch_pipeline_test(None, None, gas, None, None, 0.01, False, cam, params[3], rgb, *params[:3], 4096, stats=st[0])
    rec = torch.empty(u_ox.records_bytes(cs, 16384 * 4), dtype=torch.uint8, device=gx.DEV)
    image = u_ox.march_forward(gas, cs, prims, 0.01, False, 4096, True, records=rec, stats=st[1])
    u_ox.march_forward(gas, cs, prims, 0.01, False, 4096, True, stats=st[2])
    u_ox.march_backward(gas, cs, prims, image, torch.ones_like(image), 0.01, False, 4096, True, records=torch.zeros_like(rec), stats=st[3])
    got = [u_ox.read_stats(s) for s in st]
    assert [(g["slabs"], g["hit_pairs"]) for g in got] == [(want["slabs"], want["hit_pairs"])] * 4


@pytest.mark.parametrize("w,h", [(52, 44), (216, 224), (253, 256)])              # by 4x4 blocks
def test_record_forms_of_a_small_image_with_the_fixed_step(gx, w, h):
    """What the parts of a tile leave for the backward, in each form: sample sums in floats and in half
    precision, and hit lists alone.  The image does not depend on the form.  Float sums and lists give the gradients of
    a backward that searches the tree; half precision rounds a colour sum by at most 2^-12 of the chunk's
    largest, and a gradient's norm is that of many of them: 2^-12 of it."""
    sc = scenes.scene_to_numpy(scenes.make_scene(0, n=5000, sh_degree=1, seed=21))
    sc["scales"] = sc["scales"] * 2.0
    cam = scenes.make_camera(0, 0, width=w, height=h)
    cfg = dict(dt_step=0.004, dynamic_sampling=False, max_prim_slice=4096)
    dloss = np.random.default_rng(3).normal(size=(w * h, 3)).astype(np.float32)
    _step(f"record forms {w}x{h}")
    tree = gx.gpu_render(sc, cam, cfg, want_grad=dloss, record_hits=False)
    forms = [("sums", dict(), 1e-4), ("half sums", dict(half_sums=True), 2.0 ** -12), ("lists", dict(rec_tile_words=16384), 1e-4)]
    images = []
    for name, kw, tol in forms:
        for _ in range(2):                     # (the second view's pool is sized from the first)
            out = gx.gpu_render(sc, cam, cfg, want_grad=dloss, **kw)
        assert out["stats_bwd"]["nodes_visited"] == 0 and out["stats_bwd"]["hit_pairs"] == tree["stats_bwd"]["hit_pairs"] > 10000
        images.append(out["image"])
        for k in ("positions", "scales", "quaternions", "densities", "color_features"):
            cos, rel = gx.cos_rel(out["grads"][k], tree["grads"][k])
            print(f"{name}, {k}: rel {rel:.2e}", flush=True)
            assert cos >= 1 - 1e-6 and rel <= tol, (name, k, cos, rel)
    assert np.array_equal(images[0], images[1]) and np.array_equal(images[0], images[2])
    assert np.abs(images[0] - tree["image"]).max() <= 1e-5


# either side of 1 200 and of 2 000 tiles: 4x4 blocks, halves, whole tiles.  Odd sizes: parts without a ray
@pytest.mark.parametrize("w,h", [(5, 3), (237, 315), (240, 320), (243, 319), (317, 399), (319, 408)])
def test_records_by_parts_of_tiles(gx, w, h):
    """The gradients of a record by parts, in each form, with hardly room for a part's share (its lists go on in a slot of the pool) and with none in the
    pool either (some parts are searched again): those of a backward that searches whole tiles, up to the order of sums (1e-4, as above).
    Half precision rounds a colour sum by at most 2^-12 times the power of two above its chunk's largest: by 2^-11 of the largest, and a gradient's norm with it."""
    sc = scenes.scene_to_numpy(scenes.make_scene(0, n=5000, sh_degree=1, seed=21))
    sc["scales"] = sc["scales"] * 3.0
    cam = scenes.make_camera(0, 0, width=w, height=h)
    cfg = dict(dt_step=0.01, dynamic_sampling=False, max_prim_slice=4096)
    dloss = np.random.default_rng(3).normal(size=(w * h, 3)).astype(np.float32)
    _step(f"records by parts {w}x{h}")
    tree = gx.gpu_render(sc, cam, cfg, want_grad=dloss, record_hits=False)
    images = []
    for name, kw, tol in [("sums", dict(), 1e-4), ("half sums", dict(half_sums=True), 2.0 ** -11), ("lists", dict(rec_tile_words=16384), 1e-4),
                          ("few slots", dict(rec_tile_words=16384 + 2 * 8192), 1e-4), ("short lists", dict(rec_tile_words=2048), 1e-4)]:
        out = gx.gpu_render(sc, cam, cfg, want_grad=dloss, **kw)
        assert out["stats_bwd"]["hit_pairs"] == tree["stats_bwd"]["hit_pairs"], name
        assert w == 5 or (out["stats_bwd"]["nodes_visited"] > 0) == (name == "short lists"), name
        images.append(out["image"])
        for k in ("positions", "scales", "quaternions", "densities", "color_features"):
            cos, rel = gx.cos_rel(out["grads"][k], tree["grads"][k])
            assert cos >= 1 - 1e-6 and rel <= tol, (name, k, cos, rel)
    assert all(np.array_equal(images[0], i) for i in images[1:])
    assert np.abs(images[0] - tree["image"]).max() <= 1e-5


@pytest.mark.parametrize("config,n,w,h,slots", [(0, 4096, 240, 240, 7), (1, 30_011, 256, 256, None), (1, 30_011, 304, 304, None)])
def test_sums_find_room_in_a_pool_that_has_it(gx, config, n, w, h, slots):
    """The slots that parts have to begin with hold sums: a pool of seven slots a tile where the sums ask for 5.3 and no list goes on in a slot, and the
    first view's of a scene whose sums ask for 8.7 (fewer by halves).  Every part then has its sums (status 2, first word of its region)."""
    from raygaussx_amd import optix_utils as u_ox
    from raygaussx_amd.render_optix import compute_rgb
    sc = gx.to_dev(scenes.scene_to_numpy(scenes.make_scene(config, n=n, sh_degree=0, seed=33)))
    cam = scenes.make_camera(config, 1, width=w, height=h)
    params = sc["positions"], sc["scales"], sc["quaternions"], sc["densities"]
    gas = u_ox.AccelerationStructure(n, gx.DEV).build_from_gaussians(*params)
    cs = u_ox.camera_struct(cam)
    rgb = compute_rgb(cam.camera_center, sc["positions"], sc["color_features"], None, None, None, 0, 0)
    prims = u_ox.pack_prims(gas, cs, *params, rgb)
    ntiles = ((w + 7) // 8) * ((h + 7) // 8)
    parts = 4 if ntiles <= 1200 else 2
    if slots is None:
        rec = u_ox.new_records(cs, gx.DEV, n=n)
    else:
        rec = torch.empty(u_ox.records_bytes(cs, 16384 + slots * 8192), dtype=torch.uint8, device=gx.DEV)
    _step(f"room for sums, {w}x{h}")
    u_ox.march_forward(gas, cs, prims, 0.01 if config == 0 else 0.0025, False, 4096, True, records=rec)
    regions = rec[:ntiles * 16384 * 4].view(torch.int32).view(ntiles * parts, -1)
    assert torch.equal(regions[:, 0], torch.full_like(regions[:, 0], 2))


@pytest.mark.parametrize("w,h", [(1, 1), (256, 304)])                            # 4x4 blocks; halves
def test_replay_of_lists_where_a_ray_ends_on_the_floor(gx, orc, w, h):
    """A replay of lists alone, by parts, may round a ray's transmittance otherwise than its forward, whose ray ended with just t_eps left: no record is lost for it, in
    views of one ray (of an otherwise empty image) through sixty Gaussians, at every floor that the ray itself reaches."""
    from raygaussx_amd import optix_utils as u_ox
    n = 70
    cam = scenes.look_at_camera((4.0, 0.5, 0.2), fov_x_deg=1.0 if w == 1 else 170.0, width=w, height=h)
    cs = u_ox.camera_struct(cam)
    px = 0 if w == 1 else (h // 2) * w + w // 2
    along = orc.ray_dirs(orc.camera_struct(cam), np.int32([px]))[0]
    ones = torch.ones(w * h, 3, device=gx.DEV)
    rec = torch.empty(u_ox.records_bytes(cs, 16384), dtype=torch.uint8, device=gx.DEV)
    _step(f"floors, {w}x{h}")
    floors = set()
    for seed in range(12):
        rng = np.random.default_rng(seed)
        t = rng.uniform(3.7, 4.3, size=(n, 1)) + (np.arange(n)[:, None] >= 60) * 4.0
        pos = (np.float32([4.0, 0.5, 0.2]) + t * along + rng.normal(size=(n, 3)) * 0.01).astype(np.float32)
        d = gx.to_dev(dict(pos=pos, scales=rng.uniform(0.02, 0.06, size=(n, 3)).astype(np.float32),
                           quat=rng.normal(size=(n, 4)).astype(np.float32), dens=rng.uniform(0.2, 2.0, size=n).astype(np.float32), rgb=np.zeros((n, 3), np.float32)))
        params = d["pos"], d["scales"], torch.nn.functional.normalize(d["quat"]), d["dens"]
        gas = u_ox.AccelerationStructure(n, gx.DEV).build_from_gaussians(*params)
        prims = u_ox.pack_prims(gas, cs, *params, d["rgb"])
        for guess in np.linspace(0.99, 0.3, 24):
            left = lambda eps: float(u_ox.march_forward(gas, cs, prims, 0.004, False, 4096, True, t_eps=eps, records=rec)[px, 0])  # (black on white: what is left of the ray)
            eps = left(float(guess))
            image = u_ox.march_forward(gas, cs, prims, 0.004, False, 4096, True, t_eps=eps, records=rec)
            if float(image[px, 0]) != eps or eps in floors:
                continue
            floors.add(eps)
            st = u_ox.new_stats(gx.DEV)
            u_ox.march_backward(gas, cs, prims, image, ones, 0.004, False, 4096, True, t_eps=eps, records=rec, stats=st)
            assert u_ox.read_stats(st)["replay_lost"] == 0 == u_ox.march_faults(n, gx.DEV)[0], (seed, eps)
    assert len(floors) > 30


# with the fixed step: up to 1 200 tiles by 4x4 blocks; 1 482 by halves; 2 500 whole tiles by pairs of nodes, 18 632 by nodes
@pytest.mark.parametrize("w,h", [(52, 44), (100, 80), (253, 256), (257, 256), (312, 304), (400, 400), (1089, 1082)])
@pytest.mark.parametrize("dyn,cap", [(False, 8), (False, 32), (False, 4096), (True, 32)])
def test_a_tile_whose_record_overflowed_keeps_the_hits_that_its_forward_kept(gx, w, h, dyn, cap):
    """Where max_prim_slice cuts a ray's list the order of the sweep decides which hits it keeps, so the backward has to
    search the tiles whose region overflowed as their forward did: the gradients of the same view with room
    for its record, up to the order of sums and samples at a cut-off (1e-4, as for the forms of a record; measured 4e-5).
    With lists cut to other hits they were off by as much as the gradient itself, and by 1.1e-4 at 312x304 where only the
    box test and the clipping of the slabs were not the forward's."""
    sc = scenes.scene_to_numpy(scenes.make_scene(2 if dyn else 0, n=6000, sh_degree=0, seed=21))
    sc["scales"] = sc["scales"] * np.float32(6.0)
    cam = scenes.make_camera(2 if dyn else 0, 1, width=w, height=h)
    cfg = dict(dt_step=0.01, dynamic_sampling=dyn, max_prim_slice=cap)
    dloss = np.random.default_rng(3).normal(size=(w * h, 3)).astype(np.float32)
    _step(f"cut lists, {w}x{h}, adaptive {dyn}, cap {cap}")
    room = gx.gpu_render(sc, cam, cfg, want_grad=dloss, rec_tile_words=16384 * 4)
    small = gx.gpu_render(sc, cam, cfg, want_grad=dloss, rec_tile_words=1024)
    plain = gx.gpu_render(sc, cam, cfg, want_grad=dloss, rec_tile_words=1024, stats=False)
    assert room["stats_bwd"]["nodes_visited"] == 0 < small["stats_bwd"]["nodes_visited"]
    assert (room["stats_fwd"]["overflow_rays"] > 100) == (cap < 4096)
    assert small["stats_bwd"]["hit_pairs"] == room["stats_bwd"]["hit_pairs"] > 10000
    for out in (small, plain):
        assert np.array_equal(out["image"], room["image"])
        for k in ("positions", "scales", "quaternions", "densities", "color_features"):
            cos, rel = gx.cos_rel(out["grads"][k], room["grads"][k])
            assert cos >= 1 - 1e-6 and rel <= 1e-4, (k, cos, rel)


@pytest.mark.parametrize("n", [1, 2, 3, 64, 65, 129, 257, 1025, -3000])      # (negative: at one place, a tree of chains)
@pytest.mark.parametrize("w,h", [(52, 44), (264, 264), (312, 304), (400, 400)])  # by 4x4 blocks; halves; whole tiles, by pairs of nodes
@pytest.mark.parametrize("cap", [4, 4096])
def test_searches_in_the_place_of_a_replay_find_what_the_forward_found(gx, n, w, h, cap):
    """Trees from a single leaf up, with the backward handed an empty record: every tile is searched, in the forward's order, and the gradients are
    those of the replay (1e-4, as above)."""
    from raygaussx_amd import optix_utils as u_ox
    from raygaussx_amd.render_optix import compute_rgb
    one_place, n = n < 0, abs(n)
    sc = gx.to_dev(scenes.scene_to_numpy(scenes.make_scene(0, n=n, sh_degree=0, seed=33)))
    if one_place:
        sc["positions"] = sc["positions"][:1].repeat(n, 1).contiguous()
        sc["densities"] = sc["densities"] * 0.02 + 0.101          # (barely seen: the rays go on through all of them)
    cam = scenes.make_camera(0, 1, width=w, height=h)
    params = sc["positions"], sc["scales"] * 8.0, sc["quaternions"], sc["densities"]
    gas = u_ox.AccelerationStructure(n, gx.DEV).build_from_gaussians(*params)
    cs = u_ox.camera_struct(cam)
    rgb = compute_rgb(cam.camera_center, sc["positions"], sc["color_features"], None, None, None, 0, 0)
    prims = u_ox.pack_prims(gas, cs, *params, rgb)
    dloss = torch.from_numpy(np.random.default_rng(3).normal(size=(w * h, 3)).astype(np.float32)).to(gx.DEV)
    _step(f"search for a replay, n={n} {w}x{h} cap {cap}")
    rec = torch.empty(u_ox.records_bytes(cs, 16384 * 4), dtype=torch.uint8, device=gx.DEV)
    image = u_ox.march_forward(gas, cs, prims, 0.01, False, cap, True, records=rec)
    stats = [u_ox.new_stats(gx.DEV) for _ in range(2)]
    a = u_ox.march_backward(gas, cs, prims, image, dloss, 0.01, False, cap, True, records=rec, stats=stats[0])
    b = u_ox.march_backward(gas, cs, prims, image, dloss, 0.01, False, cap, True, records=torch.zeros_like(rec), stats=stats[1])
    c = u_ox.march_backward(gas, cs, prims, image, dloss, 0.01, False, cap, True, records=torch.zeros_like(rec))
    sa, sb = (u_ox.read_stats(s) for s in stats)
    assert sa["hit_pairs"] == sb["hit_pairs"] and sb["candidates"] > 0 and u_ox.march_faults(n, gx.DEV) == (0, 0)
    assert sa["candidates"] == 0 or one_place                      # (the lists of all of them in a tile have no room)
    for x, y, z in zip(a, b, c):
        for got in (y, z):
            cos, rel = gx.cos_rel(got.cpu().numpy(), x.cpu().numpy())
            assert not x.any() and not got.any() or (cos >= 1 - 1e-6 and rel <= 1e-4), (cos, rel)


@pytest.mark.parametrize("w,h", [(52, 44), (312, 304), (400, 400)])              # fixed step: 4x4 blocks, halves, whole tiles; adaptive: whole tiles
@pytest.mark.parametrize("dyn", [False, True])
def test_a_record_of_the_other_kind_of_step_is_searched_again(gx, dyn, w, h):
    """A record is laid out as its forward's kind of step says.  A backward of the other kind takes no tile from it: the gradients of an empty record (1e-4, as above)."""
    from raygaussx_amd import optix_utils as u_ox
    from raygaussx_amd.render_optix import compute_rgb
    n = 3000
    sc = gx.to_dev(scenes.scene_to_numpy(scenes.make_scene(0, n=n, sh_degree=0, seed=33)))
    cam = scenes.make_camera(0, 1, width=w, height=h)
    params = sc["positions"], sc["scales"] * 3.0, sc["quaternions"], sc["densities"]
    gas = u_ox.AccelerationStructure(n, gx.DEV).build_from_gaussians(*params)
    cs = u_ox.camera_struct(cam)
    rgb = compute_rgb(cam.camera_center, sc["positions"], sc["color_features"], None, None, None, 0, 0)
    prims = u_ox.pack_prims(gas, cs, *params, rgb)
    dloss = torch.from_numpy(np.random.default_rng(3).normal(size=(w * h, 3)).astype(np.float32)).to(gx.DEV)
    _step(f"record of the other step, {w}x{h}, backward adaptive {dyn}")
    rec = torch.zeros(u_ox.records_bytes(cs, 16384 * 4), dtype=torch.uint8, device=gx.DEV)
    empty = torch.zeros_like(rec)
    image = u_ox.march_forward(gas, cs, prims, 0.01, not dyn, 4096, True, records=rec)
    st = [u_ox.new_stats(gx.DEV) for _ in range(2)]
    a = u_ox.march_backward(gas, cs, prims, image, dloss, 0.01, dyn, 4096, True, records=rec, stats=st[0])
    b = u_ox.march_backward(gas, cs, prims, image, dloss, 0.01, dyn, 4096, True, records=empty, stats=st[1])
    sa, sb = (u_ox.read_stats(s) for s in st)
    assert all(sa[k] == sb[k] for k in ("slabs", "hit_pairs", "candidates", "nodes_visited")) and sa["candidates"] > 0 == sa["replay_lost"]
    assert u_ox.march_faults(n, gx.DEV) == (0, 0)
    for x, y in zip(a, b):
        cos, rel = gx.cos_rel(y.cpu().numpy(), x.cpu().numpy())
        assert cos >= 1 - 1e-6 and rel <= 1e-4, (cos, rel)


# the image by 4x2 pixels (two sizes), 4x4 blocks (two), halves, whole tiles by pairs of nodes, by nodes; the record by 4x4 blocks (three), halves, whole tiles
@pytest.mark.parametrize("w,h", [(19, 13), (221, 216), (225, 224), (289, 288), (400, 408), (456, 456), (1096, 1084)])
@pytest.mark.parametrize("config,scale", [(0, 6.0), (0, 1.0)])
def test_hits_counted_are_those_of_whole_lists_on_every_way(gx, w, h, config, scale):
    """``hit_pairs`` says how many hits a view's slabs have, not how a kernel came by them: an image that collects its crowded slabs half by
    half counts what the recording forward counts.  (A ray whose transmittance is within rounding of its end may end a slab
    earlier or later, some hundred hits.)"""
    sc = scenes.scene_to_numpy(scenes.make_scene(config, n=6000, sh_degree=0, seed=21))
    sc["scales"] = sc["scales"] * np.float32(scale)
    cam = scenes.make_camera(config, 1, width=w, height=h)
    cfg = dict(dt_step=0.01, dynamic_sampling=False, max_prim_slice=4096)
    _step(f"hits counted, {w}x{h}, scale {scale}")
    whole = gx.gpu_render(sc, cam, cfg, want_grad=np.ones((w * h, 3), np.float32))["stats_fwd"]
    none = gx.gpu_render(sc, cam, cfg, want_grad=np.ones((w * h, 3), np.float32), record_hits=False)
    test = gx.gpu_render(sc, cam, cfg)
    assert np.array_equal(test["image"], gx.gpu_render(sc, cam, cfg, stats=False)["image"])
    for st in (none["stats_fwd"], none["stats_bwd"], test["stats_fwd"]):
        assert abs(st["slabs"] - whole["slabs"]) <= 1 and abs(st["hit_pairs"] - whole["hit_pairs"]) <= 100 * abs(st["slabs"] - whole["slabs"]), (st, whole)


@pytest.mark.parametrize("dyn,w,h,scale", [(True, 100, 80, 6.0), (True, 257, 256, 12.0), (False, 1089, 1082, 6.0)])    # (records by nodes, as without one)
@pytest.mark.parametrize("cap", [8, 32, 4096])
def test_forward_without_a_record_keeps_the_hits_that_its_backward_keeps(gx, dyn, w, h, scale, cap):
    """Crowded slabs (more Gaussians than a table) with lists cut at max_prim_slice: a forward that a backward follows keeps the hits
    of the slab's one list, with a record or without, so image and counts are the same, and so are the gradients that
    the replay and the search give (to 1e-4, as above; 2e-2 to 1 where the lists were collected half a slab at a time)."""
    sc = scenes.scene_to_numpy(scenes.make_scene(2 if dyn else 0, n=6000, sh_degree=0, seed=21))
    sc["scales"] = sc["scales"] * np.float32(scale)
    cam = scenes.make_camera(2 if dyn else 0, 1, width=w, height=h)
    cfg = dict(dt_step=0.01, dynamic_sampling=dyn, max_prim_slice=cap)
    dloss = np.random.default_rng(3).normal(size=(w * h, 3)).astype(np.float32)
    _step(f"no record, crowded slabs, {w}x{h}, adaptive {dyn}, cap {cap}")
    rec = gx.gpu_render(sc, cam, cfg, want_grad=dloss, rec_tile_words=16384 * 4)
    none = gx.gpu_render(sc, cam, cfg, want_grad=dloss, record_hits=False)
    assert (rec["stats_fwd"]["overflow_rays"] > 1000) == (cap < 4096)
    assert np.array_equal(none["image"], rec["image"])
    for k in ("hit_pairs", "slabs", "empty_slabs", "overflow_rays", "rays_hit"):
        assert none["stats_fwd"][k] == rec["stats_fwd"][k], k
    for k in ("positions", "scales", "quaternions", "densities", "color_features"):
        cos, rel = gx.cos_rel(none["grads"][k], rec["grads"][k])
        print(f"{k}: rel {rel:.2e}", flush=True)
        assert cos >= 1 - 1e-6 and rel <= 1e-4, (k, cos, rel)


def test_long_hit_lists_spill_and_truncation(gx, orc):
    """Fat Gaussians: slabs with far more than 32 hits (LDS part + spill area), then a tiny
    max_prim_slice to exercise the silent truncation path and its counter."""
    sc = scenes.scene_to_numpy(scenes.make_scene(0, n=4000, sh_degree=1, seed=9))
    sc["scales"] = sc["scales"] * 8.0
    cam = scenes.make_camera(0, 0, width=40, height=40)
    cfg = dict(dt_step=0.0025, dynamic_sampling=False, max_prim_slice=4000)
    img, st, ctx = orc.render_forward(sc, cam, 0.0025, False, 4000)
    centre, _ = orc.march_trace(ctx["cs"], ctx["ms"], ctx["bmin"], ctx["bmax"], ctx["prims"], 20 * 40 + 20)
    assert max(len(s[4]) for s in centre) > 40        # well past the 32 LDS entries per ray
    dloss = np.random.default_rng(2).normal(size=img.shape).astype(np.float32)
    og, _ = orc.render_backward(sc, ctx, img, dloss)
    _step("long hit lists")
    out = gx.gpu_render(sc, cam, cfg, want_grad=dloss)
    assert np.abs(out["image"] - img).max() <= IMG_TOL
    assert out["stats_fwd"]["hit_pairs"] == st["hit_pairs"]
    _check_grads(gx, out["grads"], og)
    _step("truncated hit lists")
    cfg_small = dict(cfg, max_prim_slice=8)
    out_s = gx.gpu_render(sc, cam, cfg_small)
    _, st_s, _ = orc.render_forward(sc, cam, 0.0025, False, 8)
    assert out_s["stats_fwd"]["overflow_rays"] > 0 and st_s["overflow_rays"] > 0
    assert np.isfinite(out_s["image"]).all()


def test_degenerate_scenes(gx, orc):
    cam = scenes.make_camera(0, 0, width=19, height=13)
    cfg = dict(dt_step=0.0025, dynamic_sampling=False, max_prim_slice=64)
    base = scenes.scene_to_numpy(scenes.make_scene(0, n=50, sh_degree=0, seed=4))
    # all Gaussians below the density threshold: nothing can be hit
    inv = dict(base)
    inv["densities"] = np.full(50, 0.05, np.float32)
    _step("invisible scene")
    out = gx.gpu_render(inv, cam, cfg, want_grad=np.ones((19 * 13, 3), np.float32))
    np.testing.assert_array_equal(out["image"], 1.0)
    for k in ("positions", "scales", "quaternions", "densities", "color_features"):
        assert not out["grads"][k].any()
    # a single Gaussian, and a camera sitting inside the scene box
    one = {k: v[:1].copy() for k, v in base.items()}
    one["positions"][:] = 0
    one["scales"][:] = 0.3
    one["densities"][:] = 2.0
    for eye in ((2.0, 0.1, 0.2), (0.05, 0.02, 0.0)):
        _step(f"single gaussian eye={eye}")
        cam1 = scenes.look_at_camera(eye, target=(-1.0, 0.0, 0.0), fov_x_deg=60, width=19, height=13)
        img, st, ctx = orc.render_forward(one, cam1, 0.0025, False, 64)
        out = gx.gpu_render(one, cam1, cfg)
        assert np.abs(out["image"] - img).max() <= IMG_TOL
        assert out["stats_fwd"]["hit_pairs"] == st["hit_pairs"]
    # axis-parallel rays (a zero direction component) and rays missing the scene box
    _step("axis-parallel camera")
    cam2 = scenes.look_at_camera((3.0, 0.0, 0.0), fov_x_deg=30, width=9, height=9)
    img, st, _ = orc.render_forward(base, cam2, 0.0025, False, 64)
    out = gx.gpu_render(base, cam2, cfg)
    assert np.abs(out["image"] - img).max() <= IMG_TOL


def test_morton_order_bit_exact(gx, orc):
    from raygaussx_amd.reordering import morton_order
    for n in (1, 77, 5000, 300_000):
        _step(f"morton n={n}")
        pos = np.random.default_rng(n).normal(size=(n, 3)).astype(np.float32)
        if n == 77:
            pos[:, 2] = 0.25            # zero extent on one axis
        order, codes = morton_order(torch.from_numpy(pos).to(gx.DEV), return_codes=True)
        np.testing.assert_array_equal(codes.cpu().numpy(), orc.morton_codes(pos))
        np.testing.assert_array_equal(order.cpu().numpy(), orc.morton_order(pos))


@pytest.mark.parametrize("n", [1, 2, 63, 65, 1023, 1025, 4096, 8191, 8192, 8193])
def test_orders_of_few_keys(gx, orc, n):
    """Both sorts on either side of the sizes at which one workgroup sorts, with keys that tie: the points' order against the
    oracle's, the tree's against the codes recomputed from the boxes and scene box it left in its workspace."""
    import ctypes as C
    from raygaussx_amd import _lib
    from raygaussx_amd import optix_utils as u_ox
    from raygaussx_amd.reordering import morton_order
    rng = np.random.default_rng(n)
    pos = rng.normal(size=(n, 3)).astype(np.float32)
    pos[n // 2:] = pos[:n - n // 2]
    _step(f"orders of {n} keys")
    np.testing.assert_array_equal(morton_order(torch.from_numpy(pos).to(gx.DEV)).cpu().numpy(), orc.morton_order(pos))
    scale, quat = np.full((n, 3), 0.01, np.float32), np.tile(np.float32([1, 0, 0, 0]), (n, 1))
    dens = np.ones(n, np.float32)
    gas = u_ox.AccelerationStructure(n, gx.DEV).build_from_gaussians(*(torch.from_numpy(a).to(gx.DEV) for a in (pos, scale, quat, dens)))
    lay = (C.c_size_t * 6)()
    _lib.check(_lib.lib().rgx_build_layout(C.c_int64(n), lay))
    torch.cuda.synchronize()
    view = lambda k, nbytes, t: gas.ws[lay[k]:lay[k] + nbytes].view(t).cpu().numpy()
    boxes, order, header = view(0, n * 24, torch.float32).reshape(n, 6), view(1, n * 4, torch.int32), view(5, 24, torch.float32)
    np.testing.assert_array_equal(header[:3], boxes[:, :3].min(0))
    np.testing.assert_array_equal(header[3:], boxes[:, 3:].max(0))
    ext = header[3:] - header[:3]
    centre = np.float32(0.5) * boxes[:, :3] + np.float32(0.5) * boxes[:, 3:]
    u = np.clip((centre - header[:3]) / np.where(ext > 0, ext, 1), 0, 1).astype(np.float32) * np.float32(2 ** 21)
    q = np.minimum(u.astype(np.int64), 2 ** 21 - 1)
    code = np.zeros(n, np.int64)
    for b in range(21):
        for a in range(3):
            code |= ((q[:, a] >> b) & 1) << (3 * b + 2 - a)
    np.testing.assert_array_equal(order, np.argsort(code, kind="stable"))


@pytest.mark.parametrize("n", [8_704, 65_536, 65_537, 196_608, 196_609])
def test_orders_of_more_keys(gx, orc, n):
    """Either side of the sizes at which the sort changes its tiles and its launches per pass."""
    test_orders_of_few_keys(gx, orc, n)


def test_reorder_tensors_is_the_per_tensor_gather(gx):
    """PointCloud.reorder_zordercurve's gathers (classes/point_cloud.py:1031-1044) in one launch:
    every tensor equals numpy's `t[index]`, for the parameter shapes of a point cloud with Adam
    moments (30 tensors: more than one launch holds), ragged sizes and an empty cloud."""
    from raygaussx_amd.reordering import morton_order, reorder_tensors
    rng = np.random.default_rng(8)
    for n in (0, 1, 1000, 100_003):
        _step(f"reorder_tensors n={n}")
        shapes = [(n, 3), (n, 3), (n, 4), (n,), (n, 3, 16), (n, 3, 2), (n, 2), (n, 2, 3), (n, 1), (n,)]
        params = [rng.normal(size=sh).astype(np.float32) for sh in shapes]
        tensors = params + [p * 2 for p in params] + [p * p for p in params]          # + exp_avg, exp_avg_sq
        tensors[9] = rng.integers(0, 1 << 40, size=n).astype(np.int64)                # an 8-byte counter
        order = morton_order(torch.from_numpy(params[0]).to(gx.DEV)) if n else torch.zeros(0, dtype=torch.int64, device=gx.DEV)
        dev = [torch.from_numpy(t).to(gx.DEV) for t in tensors]
        dev.insert(3, None)
        out = reorder_tensors(order, dev)
        assert out[3] is None and len(out) == len(dev)
        idx = order.cpu().numpy()
        for got, src in zip([o for o in out if o is not None], tensors):
            np.testing.assert_array_equal(got.cpu().numpy(), src[idx])


@pytest.mark.parametrize("n,words,offset", [
    (5, 4 * 4096, 0), (3, 4 * 4095, 0), (130, 4 * 4097, 0),        # a row of 16-byte pieces, either side of the long ones
    (3, 3 * 4099, 0), (3, 2 * 4097, 0), (2, 4099, 0), (2, 8195, 0),   # 12-, 8- and 4-byte pieces (4099, 8195: primes' worth)
    (257, 4, 1), (257, 8, 2), (257, 6, 1), (257, 2, 1), (257, 9, 1), (4, 4 * 4096, 1), (4, 4 * 4096, 2),   # off a 16- or 8-byte boundary
    (262_145, 1, 0), (262_145, 12, 0)])                              # one workgroup for all tensors of its rows
def test_reorder_tensors_of_long_rows_and_off_alignment(gx, n, words, offset):
    """Rows of every width of piece, so long that a workgroup moves them one by one, and tensors that begin off the
    boundary that the widest pieces ask for (``offset`` words into their storage)."""
    from raygaussx_amd.reordering import reorder_tensors
    gen = torch.Generator(gx.DEV).manual_seed(n + words)
    store = torch.randint(-2 ** 31, 2 ** 31 - 1, (n * words + offset,), dtype=torch.int32, device=gx.DEV, generator=gen)
    t = store[offset:].view(n, words)
    assert t.data_ptr() % 16 == 4 * offset
    order = torch.randperm(n, device=gx.DEV, generator=gen)
    _step(f"gather {n} rows of {words} words at {offset}")
    plain = torch.arange(n, device=gx.DEV, dtype=torch.float32)
    got, second = reorder_tensors(order, [t, plain])
    assert torch.equal(got, t[order]) and torch.equal(second, plain[order])


@pytest.mark.parametrize("n", [262_143, 262_144, 262_145, 300_031])
@pytest.mark.parametrize("words,odd", [
    ((3, 4, 3, 1, 3, 4, 3, 1, 3, 4, 3, 1), None),      # the short tensors of a cloud: one word more than a record holds
    ((8, 8, 8, 8, 2, 9, 7), None),                     # a full record, a second one, and a row too long for either
    ((1,) * 34, None), ((5, 12), None), ((6, 3, 2), 1)])   # more tensors than a record; one short alone; one off a 16-byte boundary
def test_reorder_tensors_of_many_short_rows(gx, n, words, odd):
    """Short rows put together in records: record sizes, what is left over, numbers of rows around the tile of 128 and the
    line from which on it is done."""
    from raygaussx_amd.reordering import reorder_tensors
    gen = torch.Generator(gx.DEV).manual_seed(n)
    tensors = []
    for i, w in enumerate(words):
        off = 1 if i == odd else 0
        tensors.append(torch.randint(-2 ** 31, 2 ** 31 - 1, (n * w + off,), dtype=torch.int32, device=gx.DEV, generator=gen)[off:].view(n, w))
    order = torch.randperm(n, device=gx.DEV, generator=gen)
    _step(f"short rows n={n} words={words}")
    for got, src in zip(reorder_tensors(order, tensors), tensors):
        assert torch.equal(got, src[order])


def test_reorder_tensors_without_room_for_its_records(gx, monkeypatch):
    """The records in which short rows are put together are a matter of speed: with no memory left for them the gather goes without."""
    from raygaussx_amd.reordering import reorder_tensors
    n = 262_144
    gen = torch.Generator(gx.DEV).manual_seed(4)
    tensors = [torch.randint(-2 ** 31, 2 ** 31 - 1, (n, w), dtype=torch.int32, device=gx.DEV, generator=gen) for w in (3, 4, 3, 1, 48)]
    order = torch.randperm(n, device=gx.DEV, generator=gen)
    empty, refused = torch.empty, []

    def no_room(*size, **kw):
        if kw.get("dtype") == torch.uint8:
            refused.append(size)
            raise torch.cuda.OutOfMemoryError("no room")
        return empty(*size, **kw)
    monkeypatch.setattr(torch, "empty", no_room)
    _step("short rows without room for records")
    got = reorder_tensors(order, tensors)
    monkeypatch.undo()
    assert refused == [(n * 128,)]
    for a, src in zip(got, tensors):
        assert torch.equal(a, src[order])


def test_reference_style_inference_loop_reuses_the_tree(gx, orc, c0):
    """scripts/test.py:50-126 pattern: boxes -> one acceleration structure -> several cameras."""
    from raygaussx_amd import optix_utils as u_ox
    from raygaussx_amd.render_optix import compute_rgb
    sc, _, cfg = c0
    d = gx.to_dev(sc)
    ctx = u_ox.create_context(None)
    module = u_ox.create_module(ctx, None, "test")
    pipeline = u_ox.create_pipeline(ctx, u_ox.create_program_groups(ctx, module), None)
    L1, L2, L3 = u_ox.quaternion_to_rotation(d["quaternions"])
    boxes = u_ox.compute_ellipsoids_bbox(d["positions"], d["scales"], L1, L2, L3, d["densities"])
    gas = u_ox.create_acceleration_structure(ctx, boxes)
    bb_min, bb_max = boxes[:, :3].min(0).values, boxes[:, 3:].max(0).values
    for idx in (0, 3):
        _step(f"inference camera {idx}")
        cam = scenes.make_camera(1, idx, width=64, height=48)
        rgb = compute_rgb(cam.camera_center, d["positions"], d["color_features"], None, None, None, 0, 3)
        img = u_ox.launch_pipeline_test(pipeline, None, gas, bb_min, bb_max, cfg["dt_step"], False, cam.to(gx.DEV),
                                        d["densities"], rgb, d["positions"], d["scales"], d["quaternions"],
                                        max_prim_slice=2048)
        want, _, _ = orc.render_forward(sc, cam, cfg["dt_step"], False, 2048)
        # boxes from the legacy torch routine differ from the canonical ones by rounding, so the scene
        # box (hence texit) may differ in the last ulp; colours still agree to tolerance
        assert np.abs(img.cpu().numpy() - want).max() <= IMG_TOL


def test_reduce_supersampling_clip_and_quantise_bit_exact(gx, orc):
    """The inference loop's image epilogue against the oracle's restatement: floats equal bit for
    bit (same summation order), clip and uint8(255 x) as numpy computes them."""
    from raygaussx_amd.general_utils import reduce_supersampling
    rng = np.random.default_rng(4)
    for W, H, f in ((33, 21, (1, 1)), (33, 21, (2, 1)), (16, 9, (2, 2)), (5, 7, (3, 2)), (800, 800, (2, 2))):
        rays = (rng.random((W * f[0] * H * f[1], 3), dtype=np.float32) * 1.4 - 0.2).astype(np.float32)
        _step(f"reduce_supersampling {W}x{H} x{f}")
        t = torch.from_numpy(rays).to(gx.DEV)
        want = orc.reduce_supersampling(W, H, rays, f)
        got = reduce_supersampling(W, H, t, f).cpu().numpy()
        np.testing.assert_array_equal(got.view(np.uint32), want.view(np.uint32))
        clipped, q = reduce_supersampling(W, H, t, f, clip=True, to_uint8=True)
        np.testing.assert_array_equal(clipped.cpu().numpy(), want.clip(0, 1))
        np.testing.assert_array_equal(q.cpu().numpy(), np.uint8(255 * want.clip(0, 1)))


def test_viewer_frame_depth_and_strided_colours(gx, orc, c0):
    """The interactive viewer's two kernels: the march with uchar4 colours and expected depth
    (cuda_gui/gaussians_aabb.cu) against the oracle's restatement, and gui_sh's strided tensors
    against the plain colour evaluation of the coefficients and lobes it selects."""
    from raygaussx_amd import optix_utils as u_ox
    sc, cam, cfg = c0
    sc = dict(sc)
    sc["scales"] = sc["scales"] * 2.0
    img, st, ctx = orc.render_forward(sc, cam, cfg["dt_step"], False, cfg["max_prim_slice"], white_background=False)
    frame, depth, colors = orc.march_gui(ctx["cs"], ctx["ms"], ctx["bmin"], ctx["bmax"], ctx["prims"])
    d = gx.to_dev(sc)
    gas = u_ox.AccelerationStructure(4096, gx.DEV).build_from_gaussians(d["positions"], d["scales"], d["quaternions"],
                                                                         d["densities"])
    ps = u_ox.pack_prims(gas, ctx["eye"], d["positions"], d["scales"], d["quaternions"], d["densities"],
                         torch.from_numpy(ctx["rgb"]).to(gx.DEV))
    _step("viewer march")
    f_gpu, z_gpu = u_ox.march_viewer(gas, u_ox.camera_struct(cam), ps, cfg["dt_step"], False, cfg["max_prim_slice"])
    # the same launch with a statistics block runs the counting variant of the kernel: same frame
    st_v = u_ox.new_stats(gx.DEV)
    f_cnt, z_cnt = u_ox.march_viewer(gas, u_ox.camera_struct(cam), ps, cfg["dt_step"], False, cfg["max_prim_slice"], stats=st_v)
    assert torch.equal(f_cnt, f_gpu) and torch.equal(z_cnt, z_gpu) and u_ox.read_stats(st_v)["hit_pairs"] == st["hit_pairs"]
    f_gpu, z_gpu = f_gpu.cpu().numpy().reshape(-1, 4), z_gpu.cpu().numpy().reshape(-1)
    assert (depth > 0).sum() > 5000
    assert np.abs(z_gpu - depth).max() <= 1e-4 * depth.max()
    np.testing.assert_array_equal(z_gpu == 0, depth == 0)
    # colours agree to 1e-4, so a quantised channel may differ by one step where it sits on a boundary
    diff = np.abs(f_gpu.astype(np.int32) - frame.astype(np.int32))
    assert diff.max() <= 1 and (diff > 0).mean() < 0.02 and (f_gpu[:, 3] == 255).all()
    _step("viewer colours")
    rng = np.random.default_rng(6)
    n, kmax, gmax = 3000, 16, 4
    pos = rng.normal(size=(n, 3)).astype(np.float32)
    sh = (rng.normal(size=(n, 3, kmax)) * 0.2).astype(np.float32)
    sg = (rng.normal(size=(n, 3, gmax)) * 0.1).astype(np.float32)
    sharp = rng.uniform(0.5, 3, size=(n, gmax)).astype(np.float32)
    ax = rng.normal(size=(n, gmax, 3)).astype(np.float32)
    ax /= np.linalg.norm(ax, axis=2, keepdims=True)
    eye = np.array([0.3, -4.0, 1.0], np.float32)
    for deg, g in ((0, 0), (1, 2), (2, 4), (3, 1)):
        k = (deg + 1) ** 2
        want = orc.sh_forward(eye, pos, np.ascontiguousarray(sh[:, :, :k]),
                              *((np.ascontiguousarray(sg[:, :, :g]), np.ascontiguousarray(sharp[:, :g]),
                                 np.ascontiguousarray(ax[:, :g])) if g else (None, None, None)))
        got = u_ox.sh_viewer(eye, *[torch.from_numpy(a).to(gx.DEV) for a in (pos, sh, sg, sharp, ax)], g, deg, kmax, gmax)
        np.testing.assert_allclose(got.cpu().numpy(), want, rtol=2e-5, atol=2e-6)


def test_dist2_knn3_bit_exact(gx, orc):
    """distCUDA2: exact three-nearest-neighbour mean, so equal to the oracle's brute force bit for
    bit, for clustered points, duplicates, points on a plane and sizes around the box sizes."""
    from raygaussx_amd.simple_knn import distCUDA2
    rng = np.random.default_rng(9)
    for n in (1, 2, 3, 4, 255, 257, 20_000):
        _step(f"distCUDA2 n={n}")
        p = rng.normal(size=(n, 3)).astype(np.float32)
        if n == 20_000:
            p[:5000] = p[:5000] * 0.01 + 3.0     # a dense cluster
            p[5000:5100] = p[5000]               # a hundred copies of one point
            p[6000:9000, 2] = 0.5                # a plane
        got = distCUDA2(torch.from_numpy(p).to(gx.DEV)).cpu().numpy()
        np.testing.assert_array_equal(got.view(np.uint32), orc.dist2_knn3(p).view(np.uint32))
    _step("distCUDA2 n=1M")                      # full size: against a k-d tree on a sample
    from scipy.spatial import cKDTree
    p = scenes.scene_to_numpy(scenes.make_scene(4, n=1_000_000))["positions"]
    got = distCUDA2(torch.from_numpy(p).to(gx.DEV)).cpu().numpy()
    ids = rng.choice(1_000_000, 2000, replace=False)
    d, _ = cKDTree(p.astype(np.float64)).query(p[ids].astype(np.float64), k=4)
    np.testing.assert_allclose(got[ids], (d[:, 1:] ** 2).mean(1), rtol=1e-5)


@pytest.mark.parametrize("n", [15, 16, 17, 63, 64, 65, 1023, 1024, 1025, 65_535, 65_536, 65_537])
def test_dist2_knn3_at_the_sizes_of_its_boxes(gx, orc, n):
    """Either side of a leaf, a wavefront, a box and a box of boxes."""
    from raygaussx_amd.simple_knn import distCUDA2
    p = np.random.default_rng(n).normal(size=(n, 3)).astype(np.float32)
    p[n // 2:] *= 30.0
    _step(f"distCUDA2 n={n}")
    got = distCUDA2(torch.from_numpy(p).to(gx.DEV)).cpu().numpy()
    np.testing.assert_array_equal(got.view(np.uint32), orc.dist2_knn3(p).view(np.uint32))


@pytest.mark.parametrize("n", [65_535, 65_536, 65_537, 262_143, 262_144, 262_145, 1_048_576, 1_048_577])
def test_dist2_knn3_with_any_number_of_lanes_per_point(gx, n):
    """Either side of the sizes at which the search changes its number of lanes per point: the first 9 001 points, with a nan and an
    outlier among them, are far from all others, so their distances are those of the small cloud alone, bit for bit."""
    from raygaussx_amd.simple_knn import distCUDA2
    rng = np.random.default_rng(n)
    near = rng.normal(size=(9001, 3)).astype(np.float32)
    near[5] = np.nan
    near[17] = (40.0, 0.0, 0.0)
    far = (rng.normal(size=(n - 9001, 3)) + np.array([1000.0, 0.0, 0.0])).astype(np.float32)
    _step(f"knn lanes n={n}")
    small = distCUDA2(torch.from_numpy(near).to(gx.DEV)).cpu().numpy()
    got = distCUDA2(torch.from_numpy(np.concatenate([near, far])).to(gx.DEV)).cpu().numpy()
    np.testing.assert_array_equal(got[:9001], small)
    assert np.isfinite(got[9001:]).all()


@pytest.mark.parametrize("n", [7, 8, 9, 511, 512, 513, 8192, 8193, 32_767, 32_768, 32_769])
def test_dist2_knn3_at_the_sizes_of_leaves_and_boxes(gx, orc, n):
    """Either side of a leaf of eight, a box of 64 leaves, a box of 64 boxes and the sort in one workgroup; half of the points far out and
    sparse, so that the runs between the two halves have many boxes open at first."""
    from raygaussx_amd.simple_knn import distCUDA2
    rng = np.random.default_rng(n)
    p = rng.normal(size=(n, 3)).astype(np.float32)
    p[n // 2:] *= (rng.uniform(10.0, 50.0, size=(n - n // 2, 1)) / np.linalg.norm(p[n // 2:], axis=1, keepdims=True)).astype(np.float32)
    _step(f"distCUDA2 n={n}")
    got = distCUDA2(torch.from_numpy(p).to(gx.DEV)).cpu().numpy()
    np.testing.assert_array_equal(got.view(np.uint32), orc.dist2_knn3(p).view(np.uint32))


@pytest.mark.parametrize("n", [524_287, 524_288, 524_289])
def test_dist2_knn3_where_its_grid_changes(gx, n):
    """Either side of the size from which the curve's grid has ten bits per axis and a point two lanes, against a k-d tree: squared distances are
    rounded five times, 3e-7 of themselves, and their mean three times."""
    from scipy.spatial import cKDTree
    from raygaussx_amd.simple_knn import distCUDA2
    rng = np.random.default_rng(n)
    p = rng.normal(size=(n, 3)).astype(np.float32)
    p[: n // 3] *= 20.0
    p[5] = p[6] = p[7] = p[8]
    _step(f"distCUDA2 n={n}")
    got = distCUDA2(torch.from_numpy(p).to(gx.DEV)).cpu().numpy()
    ids = np.concatenate([[5, n - 1], rng.choice(n, 3000, replace=False)])
    d, _ = cKDTree(p.astype(np.float64)).query(p[ids].astype(np.float64), k=4)
    np.testing.assert_allclose(got[ids], (d[:, 1:] ** 2).mean(1), rtol=1e-6)


def _crowded_cloud(kind, n, rng):
    if kind == "line":
        return (rng.uniform(-1.0, 1.0, size=(n, 1)) * [1.0, 0.7, 0.4] + rng.normal(size=(n, 3)) * 1e-4).astype(np.float32)
    if kind == "one place":
        return np.full((n, 3), 0.3, np.float32)
    if kind == "lattice":
        return (rng.integers(0, 12, size=(n, 3)) * 0.25).astype(np.float32)
    count, width = {"3 clumps": (3, 0.002), "10 clumps": (10, 0.005), "clumps and nan": (3, 0.002)}[kind]
    p = (rng.uniform(-1.0, 1.0, size=(count, 3))[rng.integers(0, count, n)] + rng.normal(size=(n, 3)) * width).astype(np.float32)
    if kind == "clumps and nan":
        p[3::50, 1] = np.nan
        p[5::60, 0] = np.inf
        p[n // 2: n // 2 + 700] = np.nan
    return p


@pytest.mark.parametrize("n", [1025, 8192, 8193, 16_385, 32_769])                # from 8 193 on a cloud can be crowded; boxes of 512
@pytest.mark.parametrize("kind", ["3 clumps", "10 clumps", "clumps and nan", "line", "one place", "lattice"])
def test_dist2_knn3_of_crowded_clouds(gx, orc, kind, n):
    """Clouds of which a cell of the first grid holds hundreds: sorted by quantiles, and box by box."""
    from raygaussx_amd.simple_knn import distCUDA2
    p = _crowded_cloud(kind, n, np.random.default_rng(n))
    _step(f"distCUDA2, {kind} n={n}")
    got = distCUDA2(torch.from_numpy(p).to(gx.DEV)).cpu().numpy()
    np.testing.assert_array_equal(got.view(np.uint32), orc.dist2_knn3(p).view(np.uint32))


def test_dist2_knn3_of_a_large_crowded_cloud(gx):
    """Ten bits per axis; against a k-d tree, with the tolerance of test_dist2_knn3_where_its_grid_changes."""
    from scipy.spatial import cKDTree
    from raygaussx_amd.simple_knn import distCUDA2
    n = 524_289
    p = _crowded_cloud("10 clumps", n, np.random.default_rng(3))
    _step("distCUDA2, ten clumps")
    got = distCUDA2(torch.from_numpy(p).to(gx.DEV)).cpu().numpy()
    ids = np.random.default_rng(4).choice(n, 3000, replace=False)
    d, _ = cKDTree(p.astype(np.float64)).query(p[ids].astype(np.float64), k=4)
    np.testing.assert_allclose(got[ids], (d[:, 1:] ** 2).mean(1), rtol=1e-6)


@pytest.mark.parametrize("n", [54_000, 300_000])
def test_dist2_knn3_is_not_slow_where_points_are_crowded(gx, n):
    """Three tight clumps cost at most three times what a ball of as many points costs (measured 1.3; by one grid for all clouds 7 and 89 times), the best
    of eight calls of each."""
    from raygaussx_amd.simple_knn import distCUDA2
    rng = np.random.default_rng(1)
    v = rng.normal(size=(n, 3))
    ball = torch.from_numpy((v / np.linalg.norm(v, axis=1, keepdims=True) * np.cbrt(rng.uniform(size=(n, 1)))).astype(np.float32)).to(gx.DEV)
    clumps = torch.from_numpy(_crowded_cloud("3 clumps", n, rng)).to(gx.DEV)
    _step(f"distCUDA2, times n={n}")

    def best(p):
        distCUDA2(p)
        times = []
        for _ in range(8):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            distCUDA2(p)
            b.record()
            b.synchronize()
            times.append(a.elapsed_time(b))
        return min(times)

    assert best(clumps) <= 3.0 * best(ball)


@pytest.mark.parametrize("kind", ["outliers", "two clumps", "nan", "inf", "nan and inf", "all nan", "huge"])
def test_dist2_knn3_of_clouds_that_the_curve_does_not_sort(gx, orc, kind):
    """A few far points leave nearly all the others in one or two cells of the Morton grid, in whose order they say nothing of
    where they lie.  A point with a coordinate that is no number, or infinite, is no one's neighbour and has none."""
    from raygaussx_amd.simple_knn import distCUDA2
    rng = np.random.default_rng(5)
    n = 6000
    p = rng.normal(size=(n, 3)).astype(np.float32)
    if kind == "outliers":
        p[::900] *= 1e5
    elif kind == "two clumps":
        p *= 1e-3
        p[1::2] += 1e4
    elif kind == "all nan":
        p[:] = np.nan
    elif kind == "huge":
        p[:10] *= 1e30                                 # squared distances beyond the float range
    if "nan" in kind and kind != "all nan":
        p[3::50, 1] = np.nan
        p[64:128] = np.nan                             # a whole wavefront's worth
    if "inf" in kind:
        p[7::40, 2] = np.inf
        p[9::71, 0] = -np.inf
        p[200:264, 0] = np.inf
    _step(f"distCUDA2, {kind}")
    got = distCUDA2(torch.from_numpy(p).to(gx.DEV)).cpu().numpy()
    ref = orc.dist2_knn3(p)
    assert (np.isfinite(ref).all(), np.isfinite(ref).any()) == (kind in ("outliers", "two clumps"), kind != "all nan")
    np.testing.assert_array_equal(got.view(np.uint32), ref.view(np.uint32))


def test_training_loop_as_the_reference_writes_it_reduces_the_loss(gx):
    """scripts/train.py:101-148 in miniature: OptiX set-up calls, RenderOptixSettings with the
    reference's positional arguments, RenderOptixFunction.apply on activated parameters, an L1 loss,
    Adam.  A perturbed copy of a scene must move back towards the images of the original."""
    from raygaussx_amd import optix_utils as u_ox
    from raygaussx_amd.render_optix import RenderOptixFunction, RenderOptixSettings
    torch.manual_seed(0)
    truth = {k: v.to(gx.DEV) for k, v in scenes.make_scene(0, n=1500, sh_degree=1, seed=31).items()}
    truth["scales"] = truth["scales"] * 2.0
    cams = [scenes.make_camera(1, i, width=48, height=48).to(gx.DEV) for i in (0, 17, 43, 71)]
    ctx = u_ox.create_context(log=None)
    mod_f, mod_b = u_ox.create_module(ctx, None, stage="forward"), u_ox.create_module(ctx, None, stage="backward")
    pg_f, pg_b = u_ox.create_program_groups(ctx, mod_f), u_ox.create_program_groups(ctx, mod_b)
    pl_f, pl_b = u_ox.create_pipeline(ctx, pg_f, None), u_ox.create_pipeline(ctx, pg_b, None)
    empty = (torch.zeros(1500, 3, 0, device=gx.DEV), torch.zeros(1500, 0, device=gx.DEV), torch.zeros(1500, 0, 3, device=gx.DEV))

    def render(p, cam):
        settings = RenderOptixSettings(ctx, False, None, pg_f, pl_f, pg_b, pl_b, 0.005, False, cam, 512, 0, 0, 0, 0,
                                       (1, 1), True, None)
        quat = torch.nn.functional.normalize(p["quaternions"], dim=1)
        return RenderOptixFunction.apply(p["positions"], torch.exp(p["log_scales"]), quat, p["densities"],
                                         p["color_features"], *empty, settings)

    with torch.no_grad():
        t = dict(truth, log_scales=truth["scales"].log())
        targets = [render(t, c) for c in cams]
    params = {"positions": truth["positions"] + 0.01 * torch.randn_like(truth["positions"]),
              "log_scales": truth["scales"].log() + 0.1 * torch.randn_like(truth["scales"]),
              "quaternions": truth["quaternions"] + 0.05 * torch.randn_like(truth["quaternions"]),
              "densities": truth["densities"] * (1 + 0.2 * torch.randn_like(truth["densities"])).clamp(min=0.3),
              "color_features": truth["color_features"] + 0.1 * torch.randn_like(truth["color_features"])}
    params = {k: v.clone().requires_grad_(True) for k, v in params.items()}
    opt = torch.optim.Adam([{"params": [params["positions"]], "lr": 2e-4}, {"params": [params["log_scales"]], "lr": 5e-3},
                            {"params": [params["quaternions"]], "lr": 2e-3}, {"params": [params["densities"]], "lr": 1e-2},
                            {"params": [params["color_features"]], "lr": 5e-3}])
    _step("60 Adam steps")
    losses = []
    for it in range(60):
        cam, target = cams[it % 4], targets[it % 4]
        loss = (render(params, cam) - target).abs().mean()
        opt.zero_grad()
        loss.backward()
        opt.step()
        losses.append(loss.item())
        assert all(torch.isfinite(p.grad).all() for p in params.values())
    first, last = np.mean(losses[:4]), np.mean(losses[-4:])
    assert last < 0.6 * first, (first, last)


def test_direct_ctypes_binding_matches_the_python_mirror(gx, c0):
    """The stand-alone ctypes stub a maintainer would write (no raygaussx_amd imports in the call
    path): build, colour, pack, forward with a record, backward, colour gradient -- equal to what
    RenderOptixFunction returns for the same inputs."""
    import ctypes as C
    from raygaussx_amd import _lib
    lib = C.CDLL(_lib.LIB_PATH)

    class RgxCamera(C.Structure):
        _fields_ = [("eye", C.c_float * 3), ("u", C.c_float * 3), ("v", C.c_float * 3), ("w", C.c_float * 3),
                    ("tan_half_fov_x", C.c_float), ("tan_half_fov_y", C.c_float),
                    ("principal_x", C.c_float), ("principal_y", C.c_float),
                    ("width", C.c_int32), ("height", C.c_int32)]

    class RgxMarch(C.Structure):
        _fields_ = [("dt_step", C.c_float), ("dynamic_sampling", C.c_int32), ("max_prim_slice", C.c_int32),
                    ("white_background", C.c_int32), ("t_eps", C.c_float), ("record_format", C.c_int32)]

    def p(t):
        return C.c_void_p(t.data_ptr())

    def ws(fn, *a):
        n = C.c_size_t()
        assert fn(*a, C.byref(n)) == 0
        return torch.empty(n.value, dtype=torch.uint8, device=gx.DEV)

    sc, camera, cfg = c0
    d = gx.to_dev(sc)
    pos, scale, quat, dens, sh = (d[k] for k in ("positions", "scales", "quaternions", "densities", "color_features"))
    N, W, H = pos.shape[0], camera.image_width, camera.image_height
    rot = camera.world_view_transform[:3, :3]
    import math
    cam = RgxCamera((C.c_float * 3)(*camera.camera_center.tolist()), (C.c_float * 3)(*rot[:, 0].tolist()),
                    (C.c_float * 3)(*rot[:, 1].tolist()), (C.c_float * 3)(*rot[:, 2].tolist()),
                    math.tan(camera.FoVx / 2), math.tan(camera.FoVy / 2), camera.Px, camera.Py, W, H)
    march = RgxMarch(cfg["dt_step"], 0, cfg["max_prim_slice"], 1, 1e-3)
    s = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    bvh = ws(lib.rgx_build_workspace_bytes, C.c_int64(N))
    mws = ws(lib.rgx_march_workspace_bytes, C.c_int64(N), C.c_int64(W * H), C.c_int32(cfg["max_prim_slice"]))
    rec = ws(lib.rgx_march_records_bytes, C.c_int32(W), C.c_int32(H), C.c_int32(16384 + 64 * 8192))
    eye = (C.c_float * 3)(*camera.camera_center.tolist())
    f = dict(dtype=torch.float32, device=gx.DEV)
    rgb, prims, img = torch.empty(N, 3, **f), torch.empty(N, 16, **f), torch.empty(W * H, 3, **f)
    dimg = torch.from_numpy(np.random.default_rng(2).normal(size=(W * H, 3)).astype(np.float32)).to(gx.DEV)
    ddens, drgb, dpos, dscale, dquat = (torch.empty(N, **f), torch.empty(N, 3, **f), torch.empty(N, 3, **f),
                                        torch.empty(N, 3, **f), torch.empty(N, 4, **f))
    dsh, dpos_dir = torch.empty_like(sh), torch.empty(N, 3, **f)
    _step("direct ctypes calls")
    assert lib.rgx_build(p(pos), p(scale), p(quat), p(dens), C.c_int64(N), C.c_float(0.1), p(bvh), C.c_size_t(bvh.numel()), s) == 0
    assert lib.rgx_sh_forward(eye, p(pos), p(sh), None, None, None, 0, 3, C.c_int64(N), p(rgb), s) == 0
    assert lib.rgx_pack_prims(p(bvh), eye, p(pos), p(scale), p(quat), p(dens), p(rgb), C.c_int64(N), C.c_float(0.1), p(prims), s) == 0
    assert lib.rgx_march_forward(p(bvh), C.byref(cam), C.byref(march), p(prims), C.c_int64(N), p(img),
                                 p(mws), C.c_size_t(mws.numel()), p(rec), C.c_size_t(rec.numel()), None, s) == 0
    assert lib.rgx_march_backward(p(bvh), C.byref(cam), C.byref(march), p(prims), C.c_int64(N), p(img), p(dimg),
                                  p(ddens), p(drgb), p(dpos), p(dscale), p(dquat), p(mws), C.c_size_t(mws.numel()),
                                  p(rec), C.c_size_t(rec.numel()), None, s) == 0
    assert lib.rgx_sh_backward(eye, p(pos), p(sh), None, None, None, 0, 3, C.c_int64(N), p(drgb),
                               p(dsh), p(dpos_dir), None, None, None, s) == 0
    dpos += dpos_dir
    torch.cuda.synchronize()
    # a march workspace with room for the gradient block only (sized for another image, say): the replay
    # then takes the tiles in launch order instead of heaviest first, and returns the same gradients
    _step("direct ctypes calls, workspace without room for a tile order")
    small = (N * 64 + 255) // 256 * 256
    ddens2, dscale2 = torch.empty_like(ddens), torch.empty_like(dscale)
    assert lib.rgx_march_backward(p(bvh), C.byref(cam), C.byref(march), p(prims), C.c_int64(N), p(img), p(dimg),
                                  p(ddens2), p(drgb), p(dpos_dir), p(dscale2), p(dquat), p(mws), C.c_size_t(small),
                                  p(rec), C.c_size_t(rec.numel()), None, s) == 0
    torch.cuda.synchronize()
    for a, b in ((ddens2, ddens), (dscale2, dscale)):
        cos, rel = gx.cos_rel(a.cpu().numpy(), b.cpu().numpy())
        assert cos >= 1 - 1e-6 and rel <= 1e-5, (cos, rel)
    assert lib.rgx_march_backward(p(bvh), C.byref(cam), C.byref(march), p(prims), C.c_int64(N), p(img), p(dimg),
                                  p(ddens2), p(drgb), p(dpos_dir), p(dscale2), p(dquat), p(mws), C.c_size_t(small - 256),
                                  p(rec), C.c_size_t(rec.numel()), None, s) == -2   # RGX_EWORKSPACE
    ref = gx.gpu_render(sc, camera, cfg, want_grad=dimg.cpu().numpy(), stats=False)
    np.testing.assert_array_equal(img.cpu().numpy(), ref["image"])
    for name, got in (("positions", dpos), ("scales", dscale), ("quaternions", dquat), ("densities", ddens), ("color_features", dsh)):
        cos, rel = gx.cos_rel(got.cpu().numpy(), ref["grads"][name])
        assert cos >= 1 - 1e-6 and rel <= 1e-4, (name, cos, rel)


def test_empty_cloud_and_one_pixel_image(gx):
    """No Gaussians at all renders the background and returns empty gradients; a 1x1 image works."""
    cam = scenes.make_camera(0, 0, width=16, height=8)
    cfg = dict(dt_step=0.0025, dynamic_sampling=False, max_prim_slice=64)
    empty = {k: v[:0].copy() for k, v in scenes.scene_to_numpy(scenes.make_scene(0, n=4, sh_degree=1, seed=1)).items()
             if k in ("positions", "scales", "quaternions", "densities", "color_features")}
    _step("empty cloud")
    out = gx.gpu_render(empty, cam, cfg, want_grad=np.ones((16 * 8, 3), np.float32))
    np.testing.assert_array_equal(out["image"], 1.0)
    assert out["grads"]["positions"].shape == (0, 3) and out["grads"]["color_features"].shape == (0, 3, 4)
    _step("1x1 image")
    sc = scenes.scene_to_numpy(scenes.make_scene(0, n=300, sh_degree=0, seed=2))
    sc["scales"] = sc["scales"] * 3
    cam1 = scenes.make_camera(0, 0, width=1, height=1)
    out = gx.gpu_render(sc, cam1, cfg, want_grad=np.ones((1, 3), np.float32))
    assert out["image"].shape == (1, 3) and np.isfinite(out["image"]).all()
    assert out["stats_fwd"]["hit_pairs"] == out["stats_bwd"]["hit_pairs"] > 0
    assert np.isfinite(out["grads"]["positions"]).all() and np.abs(out["grads"]["positions"]).sum() > 0


def test_plain_division_and_square_root_are_correctly_rounded(gx):
    """The hit predicate's quotients and square root are formed without the compiler's handling of
    extreme exponents wherever a Gaussian's scales and distance allow (which is everywhere in
    practice).  Inside the granted range the short forms must equal `/` and sqrtf() in every bit:
    8 million operand pairs with exponents over the whole range and mantissas that include the
    all-zeros / all-ones patterns and near-ties."""
    import ctypes as C
    from raygaussx_amd import _lib
    rng = np.random.default_rng(31)
    n = 1 << 23

    def operands():
        mant = rng.integers(0, 1 << 23, n, dtype=np.uint32)
        special = rng.integers(0, 8, n)
        mant = np.where(special == 0, 0, mant)
        mant = np.where(special == 1, (1 << 23) - 1, mant)
        mant = np.where(special == 2, mant & 0x7, mant)              # just above a power of two
        mant = np.where(special == 3, mant | 0x7FFFF8, mant)         # just below one
        expo = rng.integers(127 - 46, 127 + 46, n, dtype=np.uint32)  # 2^-46 <= |v| < 2^46
        sign = rng.integers(0, 2, n, dtype=np.uint32)
        return ((sign << 31) | (expo << 23) | mant.astype(np.uint32)).astype(np.uint32).view(np.float32)

    a, b = torch.from_numpy(operands()).to(gx.DEV), torch.from_numpy(operands()).to(gx.DEV)
    bad = torch.zeros(1, dtype=torch.int32, device=gx.DEV)
    _step("plain division / square root against the full sequences")
    _lib.check(_lib.lib().rgx_check_plain_arith(_lib.ptr(a), _lib.ptr(b), C.c_int64(n), _lib.ptr(bad), _lib.stream()))
    torch.cuda.synchronize()
    assert int(bad.item()) == 0
    # and the check itself can fail: far outside the range the short division loses its footing
    tiny = torch.full((1024,), 1e-38, dtype=torch.float32, device=gx.DEV)
    huge = torch.full((1024,), 3e38, dtype=torch.float32, device=gx.DEV)
    _lib.check(_lib.lib().rgx_check_plain_arith(_lib.ptr(tiny), _lib.ptr(huge), C.c_int64(1024), _lib.ptr(bad), _lib.stream()))
    torch.cuda.synchronize()
    assert int(bad.item()) > 0


def test_seeded_sweep_over_scenes_image_shapes_and_settings(gx, orc):
    """Twenty seeded draws of scene generator, Gaussian count, scale factor, SH degree, camera, ragged
    image shape, background, max_prim_slice and record size against the oracle: counters equal and
    the gates held wherever no hit list was cut (a cut list keeps different hits on the two sides)."""
    rng = np.random.default_rng(2024)
    compared = 0
    for case in range(20):
        config = int(rng.choice([0, 1, 2, 4]))
        n = int(rng.choice([300, 2000, 8000, 25000]))
        mult = float(rng.choice([0.5, 1.0, 2.0, 4.0, 8.0]))
        w, h = int(rng.integers(9, 140)), int(rng.integers(9, 120))
        cap = int(rng.choice([16, 64, 2048]))
        white = bool(rng.integers(0, 2))
        words = [None, 16384, 16384 + 2 * 8192, 2048][int(rng.integers(0, 4))]
        sc = scenes.scene_to_numpy(scenes.make_scene(config, n=n, sh_degree=int(rng.integers(0, 4)), seed=int(rng.integers(0, 1000))))
        sc = {k: sc[k] for k in ("positions", "scales", "quaternions", "densities", "color_features")}
        sc["scales"] = sc["scales"] * mult
        cam = scenes.make_camera(config, int(rng.integers(0, 5)), width=w, height=h)
        cfg = dict(scenes.CONFIGS[config], dynamic_sampling=False, max_prim_slice=cap)
        img, st, ctx = orc.render_forward(sc, cam, cfg["dt_step"], False, cap, white_background=white, t_eps=cfg.get("t_eps", 1e-3))
        dloss = rng.normal(size=img.shape).astype(np.float32)
        og, _ = orc.render_backward(sc, ctx, img, dloss)
        _step(f"sweep case {case}: config {config}, n {n}, scales x{mult}, {w}x{h}, cap {cap}, white {white}, record {words}")
        out = gx.gpu_render(sc, cam, cfg, white=white, want_grad=dloss, rec_tile_words=words)
        assert (out["stats_fwd"]["overflow_rays"] > 0) == (st["overflow_rays"] > 0)
        if st["overflow_rays"]:
            continue
        for k in ("hit_pairs", "slabs", "empty_slabs", "rays_hit"):
            assert out["stats_fwd"][k] == st[k], (case, k)
        assert np.abs(out["image"] - img).max() <= IMG_TOL
        _check_grads(gx, out["grads"], og)
        # the same case through the kernels without counters (what a training loop launches)
        out = gx.gpu_render(sc, cam, cfg, white=white, want_grad=dloss, rec_tile_words=words, stats=False)
        assert np.abs(out["image"] - img).max() <= IMG_TOL
        _check_grads(gx, out["grads"], og)
        compared += 1
    assert compared >= 10


def test_views_in_flight_on_two_streams_equal_the_views_one_after_another(gx):
    """A training loop that accumulates gradients over several views (scripts/train.py:119-148 with
    gradient accumulation) may keep two views in flight, each on a stream of its own: the library's
    scratch memory is per stream and its records are per call.  Images must be those of the serial
    loop in every bit, and the accumulated gradients equal up to the order of the atomic adds."""
    from raygaussx_amd.render_optix import RenderOptixFunction, default_settings
    names = ("positions", "scales", "quaternions", "densities", "color_features")
    scene = {k: v.to(gx.DEV) for k, v in scenes.make_scene(1, n=40000, seed=5).items()}
    scene["scales"] = scene["scales"] * 3.0
    cams = [scenes.make_camera(1, i, width=200, height=152).to(gx.DEV) for i in (0, 9, 31, 58, 77, 90)]
    targets = [torch.rand(200 * 152, 3, device=gx.DEV, generator=torch.Generator(gx.DEV).manual_seed(i)) for i in range(len(cams))]
    empty = (torch.zeros(40000, 3, 0, device=gx.DEV), torch.zeros(40000, 0, device=gx.DEV), torch.zeros(40000, 0, 3, device=gx.DEV))

    def loop(streams):
        params = [scene[k].clone().requires_grad_(True) for k in names]
        gas = [None] * len(streams)
        images = []
        torch.cuda.synchronize()
        for i, cam in enumerate(cams):
            k = i % len(streams)
            with torch.cuda.stream(streams[k]):
                s = default_settings(cam, 0.005, False, 512, gas=gas[k])
                img = RenderOptixFunction.apply(*params, *empty, s)
                gas[k] = s.gas
                ((img - targets[i]) ** 2).mean().backward()
                images.append(img.detach())
        torch.cuda.synchronize()
        return images, [p.grad.clone() for p in params]

    _step("six views, one stream")
    img1, g1 = loop([torch.cuda.current_stream(gx.DEV)])
    _step("six views, two in flight")
    img2, g2 = loop([torch.cuda.Stream(gx.DEV), torch.cuda.Stream(gx.DEV)])
    for a, b in zip(img1, img2):
        assert torch.equal(a, b)
    for k, a, b in zip(names, g1, g2):
        rel = float((a - b).norm() / a.norm())
        assert rel <= 1e-5, (k, rel)
        assert float(a.norm()) > 0


def test_a_tree_marked_current_is_not_rebuilt_and_gives_the_same_view(gx):
    """``settings.gas_is_current``: the views of one accumulation window share the Gaussians, so all
    but the first may skip the rebuild.  Same image and gradients, and no build launch."""
    from raygaussx_amd.render_optix import RenderOptixFunction, default_settings
    names = ("positions", "scales", "quaternions", "densities", "color_features")
    scene = {k: v.to(gx.DEV) for k, v in scenes.make_scene(0, n=6000, seed=3).items()}
    scene["scales"] = scene["scales"] * 2.0
    cam = scenes.make_camera(0, 0, width=96, height=80).to(gx.DEV)
    empty = (torch.zeros(6000, 3, 0, device=gx.DEV), torch.zeros(6000, 0, device=gx.DEV), torch.zeros(6000, 0, 3, device=gx.DEV))

    def view(gas, current, src=scene):
        params = [src[k].clone().requires_grad_(True) for k in names]
        s = default_settings(cam, 0.01, False, 512, gas=gas)
        s.gas_is_current = current
        img = RenderOptixFunction.apply(*params, *empty, s)
        (img ** 2).sum().backward()
        torch.cuda.synchronize()
        return img.detach(), [p.grad for p in params], s.gas

    _step("rebuilt, then reused")
    img_a, g_a, gas = view(None, False)
    img_b, g_b, gas_b = view(gas, True)
    assert gas_b is gas and torch.equal(img_a, img_b)
    for a, b in zip(g_a, g_b):
        assert float((a - b).norm() / a.norm()) <= 1e-5
    img_c, _, _ = view(None, True)      # nothing to reuse: built regardless of the flag
    assert torch.equal(img_a, img_c)
    from raygaussx_amd import _lib
    _lib.timing_enable(True)        # and the flag is honoured: no build launch for the reused view
    try:
        view(gas, True)
        torch.cuda.synchronize()
        assert _lib.timing_read()["build"][1] == 0
        view(gas, False)
        torch.cuda.synchronize()
        assert _lib.timing_read()["build"][1] == 1
    finally:
        _lib.timing_enable(False)


def test_off_centre_principal_point_and_rolled_camera(gx, orc):
    """COLMAP cameras carry a principal point away from the image centre (optix_utils.py:258-266 passes
    Px, Py on; gaussians_aabb.cu:200-206 shifts the pixel grid by them).  The tile frusta that cull the
    tree must follow that shift: counters, image and gradients against the oracle for a rolled camera
    with the principal point well off centre, looking past the scene's middle."""
    sc = scenes.scene_to_numpy(scenes.make_scene(0, n=5000, seed=17))
    sc = {k: sc[k] for k in ("positions", "scales", "quaternions", "densities", "color_features")}
    sc["scales"] = sc["scales"] * 2.0
    rng = np.random.default_rng(4)
    for px, py, up, target in ((0.31, 0.66, (0.3, -0.2, 1.0), (0.2, -0.1, 0.1)), (0.72, 0.4, (1.0, 0.1, 0.2), (-0.3, 0.2, 0.0))):
        cam = scenes.look_at_camera((2.1, -2.4, 1.7), target=target, up=up, fov_x_deg=52.0, width=150, height=90, px=px, py=py)
        cfg = dict(scenes.CONFIGS[0])
        img, st, ctx = orc.render_forward(sc, cam, cfg["dt_step"], False, cfg["max_prim_slice"], t_eps=cfg.get("t_eps", 1e-3))
        dloss = rng.normal(size=img.shape).astype(np.float32)
        og, _ = orc.render_backward(sc, ctx, img, dloss)
        _step(f"principal point ({px}, {py})")
        out = gx.gpu_render(sc, cam, cfg, want_grad=dloss)
        assert st["rays_hit"] > 5000 and st["overflow_rays"] == 0
        for k in ("hit_pairs", "slabs", "empty_slabs", "rays_hit"):
            assert out["stats_fwd"][k] == st[k], k
        assert np.abs(out["image"] - img).max() <= IMG_TOL
        _check_grads(gx, out["grads"], og)


def test_launch_faults_are_counted_without_a_statistics_block(gx):
    """A replay that cannot follow its record stops that tile and is counted in the march workspace
    whether or not the launch carries a statistics block (rgx_march_faults); clean launches count
    nothing.  The record is made unreadable on the host side of the test (a tile's `words used` cut
    short), so the replay runs out of items and leaves through its ordinary exit."""
    from raygaussx_amd import optix_utils as u_ox
    from raygaussx_amd.render_optix import compute_rgb
    n = 3000
    sc = gx.to_dev(scenes.scene_to_numpy(scenes.make_scene(0, n=n, sh_degree=0, seed=5)))
    cam = scenes.make_camera(0, 0, width=40, height=32)
    cs = u_ox.camera_struct(cam)
    gas = u_ox.AccelerationStructure(n, gx.DEV).build_from_gaussians(sc["positions"], sc["scales"] * 1.5, sc["quaternions"], sc["densities"])
    rgb = compute_rgb(cam.camera_center, sc["positions"], sc["color_features"], None, None, None, 0, 0)
    ps = u_ox.pack_prims(gas, cs, sc["positions"], sc["scales"] * 1.5, sc["quaternions"], sc["densities"], rgb)
    dloss = torch.from_numpy(np.random.default_rng(1).normal(size=(40 * 32, 3)).astype(np.float32)).to(gx.DEV)
    for words in (None, u_ox.REC_LIST_WORDS):
        rec = u_ox.new_records(cs, gx.DEV) if words is None else u_ox.new_records(cs, gx.DEV, tile_words=words)
        _step(f"clean forward + backward, record words {words}")
        img = u_ox.march_forward(gas, cs, ps, 0.004, False, 512, True, records=rec)
        clean = u_ox.march_backward(gas, cs, ps, img, dloss, 0.004, False, 512, True, records=rec)
        assert u_ox.march_faults(n, gx.DEV) == (0, 0)
        # cut two tiles' records short: their replays run out of items
        tile_words = u_ox.REC_LIST_WORDS
        view = rec[:20 * tile_words * 4].view(torch.int32).view(20, tile_words)
        a, b = (int(t) for t in torch.argsort(view[:, 1], descending=True)[:2])     # the two busiest tiles
        assert int(view[b, 1]) > 200
        view[a, 1] = 100
        view[b, 1] = 60
        _step("backward with two truncated tile records")
        img = u_ox.march_forward(gas, cs, ps, 0.004, False, 512, True)           # clears the counters
        got = u_ox.march_backward(gas, cs, ps, img, dloss, 0.004, False, 512, True, records=rec)
        lost, dropped = u_ox.march_faults(n, gx.DEV)
        assert lost == 2 and dropped == 0
        assert all(torch.isfinite(g).all() for g in got)
        # the other 18 tiles' gradients are there: the result stays close to the clean one
        cos, _ = gx.cos_rel(got[2].cpu().numpy(), clean[2].cpu().numpy())
        assert cos > 0.9


def test_deep_tree_of_coincident_and_nested_gaussians(gx, orc):
    """A tree far deeper than any ordinary scene gives: 1500 Gaussians sharing one centre (equal Morton
    keys, split by index alone) and a chain of Gaussians at 2^-i from it (keys that differ one bit level
    at a time).  The cooperative sweep's node stack has to take it without dropping a subtree: counters,
    image and gradients against the oracle, and no dropped-node count."""
    import ctypes as C
    from raygaussx_amd import _lib, optix_utils as u_ox
    rng = np.random.default_rng(12)
    base = scenes.scene_to_numpy(scenes.make_scene(0, n=2000, sh_degree=1, seed=8))
    sc = {k: base[k].copy() for k in ("positions", "scales", "quaternions", "densities", "color_features")}
    centre = np.array([0.11, -0.07, 0.05], np.float32)
    sc["positions"][:1500] = centre
    sc["scales"][:1500] = rng.uniform(0.03, 0.15, size=(1500, 3)).astype(np.float32)
    sc["densities"][:1500] = rng.uniform(0.2, 1.0, size=1500).astype(np.float32)
    for i in range(60):                       # a nested chain: each one half as far from the shared centre
        sc["positions"][1500 + i] = centre + np.float32(0.9) * np.float32(2.0) ** -i * np.array([1, 1, 1], np.float32)
        sc["scales"][1500 + i] = 0.04
    cam = scenes.make_camera(0, 0, width=24, height=24)
    cfg = dict(dt_step=0.0025, dynamic_sampling=False, max_prim_slice=4096)
    img, st, ctx = orc.render_forward(sc, cam, 0.0025, False, 4096)
    dloss = rng.normal(size=img.shape).astype(np.float32)
    og, _ = orc.render_backward(sc, ctx, img, dloss)
    assert st["overflow_rays"] == 0 and st["hit_pairs"] > 10000
    _step("deep tree: forward + backward")
    out = gx.gpu_render(sc, cam, cfg, want_grad=dloss)
    # how deep the tree really is: follow the parents of every node
    n = 2000
    lay = (C.c_size_t * 6)()
    _lib.check(_lib.lib().rgx_build_layout(C.c_int64(n), lay))
    parent = out["settings"].gas.ws[lay[3]:lay[3] + (2 * n - 1) * 4].view(torch.int32).cpu().numpy()
    depth, cur = 0, np.arange(2 * n - 1)
    while (cur >= 0).any():
        cur = np.where(cur >= 0, parent[np.maximum(cur, 0)], -1)
        depth += 1
    print("tree depth", depth - 1, flush=True)
    assert depth - 1 >= 30
    for k in ("hit_pairs", "slabs", "empty_slabs", "rays_hit"):
        assert out["stats_fwd"][k] == st[k], k
    assert np.abs(out["image"] - img).max() <= IMG_TOL
    _check_grads(gx, out["grads"], og)
    assert u_ox.march_faults(n, gx.DEV) == (0, 0)
    assert u_ox.FAULTS_SEEN["sweep_dropped"] == 0


def test_update_acceleration_structure_refits_the_tree(gx, orc):
    """update_acceleration_structure (optix_utils.py:144-146): new boxes into an existing tree.  The
    refitted tree keeps the old shape, so it culls worse, but every query stays exact: after the
    Gaussians moved, image and counters equal those of the oracle on the moved scene, and the
    refitted workspace passes the same host-side tree check as a fresh build."""
    from raygaussx_amd import optix_utils as u_ox
    from raygaussx_amd.render_optix import compute_rgb
    from test_gpu_fullsize import _check_tree, _read_tree
    sc = scenes.scene_to_numpy(scenes.make_scene(0, n=6000, sh_degree=1, seed=14))
    sc["scales"] = sc["scales"] * 2.0
    cam = scenes.make_camera(0, 0, width=72, height=56)
    cfg = dict(dt_step=0.0025, dynamic_sampling=False, max_prim_slice=2048)
    d = gx.to_dev(sc)
    boxes, _, _ = u_ox.ellipsoids_bbox_from_quat(d["quaternions"], d["positions"], d["scales"], d["densities"])
    gas = u_ox.create_acceleration_structure(None, boxes)
    moved = dict(sc)
    rng = np.random.default_rng(3)
    moved["positions"] = (sc["positions"] + rng.normal(size=sc["positions"].shape).astype(np.float32) * 0.05).astype(np.float32)
    moved["scales"] = (sc["scales"] * rng.uniform(0.7, 1.4, size=sc["scales"].shape)).astype(np.float32)
    m = gx.to_dev(moved)
    new_boxes, _, _ = u_ox.ellipsoids_bbox_from_quat(m["quaternions"], m["positions"], m["scales"], m["densities"])
    _step("refit to moved Gaussians")
    order_before = gas.order().cpu().numpy()
    u_ox.update_acceleration_structure(gas, new_boxes)
    assert np.array_equal(gas.order().cpu().numpy(), order_before)          # same shape, new boxes
    _check_tree(_read_tree(gx, gas), 6000, new_boxes.cpu().numpy())
    cs = u_ox.camera_struct(cam)
    rgb = compute_rgb(cam.camera_center, m["positions"], m["color_features"], None, None, None, 0, 1)
    prims = u_ox.pack_prims(gas, cs, m["positions"], m["scales"], m["quaternions"], m["densities"], rgb)
    stats = u_ox.new_stats(gx.DEV)
    rec = u_ox.new_records(cs, gx.DEV, tile_words=u_ox.REC_LIST_WORDS)      # the recording forward counts whole hit lists
    img = u_ox.march_forward(gas, cs, prims, cfg["dt_step"], False, cfg["max_prim_slice"], True, stats=stats, records=rec)
    want, st, _ = orc.render_forward(moved, cam, cfg["dt_step"], False, cfg["max_prim_slice"])
    got = u_ox.read_stats(stats)
    for k in ("hit_pairs", "slabs", "empty_slabs", "rays_hit"):
        assert got[k] == st[k], k
    assert st["hit_pairs"] > 20000 and np.abs(img.cpu().numpy() - want).max() <= IMG_TOL


@pytest.mark.gpu
@pytest.mark.parametrize("n", [2, 511, 512, 513, 1024, 1025, 5000])      # a workgroup of the refit has 512 leaves
@pytest.mark.parametrize("kind", ["spread", "line", "one place"])
def test_tree_at_the_edges_of_the_refits_workgroups(gx, n, kind):
    """Boxes, children, parents and skip links of a build and of a refit, checked node by node on the host."""
    from raygaussx_amd import optix_utils as u_ox
    from test_gpu_fullsize import _check_tree, _read_tree
    rng = np.random.default_rng(n)
    centre = {"spread": rng.normal(size=(n, 3)), "line": np.linspace(0, 1, n)[:, None] * np.float32([1, 0, 0]), "one place": np.zeros((n, 3))}[kind]
    half = rng.uniform(0.01, 0.1, size=(n, 3))
    boxes = torch.tensor(np.concatenate([centre - half, centre + half], 1).astype(np.float32), device=gx.DEV)
    _step(f"tree of {n}, {kind}")
    gas = u_ox.create_acceleration_structure(None, boxes)
    _check_tree(_read_tree(gx, gas), n, boxes.cpu().numpy())
    boxes = boxes + 0.25
    u_ox.update_acceleration_structure(gas, boxes)
    _check_tree(_read_tree(gx, gas), n, boxes.cpu().numpy())


@pytest.mark.gpu
def test_settings_update_refits_inside_the_render_function(gx):
    """render_optix.py:114-117: with ``settings.update`` the forward hands the new boxes to the
    existing acceleration structure instead of creating one.  A loop that moves the Gaussians between
    two views renders the second view on the refitted tree; image and gradients equal those of a
    forward that builds a new tree (same hit sets; the sums run in another order)."""
    from raygaussx_amd.render_optix import RenderOptixFunction, default_settings
    sc = scenes.scene_to_numpy(scenes.make_scene(0, n=5000, sh_degree=1, seed=21))
    sc["scales"] = sc["scales"] * 2.0
    cam = scenes.make_camera(0, 2, width=64, height=48).to(gx.DEV)
    rng = np.random.default_rng(8)
    moved = dict(sc)
    moved["positions"] = (sc["positions"] + rng.normal(size=sc["positions"].shape).astype(np.float32) * 0.03).astype(np.float32)
    dl = torch.from_numpy(rng.normal(size=(64 * 48, 3)).astype(np.float32)).to(gx.DEV)
    names = ("positions", "scales", "quaternions", "densities", "color_features")
    n = sc["positions"].shape[0]
    empty = (torch.zeros(n, 3, 0, device=gx.DEV), torch.zeros(n, 0, device=gx.DEV), torch.zeros(n, 0, 3, device=gx.DEV))

    def view(scene, settings):
        d = gx.to_dev(scene)
        args = [d[k].clone().requires_grad_(True) for k in names]
        img = RenderOptixFunction.apply(*args, *empty, settings)
        img.backward(dl)
        return img.detach().cpu().numpy(), [a.grad.cpu().numpy() for a in args]

    _step("first view builds, second refits")
    s_upd = default_settings(cam, 0.0025, False, 2048)
    view(sc, s_upd)
    tree, order = s_upd.gas, s_upd.gas.order().cpu().numpy()
    s_upd.update = True
    img_u, g_u = view(moved, s_upd)
    assert s_upd.gas is tree and np.array_equal(tree.order().cpu().numpy(), order)       # refitted, not rebuilt
    s_new = default_settings(cam, 0.0025, False, 2048)
    img_n, g_n = view(moved, s_new)
    assert np.abs(img_n).max() > 0.1 and np.abs(img_u - img_n).max() <= 1e-5
    for k, a, b in zip(names, g_u, g_n):
        c, r = gx.cos_rel(a, b)
        assert c >= 0.99999 and r <= 1e-4, (k, c, r)


@pytest.mark.gpu
def test_issue_rate_probe_runs_every_kind(gx):
    """rgx_probe_valu_rate: every instruction kind (0..9 placed by the compiler, 10..13 with named registers) launches,
    reports the instruction count of its shape and writes nothing to the sink; kinds out of range are refused."""
    import ctypes as C
    from raygaussx_amd import _lib
    sink = torch.full((4,), 7.0, device=gx.DEV)
    count = C.c_uint64(0)
    for kind in range(14):
        _step(f"issue-rate probe, kind {kind}")
        _lib.check(_lib.lib().rgx_probe_valu_rate(C.c_int32(1024), C.c_int32(8), C.c_int32(kind), _lib.ptr(sink), C.byref(count),
                                                  _lib.stream()))
        torch.cuda.synchronize()
        assert count.value == 1024 * 8 * 64
    assert bool((sink == 7.0).all())
    for kind in (-1, 14):
        assert _lib.lib().rgx_probe_valu_rate(C.c_int32(1024), C.c_int32(8), C.c_int32(kind), _lib.ptr(sink), C.byref(count),
                                              _lib.stream()) == -1


def test_scratch_of_streams_no_longer_used_is_dropped(gx, c0):
    """The host mirror keeps one set of scratch tensors per stream in use; a loop that keeps making new
    streams must not keep a set for each of them."""
    from raygaussx_amd import optix_utils as u_ox
    scene, cam, cfg = c0
    small = scenes.make_camera(0, 0, width=32, height=24)
    want = gx.gpu_render(scene, small, cfg, stats=False)["image"]
    for _ in range(2 * u_ox._SCRATCH_STREAMS + 3):
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            got = gx.gpu_render(scene, small, cfg, stats=False)["image"]
        assert np.array_equal(got, want)
    per_key = {}
    for key, dev, _stream in u_ox._scratch:
        per_key[(key, dev)] = per_key.get((key, dev), 0) + 1
    assert per_key and max(per_key.values()) <= u_ox._SCRATCH_STREAMS
