"""GPU parity: the HIP trainer step against the CPU restatement (oracle/),
through the C ABI.

Bar: bit-exact for everything the f32 restatement computes in the same order
(projection records, depth keys, tile rectangles, the sorted (tile, depth,
id) permutation, tile ranges, images, final T, end indices, dL/dC, the
reference's fixed-point gradient sums, parameter gradients, Adam updates);
the f32 atomic-accumulation mode is checked against the f64 reference
within 1e-3 relative.
"""
import math

import numpy as np
import pytest

import gsabi
import oracle as O
import scenes
from helpers import OracleTrainer, config1_setup, f32, rig_setup

pytestmark = pytest.mark.gpu


def _trainer(params, sh, cams, images, W, H, radius, opts=None, shDeg=2, **kw):
    o = dict(opts or {})
    o.update(kw)
    t = gsabi.GSTrainer(shDeg=shDeg, **o)
    g = {"data": params, "n": params.shape[0]}
    if sh is not None:
        g["sh"] = sh
    t.setup(g, cams, images, W, H, radius)
    return t


def _expected_rec(proj):
    """Raster record the kernels store (16 floats), from the restatement's
    proj rows, with the same f32 arithmetic (opa*comp, -0.5/(1+lambda_max),
    1-opa). Slot 6 (the cover level) only decides which waves skip a splat;
    a wrong level would show up as image and gradient mismatches, so it is
    not compared here."""
    p = proj.astype(np.float32)
    va, vb, vc = p[:, 12], p[:, 13], p[:, 14]
    cva = va + np.float32(0.3)
    cvc = vc + np.float32(0.3)
    cmid = np.float32(0.5) * (cva + cvc)
    lmax = cmid + np.sqrt(np.maximum(cmid * cmid - (cva * cvc - vb * vb), np.float32(0)))
    cnorm = np.float32(1) / (np.float32(1) + lmax)
    z = np.zeros_like(cnorm)
    return np.stack([p[:, 0], p[:, 1], p[:, 3], p[:, 4], p[:, 5], p[:, 7] * p[:, 6], z, z,
                     p[:, 8], p[:, 9], p[:, 10], p[:, 7], p[:, 6], np.float32(-0.5) * cnorm,
                     np.float32(1) - p[:, 7], z], 1)


REC_CMP = [0, 1, 2, 3, 4, 5, 7, 8, 9, 10, 11, 12, 13, 14, 15]


def _check_step(gpu, ref, n_tiles, label, stats_acc=None):
    vis = ref["cnt"] > 0
    # projection
    np.testing.assert_array_equal(gpu["cnt"], ref["cnt"], err_msg=label)
    np.testing.assert_array_equal(gpu["rect"][vis], ref["rect"][vis].astype(np.uint32), err_msg=label)
    exp_key = np.where(vis, ref["proj"][:, 2].astype(np.float32).view(np.uint32), np.uint32(0xFFFFFFFF))
    np.testing.assert_array_equal(gpu["depthKey"], exp_key, err_msg=label)
    np.testing.assert_array_equal(gpu["rec"][vis][:, REC_CMP].view(np.uint32),
                                  _expected_rec(ref["proj"])[vis][:, REC_CMP].view(np.uint32), err_msg=label)
    # binning + sort: bit-exact permutation and keys
    assert gpu["numKeys"] == len(ref["ids"]), label
    np.testing.assert_array_equal(gpu["ids"], ref["ids"], err_msg=label)
    np.testing.assert_array_equal(gpu["keys"], ref["keys"], err_msg=label)
    cnt_t = np.diff(ref["ts"].astype(np.int64))
    tr = gpu["tileRanges"].astype(np.int64)
    np.testing.assert_array_equal(tr[:, 1] - tr[:, 0], cnt_t, err_msg=label)
    # every tile start, empty tiles included (the reference's exclusive scan)
    np.testing.assert_array_equal(tr[:, 0], ref["ts"][:-1], err_msg=label)
    # forward composite
    np.testing.assert_array_equal(gpu["img"].view(np.uint32), ref["img"].astype(np.float32).view(np.uint32),
                                  err_msg=label)
    np.testing.assert_array_equal(gpu["T"].view(np.uint32), ref["T"].view(np.uint32), err_msg=label)
    np.testing.assert_array_equal(gpu["end"], ref["end"], err_msg=label)
    # loss gradient
    np.testing.assert_array_equal(gpu["gC"][:, :3].view(np.uint32), ref["gC"].view(np.uint32), err_msg=label)
    np.testing.assert_array_equal(gpu["gC"][:, 3] != 0, ref["valid"] != 0, err_msg=label)
    # the loss stats accumulate over steps until readLoss() (trainer.js:615-631)
    exp_stats = ref["stats"] if stats_acc is None else stats_acc
    np.testing.assert_allclose(gpu["stats"][:3], exp_stats, rtol=1e-9, atol=1e-9, err_msg=label)
    # backward (fixed point: deterministic, bit-exact) and chain
    np.testing.assert_array_equal(gpu["accum"], ref["accum"], err_msg=label)
    np.testing.assert_array_equal(gpu["gradF"][:, :14].view(np.uint32),
                                  ref["gradF"][:, :14].astype(np.float32).view(np.uint32), err_msg=label)
    if ref["shGrad"].size:
        np.testing.assert_array_equal(gpu["shGrad"].view(np.uint32), ref["shGrad"].view(np.uint32),
                                      err_msg=label)


def _run_pair(params, sh, cams, images, W, H, radius, opts, shDeg, steps, start_iter=0, cams_seq=None, **kw):
    gpu = _trainer(params, sh, cams, images, W, H, radius, opts, shDeg=shDeg, **kw)
    prec = {gsabi.GS_PREC_MIXED: "mixed", gsabi.GS_PREC_BF16: "bf16",
            gsabi.GS_PREC_FP16: "fp16"}.get(kw.get("precision", gsabi.GS_PREC_F32), "f32")
    ref = OracleTrainer(params, sh, cams, images, radius, opts=opts, shDeg=shDeg, precision=prec,
                        tile=kw.get("tile", 16))
    gpu.iter = start_iter
    ref.iter = start_iter
    n_tiles = ((W + 15) // 16) * ((H + 15) // 16)
    acc = np.zeros(3)
    for s in range(steps):
        ci = cams_seq[s] if cams_seq else 0
        g = gpu.step_debug(ci)
        r = ref.step(ci)
        acc = acc + r["stats"]
        _check_step(g, r, n_tiles, f"step {s}", stats_acc=acc)
        out = gpu.readGaussians()
        np.testing.assert_array_equal(out["data"].view(np.uint32), ref.P.view(np.uint32), err_msg=f"params step {s}")
        if ref.K:
            np.testing.assert_array_equal(out["sh"].view(np.uint32), ref.SH.view(np.uint32), err_msg=f"sh step {s}")
    gpu.destroy()
    return ref


def test_rig_deg0_bit_exact_three_steps():
    """The reference's gradcheck rig (gradcheck.js:139-185), SH off."""
    params, sh, cams, images, W, H, radius, opts = rig_setup(0)
    _run_pair(params, None, cams, images, W, H, radius, opts, 0, steps=3)


def test_rig_deg3_sh_bit_exact():
    """gradCheckSH rig (gradcheck.js:192-201): degree-3 SH, all bands active."""
    params, sh, cams, images, W, H, radius, opts = rig_setup(3)
    _run_pair(params, sh, cams, images, W, H, radius, opts, 3, steps=2, start_iter=5000)


def test_config1_bit_exact():
    """Config 1: 20k Gaussians, 320x240, SH degree 2 (first step: band ramp
    at degree 0, then full degree)."""
    p, sh, cams, images, W, H, radius = config1_setup()
    _run_pair(p, sh, cams, images, W, H, radius, {}, 2, steps=1, start_iter=0)
    _run_pair(p, sh, cams, images, W, H, radius, {}, 2, steps=2, start_iter=2500)


@pytest.mark.parametrize("tile,batch", [(8, 64), (8, 128), (8, 256), (16, 64), (16, 128), (32, 64), (32, 128),
                                        (32, 256)])
def test_config1_bit_exact_at_every_raster_shape(tile, batch):
    """Config 1 at the other raster shapes (tiles of 8 and 32 pixels, LDS
    batches of 64 and 128 keys) against the restatement run at the same tile
    size: the tile grid changes the rectangles, keys and ranges, the batch
    changes nothing; every intermediate and the updated params stay
    bit-exact."""
    print(f"config 1 at tile {tile}, batch {batch}", flush=True)
    p, sh, cams, images, W, H, radius = config1_setup()
    _run_pair(p, sh, cams, images, W, H, radius, {}, 2, steps=2, start_iter=2500, tile=tile, batch=batch)


def test_spatially_ordered_input_bit_exact():
    """Config 1 with its Gaussians in Morton order of their positions: the
    binning's blocks take equal shares of the work (keys plus one per
    Gaussian, in chunks of 256 Gaussians),
    and in this order a chunk holds 72 to 1356 keys (fixed 4096-Gaussian
    blocks would hold up to 1.31x the mean). Two steps match the restatement
    bit for bit (the block partition changes only the time)."""
    p, sh, cams, images, W, H, radius = config1_setup()
    q = np.clip(((p[:, 0:3].astype(np.float64) - p[:, 0:3].min(0)) /
                 np.ptp(p[:, 0:3], 0).astype(np.float64) * 1023).astype(np.int64), 0, 1023)
    code = np.zeros(len(p), np.int64)
    for bit in range(10):
        for a in range(3):
            code |= ((q[:, a] >> bit) & 1) << (3 * bit + a)
    perm = np.argsort(code, kind="stable")
    _run_pair(np.ascontiguousarray(p[perm]), np.ascontiguousarray(sh[perm]), cams, images, W, H, radius, {}, 2,
              steps=2, start_iter=2500)


PRECISIONS = [gsabi.GS_PREC_MIXED, gsabi.GS_PREC_BF16, gsabi.GS_PREC_FP16]


@pytest.mark.parametrize("precision", PRECISIONS, ids=["mixed", "bf16", "fp16"])
def test_mixed_precision_rig_deg3_bit_exact(precision):
    """16-bit storage modes on the degree-3 rig: bf16 SH and moments (mixed),
    or bf16 / fp16 SH and record colours with f32 moments, all with
    stochastic rounding of the stored coefficients. Every intermediate and
    the updated params/SH match the restatement's same mode bit for bit over
    four steps."""
    params, sh, cams, images, W, H, radius, opts = rig_setup(3)
    _run_pair(params, sh, cams, images, W, H, radius, opts, 3, steps=4, start_iter=5000, precision=precision)


@pytest.mark.parametrize("precision", PRECISIONS, ids=["mixed", "bf16", "fp16"])
def test_mixed_precision_config1_bit_exact(precision):
    p, sh, cams, images, W, H, radius = config1_setup()
    _run_pair(p, sh, cams, images, W, H, radius, {}, 2, steps=3, start_iter=2500, precision=precision)


def test_sort_strategies_give_the_same_permutation():
    p, sh, cams, images, W, H, radius = config1_setup(n=8000)
    outs = []
    for mode in (gsabi.GS_SORT_TILE_SEGMENTS, gsabi.GS_SORT_DEPTH_THEN_TILE, gsabi.GS_SORT_GLOBAL64):
        t = _trainer(p, sh, cams, images, W, H, radius, {}, shDeg=2, sortMode=mode)
        outs.append(t.step_debug(0, want=("ids", "keys", "tileRanges", "img")))
        t.destroy()
    a = outs[0]
    for b in outs[1:]:
        assert a["numKeys"] == b["numKeys"] > 0
        np.testing.assert_array_equal(a["ids"], b["ids"])
        np.testing.assert_array_equal(a["keys"], b["keys"])
        np.testing.assert_array_equal(a["tileRanges"], b["tileRanges"])
        np.testing.assert_array_equal(a["img"], b["img"])


@pytest.mark.parametrize("depths", ["random", "equal", "clustered"])
@pytest.mark.parametrize("n", [1024, 1025, 1537, 4099, 65537, 150000])
def test_one_long_tile_segment_sorts_as_the_radix_strategy(n, depths):
    """A one-tile view under n splats: one segment of n keys, at the last
    size sorted in one piece, the first sizes that split into three, four
    and nine buckets, and the sizes past the 128 buckets, whose larger
    buckets are merged. Equal depths order by id; clustered ones put nine
    keys in ten within 1% of the depth range, in stretches of the input, so
    that the sampled splitters are uneven. Keys, ids and image are those of
    the depth-then-tile radix strategy."""
    rng = np.random.default_rng(n)
    p = np.zeros((n, 16), np.float32)
    z = {"random": rng.uniform(1.0, 9.0, n), "equal": np.full(n, 3.0),
         "clustered": np.where(np.arange(n) // 64 % 10 == 0, rng.uniform(1.0, 9.0, n), rng.uniform(3.0, 3.08, n))}[depths]
    p[:, 0:2] = rng.uniform(-0.3, 0.3, (n, 2)) * z[:, None]
    p[:, 2] = z
    p[:, 3:6] = np.log(0.2 * z)[:, None]
    p[:, 6] = 1.0
    p[:, 10:13] = rng.normal(0, 1, (n, 3))
    p[:, 13] = rng.uniform(-3, 2, n)
    W = H = 16
    cams = [{"imgIdx": 0, "R": [1, 0, 0, 0, 1, 0, 0, 0, 1], "t": [0, 0, 0], "f": 16.0, "cx": 8, "cy": 8, "w": W, "h": H}]
    images = [{"tw": W, "th": H, "rgb": np.full((W * H, 3), 0.5, np.float32)}]
    outs = []
    for mode in (gsabi.GS_SORT_TILE_SEGMENTS, gsabi.GS_SORT_DEPTH_THEN_TILE):
        t = _trainer(p, None, cams, images, W, H, 1.0, {}, shDeg=0, sortMode=mode)
        outs.append(t.step_debug(0, want=("ids", "keys", "tileRanges", "img")))
        t.destroy()
    a, b = outs
    assert a["numKeys"] == b["numKeys"] == n
    np.testing.assert_array_equal(a["keys"], b["keys"])
    np.testing.assert_array_equal(a["ids"], b["ids"])
    np.testing.assert_array_equal(a["tileRanges"], b["tileRanges"])
    np.testing.assert_array_equal(a["img"].view(np.uint32), b["img"].view(np.uint32))


@pytest.mark.parametrize("n,big,small", [(3000, 3000, 0.0), (530000, 1500, 0.05), (530000, 600, 0.003)],
                         ids=["every_tile", "bands", "one_band"])
def test_binning_of_wide_splats_as_the_radix_strategy(n, big, small):
    """A 640x480 view (1200 tiles) whose first `big` splats cover every tile:
    their count and scatter rounds hold 1.2M keys, walked in windows of
    65536. At 530000 splats (256 blocks) of log-scale log(0.05) the view
    holds more than 12 keys per block and tile, so the scatter takes the
    tiles in bands of rows, which the splats cross; small ones stay below
    that. A tenth of the splats are culled, in runs and singly. Keys, ids,
    ranges and image are those of the depth-then-tile radix strategy."""
    rng = np.random.default_rng(7)
    W, H, f = 640, 480, 400.0
    p = np.zeros((n, 16), np.float32)
    z = rng.uniform(2.0, 4.0, n)
    z[rng.random(n) < 0.05] = -1.0                          # behind the camera
    z[n // 3:n // 3 + n // 20] = -1.0
    p[:, 0] = rng.uniform(-0.5, 0.5, n) * W / f * z
    p[:, 1] = rng.uniform(-0.5, 0.5, n) * H / f * z
    p[:, 2] = z
    p[:, 3:6] = np.log(max(small, 1e-3)) + rng.normal(0, 0.1, (n, 3))
    p[:big, 0:2] = 0.0
    p[:big, 3:6] = np.log(4.0)
    p[:, 6] = 1.0
    p[:, 10:13] = rng.normal(0, 1, (n, 3))
    p[:, 13] = rng.uniform(-4, -1, n)
    cams = [{"imgIdx": 0, "R": [1, 0, 0, 0, 1, 0, 0, 0, 1], "t": [0, 0, 0], "f": f, "cx": W / 2, "cy": H / 2, "w": W, "h": H}]
    images = [{"tw": W, "th": H, "rgb": np.full((W * H, 3), 0.5, np.float32)}]
    outs = []
    for mode in (gsabi.GS_SORT_TILE_SEGMENTS, gsabi.GS_SORT_DEPTH_THEN_TILE):
        t = _trainer(p, None, cams, images, W, H, 1.0, {}, shDeg=0, sortMode=mode, radClamp=2000,
                     entriesCap=1 << 24)
        outs.append(t.step_debug(0, want=("ids", "keys", "tileRanges", "img")))
        t.destroy()
    a, b = outs
    per_run = a["numKeys"] / (min(256, -(-n // 2048)) * 1200)
    assert a["numKeys"] == b["numKeys"] > 0.8 * big * 1200
    assert (per_run >= 12) == (small != 0.003)
    np.testing.assert_array_equal(a["keys"], b["keys"])
    np.testing.assert_array_equal(a["ids"], b["ids"])
    np.testing.assert_array_equal(a["tileRanges"], b["tileRanges"])
    np.testing.assert_array_equal(a["img"].view(np.uint32), b["img"].view(np.uint32))


def test_views_above_the_segment_tile_limit_fall_back_to_radix():
    """A 2112x2112 view has 17424 tiles, above the 16384 the tile-segment
    scan handles: the default sort falls back to depth-then-tile and gives
    the same keys, ranges and image as that strategy chosen explicitly."""
    W = H = 2112
    rng = np.random.default_rng(4)
    n = 20000
    p = np.zeros((n, 16), np.float32)
    p[:, 0:2] = rng.uniform(-1.2, 1.2, (n, 2))
    p[:, 2] = rng.uniform(2.0, 4.0, n)
    p[:, 3:6] = rng.normal(-3.5, 0.4, (n, 3))
    p[:, 6] = 1.0
    p[:, 10:13] = rng.normal(0, 1, (n, 3))
    p[:, 13] = rng.normal(0, 1, n)
    cams = [{"imgIdx": 0, "R": [1, 0, 0, 0, 1, 0, 0, 0, 1], "t": [0, 0, 0], "f": 900.0, "cx": W / 2, "cy": H / 2,
             "w": W, "h": H}]
    images = [{"tw": W, "th": H, "rgb": np.full((W * H, 3), 0.5, np.float32)}]
    outs = []
    for mode in (gsabi.GS_SORT_TILE_SEGMENTS, gsabi.GS_SORT_DEPTH_THEN_TILE):
        t = _trainer(p, None, cams, images, W, H, 1.0, {}, shDeg=0, sortMode=mode)
        outs.append(t.step_debug(0, want=("ids", "keys", "tileRanges", "img")))
        t.destroy()
    a, b = outs
    assert a["numKeys"] == b["numKeys"] > 20000
    np.testing.assert_array_equal(a["ids"], b["ids"])
    np.testing.assert_array_equal(a["keys"], b["keys"])
    np.testing.assert_array_equal(a["tileRanges"], b["tileRanges"])
    np.testing.assert_array_equal(a["img"].view(np.uint32), b["img"].view(np.uint32))


def test_f32_accumulation_matches_f64_gradients():
    """GS_ACCUM_F32: atomic f32 sums, checked against the double-precision
    analytic gradients (which central differences pin, test_oracle.py)."""
    params, sh, cams, images, W, H, radius, opts = rig_setup(0)
    t = _trainer(params, None, cams, images, W, H, radius, opts, shDeg=0, gradAccum=gsabi.GS_ACCUM_F32)
    g = t.step_debug(0, want=("gradF", "accum"))
    t.destroy()
    o = O.make_opts(eCut=opts["eCut"], aMin=opts["aMin"], radClamp=opts["radClamp"], anisoReg=0.0, shDeg=0)
    tgt = O.pack_targets(images[0]["rgb"])
    g64, _ = O.analytic_grads(O.Stage(o, "f64"), O.make_cam(cams[0]), params, None, tgt, fixed=False)
    for s in range(14):
        a, b = g["gradF"][:, s].astype(np.float64), g64[:, s]
        big = np.abs(b) > 1e-3 * max(np.abs(b).max(), 1e-12)
        rel = np.abs(a[big] - b[big]) / np.abs(b[big])
        assert np.median(rel) < 1e-4 and rel.max() < 1e-3, (s, rel.max())


def test_fixed_point_step_is_deterministic():
    p, sh, cams, images, W, H, radius = config1_setup(n=6000)
    res = []
    for _ in range(2):
        t = _trainer(p, sh, cams, images, W, H, radius, {}, shDeg=2)
        for _ in range(3):
            t.stepOnce(0)
        res.append(t.readGaussians()["data"])
        t.destroy()
    np.testing.assert_array_equal(res[0].view(np.uint32), res[1].view(np.uint32))


def test_render_view_and_read_loss():
    p, sh, cams, images, W, H, radius = config1_setup(n=6000)
    t = _trainer(p, sh, cams, images, W, H, radius, {}, shDeg=2)
    ref = OracleTrainer(p, sh, cams, images, radius, shDeg=2)
    img = t.renderView(cams[0])
    o = O.make_opts(shDeg=2)
    st = O.Stage(o, "f32")
    cam = O.make_cam(cams[0], shActiveDeg=2)
    proj, rect, cnt = st.project(cam, p, sh)
    ids, ts, _ = st.bin_sort(cam, proj, rect, cnt)
    rimg, _, _ = st.render_fwd(cam, proj, ids, ts)
    np.testing.assert_array_equal(img.reshape(-1, 4).view(np.uint32), rimg.view(np.uint32))
    assert t.readLoss() is None  # reference returns null before any step
    t.stepOnce(0)
    r = ref.step(0)
    mse = t.readLoss()
    assert abs(mse - r["stats"][0] / (r["stats"][2] * 3)) <= 1e-9 * mse
    assert t.readLoss() is None
    # evalCamPsnr = -10 log10(mse) of a fresh pass at the current parameters
    psnr = t.evalCamPsnr(0)
    assert 5 < psnr < 60
    t.destroy()


@pytest.mark.parametrize("n,min_tile", [(3000, 2048), (20000, 8192)])
def test_dense_tiles_and_ragged_image(n, min_tile):
    """Tiles with > 2048 keys (the reference's global-memory bitonic path,
    shaders.js:471-499), several LDS batches per tile, and a 70x45 view whose
    edge tiles are partial. With 20000 Gaussians some tiles hold more than
    8192 keys: their segments sort as 4096-key LDS runs merged twice."""
    rng = np.random.default_rng(11)
    p = np.zeros((n, 16), np.float32)
    p[:, 0] = rng.normal(0, 0.15, n)
    p[:, 1] = rng.normal(0, 0.1, n)
    p[:, 2] = rng.uniform(2.5, 3.5, n)
    p[:, 3:6] = rng.normal(-2.0, 0.3, (n, 3))
    q = rng.normal(size=(n, 4))
    p[:, 6:10] = q / np.linalg.norm(q, axis=1, keepdims=True)
    p[:, 10:13] = rng.normal(0, 1, (n, 3))
    p[:, 13] = rng.normal(-2.5, 0.5, n)
    W, H = 70, 45
    cams = [{"imgIdx": 0, "R": [1, 0, 0, 0, 1, 0, 0, 0, 1], "t": [0, 0, 0], "f": 60, "cx": 35, "cy": 22.5,
             "w": W, "h": H}]
    rgb = rng.random((H * W, 3)).astype(np.float32)
    rgb[rng.random(H * W) < 0.05, 0] = -1  # invalid pixels
    images = [{"tw": W, "th": H, "rgb": rgb}]
    ref = _run_pair(p, None, cams, images, W, H, 1.0, {}, 0, steps=2)
    proj, rect, cnt = ref.st.project(O.make_cam(cams[0]), ref.P, None)
    _, ts, _ = ref.st.bin_sort(O.make_cam(cams[0]), proj, rect, cnt)
    assert np.diff(ts.astype(np.int64)).max() > min_tile


def test_needle_border_and_near_plane_splats_bit_exact():
    """Splats that stress the wave-skip test and the culling end to end:
    needles (one axis e^-1, two axes e^-7 to e^-9, random rotations: the
    ill-conditioned conics the cover test's rounding margin exists for),
    splats straddling the image border and the view-frustum edge, and
    splats just in front of and behind the near plane (z = 0.05). Records,
    sort keys and ids, images, T, end, the fixed-point gradient sums,
    gradients and updated params match the restatement bit for bit over two
    steps, in both precisions; an 8x8 block the cover test skipped wrongly
    would change the image and the sums."""
    rng = np.random.default_rng(23)
    n = 4000
    p = np.zeros((n, 16), np.float32)
    W, H, f = 256, 192, 220.0
    z = rng.uniform(0.5, 4.0, n)
    z[: n // 20] = rng.uniform(0.02, 0.12, n // 20)             # around the near plane
    p[:, 2] = z
    # image-plane positions over 1.4x the view, so many splats straddle the border
    p[:, 0] = (rng.uniform(-0.7, 0.7, n) * W / f) * z
    p[:, 1] = (rng.uniform(-0.7, 0.7, n) * H / f) * z
    ls = np.empty((n, 3))
    ls[:, 0] = rng.uniform(-1.5, -0.8, n)
    ls[:, 1:] = rng.uniform(-9.0, -7.0, (n, 2))
    for r in range(n):                                           # needle along a random axis
        ls[r] = ls[r][rng.permutation(3)]
    iso = rng.random(n) < 0.3                                     # some ordinary splats too
    ls[iso] = rng.normal(-3.0, 0.5, (int(iso.sum()), 3))
    p[:, 3:6] = ls
    q = rng.normal(size=(n, 4))
    p[:, 6:10] = q / np.linalg.norm(q, axis=1, keepdims=True)
    p[:, 10:13] = rng.normal(0, 1, (n, 3))
    p[:, 13] = rng.normal(1.0, 1.0, n)
    cams = [{"imgIdx": 0, "R": [1, 0, 0, 0, 1, 0, 0, 0, 1], "t": [0, 0, 0], "f": f, "cx": W / 2, "cy": H / 2,
             "w": W, "h": H}]
    rgb = rng.random((H * W, 3)).astype(np.float32)
    images = [{"tw": W, "th": H, "rgb": rgb}]
    _run_pair(p, None, cams, images, W, H, 2.0, {}, 0, steps=2)
    _run_pair(p, None, cams, images, W, H, 2.0, {}, 0, steps=2, precision=gsabi.GS_PREC_MIXED)


def test_all_culled_and_single_gaussian():
    W, H = 48, 32
    cams = [{"imgIdx": 0, "R": [1, 0, 0, 0, 1, 0, 0, 0, 1], "t": [0, 0, 0], "f": 40, "cx": 24, "cy": 16,
             "w": W, "h": H}]
    images = [{"tw": W, "th": H, "rgb": np.full((W * H, 3), 0.5, np.float32)}]
    behind = np.zeros((5, 16), np.float32)
    behind[:, 2] = -3.0
    behind[:, 6] = 1
    _run_pair(behind, None, cams, images, W, H, 1.0, {}, 0, steps=2)
    one = np.zeros((1, 16), np.float32)
    one[0, 2] = 2.0
    one[0, 3:6] = math.log(0.3)
    one[0, 6] = 1
    one[0, 13] = 1.0
    _run_pair(one, None, cams, images, W, H, 1.0, {}, 0, steps=2)


def test_multi_camera_seeded_pick_and_holdout():
    """stepOnce() picks cameras with the seeded RNG and skips the holdout
    (trainer.js:400-406); the picks match a host replay of mulberry32."""
    p, sh, cams = scenes.config2(n=4000, views=6, W=96, H=64, f=70.0)
    rng = np.random.default_rng(2)
    images = [{"tw": 96, "th": 64, "rgb": rng.random((96 * 64, 3)).astype(np.float32)} for _ in cams]
    t = _trainer(p, sh, cams, images, 96, 64, 5.0, {}, shDeg=2, seed=1234)
    t.holdout = 2
    seen = []
    for _ in range(20):
        t.stepOnce()
        seen.append(t.info().lastCam)
    t.destroy()

    def mulberry(a):
        a = (a + 0x6D2B79F5) & 0xFFFFFFFF
        x = ((a ^ (a >> 15)) * (1 | a)) & 0xFFFFFFFF
        x = ((x + (((x ^ (x >> 7)) * (61 | x)) & 0xFFFFFFFF)) & 0xFFFFFFFF) ^ x
        return a, (x ^ (x >> 14)) & 0xFFFFFFFF
    a, exp = 1234, []
    for _ in range(20):
        a, r = mulberry(a)
        ci = int(r / 4294967296.0 * 6)
        if ci == 2:
            ci = 3
        exp.append(ci)
    assert seen == exp


def test_entry_budget_drops_whole_tiles_as_the_reference():
    """Tile segments (the default) under a budget that cannot hold every
    key: the reference's scan drops whole tiles (shaders.js:321-370). The
    kept keys, tile ranges, image and dropped-tile count equal the
    restatement's (oracle.apply_tile_budget)."""
    p, sh, cams, images, W, H, radius = config1_setup(n=4000)
    st = O.Stage(O.make_opts(shDeg=2), "f32")
    cam = O.make_cam(cams[0], shActiveDeg=0)
    proj, rect, cnt = st.project(cam, p, sh)
    ids, ts, keys = st.bin_sort(cam, proj, rect, cnt)
    cap = len(ids) // 2
    ids2, keys2, ts2, dropped = O.apply_tile_budget(ids, keys, ts, cap)
    assert 0 < dropped and 0 < len(ids2) < len(ids)
    t = _trainer(p, sh, cams, images, W, H, radius, {}, shDeg=2, entriesCap=cap)
    g = t.step_debug(0)
    assert g["numKeys"] == len(ids2)
    np.testing.assert_array_equal(g["ids"], ids2)
    np.testing.assert_array_equal(g["keys"], keys2)
    tr = g["tileRanges"].astype(np.int64)
    np.testing.assert_array_equal(tr[:, 0], ts2[:-1])
    np.testing.assert_array_equal(tr[:, 1], ts2[1:])
    img, T, end = st.render_fwd(cam, proj, ids2, ts2)
    np.testing.assert_array_equal(g["img"].view(np.uint32), img.astype(np.float32).view(np.uint32))
    np.testing.assert_array_equal(g["end"], end)
    info = t.step_stats()
    assert info.lastKeys == len(ids2) and info.overflowKeys == dropped
    # refine's telemetry reads the per-tile counts before the budget
    # (trainer.js:780-789), so it reports the largest tile even when dropped
    r = t.refine(seed=1)
    assert r["maxTile"] == int(np.diff(ts).max()) and r["overflow"] == dropped
    t.destroy()


def _budget_scene(n, W, H, wide, seed=3):
    """n splats over a W x H view, a third of them in its middle (segments past
    2048 keys), the first `wide` of them over all of it."""
    rng = np.random.default_rng(seed)
    f = float(W)
    p = np.zeros((n, 16), np.float32)
    z = rng.uniform(2.0, 4.0, n)
    spread = np.where(np.arange(n) % 3 == 0, 0.04, 1.0)
    p[:, 0] = rng.uniform(-0.5, 0.5, n) * spread * W / f * z
    p[:, 1] = rng.uniform(-0.5, 0.5, n) * spread * H / f * z
    p[:, 2] = z
    p[:, 3:6] = np.log(0.03) + rng.normal(0, 0.1, (n, 3))
    p[:wide, 0:2] = 0.0
    p[:wide, 3:6] = np.log(4.0)
    p[:, 6] = 1.0
    p[:, 10:13] = rng.normal(0, 1, (n, 3))
    p[:, 13] = rng.uniform(-4, -1, n)
    cams = [{"imgIdx": 0, "R": [1, 0, 0, 0, 1, 0, 0, 0, 1], "t": [0, 0, 0], "f": f, "cx": W / 2, "cy": H / 2, "w": W, "h": H}]
    images = [{"tw": W, "th": H, "rgb": np.full((W * H, 3), 0.5, np.float32)}]
    return p, cams, images


@pytest.mark.parametrize("share", [0.05, 0.6, 0.98])
@pytest.mark.parametrize("W,H,n,wide", [(690, 395, 20000, 0), (955, 555, 20000, 0), (1195, 890, 30000, 0), (1995, 1147, 30000, 0),
                                        (640, 480, 300000, 3000)],
                         ids=["1100_tiles", "2100_tiles", "4200_tiles", "9000_tiles", "bands"])
def test_entry_budget_at_every_width_of_the_scan(W, H, n, wide, share):
    """The budget's end inside a chunk of 64 tiles, for each number of tiles
    that a thread of the scan takes (2, 4, 8 and 16; 1 in the test above), most
    tiles dropped, about half, and fewer; the last chunks are not full. In the
    last view the scatter also takes the tiles in bands of rows. The
    kept keys, ranges and dropped tiles are the restatement's budget applied to
    the radix strategy's keys."""
    p, cams, images = _budget_scene(n, W, H, wide)
    kw = dict(shDeg=0, radClamp=2000.0)
    t = _trainer(p, None, cams, images, W, H, 1.0, {}, sortMode=gsabi.GS_SORT_DEPTH_THEN_TILE, entriesCap=1 << 24, **kw)
    r = t.step_debug(0, want=("ids", "keys", "tileRanges"))
    t.destroy()
    tiles = -(-W // 16) * -(-H // 16)
    ts = np.searchsorted(r["keys"] >> np.uint64(32), np.arange(tiles + 1, dtype=np.uint64)).astype(np.uint32)
    cap = int(share * r["numKeys"])
    ids, keys, ts2, dropped = O.apply_tile_budget(r["ids"], r["keys"], ts, cap)
    assert 0 < dropped < tiles and 0 < len(ids) < r["numKeys"]
    if wide:   # keys for bands: 12 per block and tile
        assert r["numKeys"] >= 12 * 256 * tiles
    t = _trainer(p, None, cams, images, W, H, 1.0, {}, entriesCap=cap, **kw)
    g = t.step_debug(0, want=("ids", "keys", "tileRanges"))
    stats = t.step_stats()
    t.destroy()
    assert g["numKeys"] == stats.lastKeys == len(ids) and stats.overflowKeys == dropped
    np.testing.assert_array_equal(g["ids"], ids)
    np.testing.assert_array_equal(g["keys"], keys)
    tr = g["tileRanges"].astype(np.int64)
    np.testing.assert_array_equal(tr[:, 0], ts2[:-1])
    np.testing.assert_array_equal(tr[:, 1], ts2[1:])


def test_rounds_full_of_wide_splats_as_the_radix_strategy():
    """270,000 splats over all 100 tiles of a view: every block's round of 1024
    Gaussians holds 102,400 keys, walked in two windows of 65536. (The budget
    counts 2^19 keys for each tile's 270,000.)"""
    p, cams, images = _budget_scene(270000, 160, 160, 270000)
    outs = []
    for mode in (gsabi.GS_SORT_TILE_SEGMENTS, gsabi.GS_SORT_DEPTH_THEN_TILE):
        t = _trainer(p, None, cams, images, 160, 160, 1.0, {}, shDeg=0, sortMode=mode, radClamp=2000.0, entriesCap=1 << 26)
        outs.append(t.step_debug(0, want=("ids", "keys", "tileRanges")))
        t.destroy()
    a, b = outs
    assert a["numKeys"] == b["numKeys"] == 270000 * 100
    np.testing.assert_array_equal(a["keys"], b["keys"])
    np.testing.assert_array_equal(a["ids"], b["ids"])
    np.testing.assert_array_equal(a["tileRanges"], b["tileRanges"])


def test_radix_sort_budget_drops_keys_in_sort_order():
    """The radix strategies keep the first `entriesCap` keys of the sorted
    order instead."""
    p, sh, cams, images, W, H, radius = config1_setup(n=4000)
    t = _trainer(p, sh, cams, images, W, H, radius, {}, shDeg=2, entriesCap=500,
                 sortMode=gsabi.GS_SORT_DEPTH_THEN_TILE)
    t.stepOnce(0)
    info = t.step_stats()
    assert info.lastKeys == 500
    assert info.overflowKeys > 0
    t.destroy()


def test_setup_rejects_bad_input():
    t = gsabi.GSTrainer()
    with pytest.raises(gsabi.GsError):
        t.stepOnce()
    with pytest.raises(gsabi.GsError):
        t.setup({"data": np.zeros((1, 16), np.float32), "n": 1},
                [{"imgIdx": 3, "R": [1, 0, 0, 0, 1, 0, 0, 0, 1], "t": [0, 0, 0], "f": 1, "cx": 0, "cy": 0}],
                [{"tw": 4, "th": 4, "rgb": np.zeros(48, np.float32)}], 4, 4, 1.0)
    t.destroy()


@pytest.mark.parametrize("tile,batch", [(16, 256), (32, 128), (8, 64)])
def test_l1_dssim_loss_against_f64(tile, batch):
    """L1 + 0.2 D-SSIM (the textbook loss; the reference has only
    Charbonnier): the two SSIM kernels against the double-precision
    restatement on the GPU's own forward image. f32 blur sums lose digits
    in var = E[x^2] - mu^2, so dL/dC is held to 3e-4 of its largest
    magnitude (and 1e-5 relative on the loss). The backward pass fed with
    the GPU's dL/dC stays bit-exact. The target carries an invalid border
    (4 rows and 6 columns) and a few invalid pixels inside, which enter the
    SSIM windows as zeros and take no gradient. The loss kernels keep their
    own 16x16 image tiling at every raster shape."""
    print(f"L1 + D-SSIM at tile {tile}, batch {batch}", flush=True)
    p, sh, cams, images, W, H, radius = config1_setup(n=8000)
    rgb = images[0]["rgb"].reshape(H, W, 3).copy()
    rgb[:4, :, 0] = -1.0
    rgb[:, -6:, 0] = -1.0
    rgb[100:103, 50:52, 0] = -1.0
    images = [dict(images[0], rgb=rgb.reshape(-1))]
    t = _trainer(p, sh, cams, images, W, H, radius, {}, shDeg=2, loss=gsabi.GS_LOSS_L1_DSSIM, ssimLambda=0.2,
                 tile=tile, batch=batch)
    t.iter = 2500
    g = t.step_debug(0, want=("img", "T", "end", "gC", "accum", "stats", "ids", "tileRanges"))
    t.destroy()
    cam = O.make_cam(cams[0], shActiveDeg=2, tile=tile)
    tgt = O.pack_targets(images[0]["rgb"])
    st64 = O.Stage(O.make_opts(shDeg=2), "f64")
    gC64, valid, stats64 = st64.loss_l1ssim(cam, g["img"].astype(np.float64), tgt, 0.2)
    scale = np.abs(gC64).max()
    err = np.abs(g["gC"][:, :3] - gC64)
    assert err.max() <= 3e-4 * scale, (err.max(), scale)
    assert np.median(err) <= 1e-6 * scale
    np.testing.assert_array_equal(g["gC"][:, 3] != 0, valid != 0)
    assert (valid == 0).sum() > 4 * W and not g["gC"][valid == 0].any()
    np.testing.assert_allclose(g["stats"][:3], stats64, rtol=1e-5)
    # backward given the same dL/dC: deterministic fixed-point sums, bit-exact
    st32 = O.Stage(O.make_opts(shDeg=2), "f32")
    proj, rect, cnt = st32.project(cam, p, sh)
    ids, ts, _ = st32.bin_sort(cam, proj, rect, cnt)
    np.testing.assert_array_equal(g["ids"], ids)
    acc = st32.render_bwd(cam, proj, ids, ts, g["T"], g["end"], g["gC"][:, :3].copy(), valid, fixed=True)
    np.testing.assert_array_equal(g["accum"], acc)


@pytest.mark.parametrize("W,H", [(32, 16), (33, 17), (31, 15), (1, 1), (1, 41), (70, 5), (5, 6), (64, 49)])
def test_l1_dssim_loss_at_the_edges_of_its_tiles(W, H):
    """The SSIM kernels' 32x16 tiles, whole, one pixel over and one short,
    views narrower than the window, and ragged ones; a tenth of the pixels
    invalid. The bounds are those of the larger view above (f32 blur sums
    against f64): 3e-4 of the largest gradient, 1e-5 relative on the loss."""
    rng = np.random.default_rng(100 * W + H)
    n, f = 300, 20.0
    p = np.zeros((n, 16), np.float32)
    z = rng.uniform(2.0, 4.0, n)
    p[:, 0] = rng.uniform(-0.5, 0.5, n) * W / f * z
    p[:, 1] = rng.uniform(-0.5, 0.5, n) * H / f * z
    p[:, 2] = z
    p[:, 3:6] = np.log(0.3)
    p[:, 6] = 1.0
    p[:, 10:13] = rng.normal(0, 1, (n, 3))
    p[:, 13] = rng.uniform(-2, 1, n)
    cams = [{"imgIdx": 0, "R": [1, 0, 0, 0, 1, 0, 0, 0, 1], "t": [0, 0, 0], "f": f, "cx": W / 2, "cy": H / 2, "w": W, "h": H}]
    rgb = rng.random((H * W, 3)).astype(np.float32)
    rgb[rng.random(H * W) < 0.1, 0] = -1.0
    rgb[0] = 0.5
    images = [{"tw": W, "th": H, "rgb": rgb}]
    t = _trainer(p, None, cams, images, W, H, 1.0, {}, shDeg=0, loss=gsabi.GS_LOSS_L1_DSSIM, ssimLambda=0.2)
    g = t.step_debug(0, want=("img", "gC", "stats"))
    t.destroy()
    st64 = O.Stage(O.make_opts(shDeg=0), "f64")
    gC64, valid, stats64 = st64.loss_l1ssim(O.make_cam(cams[0]), g["img"].astype(np.float64), O.pack_targets(rgb), 0.2)
    np.testing.assert_array_equal(g["gC"][:, 3] != 0, valid != 0)
    assert not g["gC"][valid == 0].any()
    assert np.abs(g["gC"][:, :3] - gC64).max() <= 3e-4 * np.abs(gC64).max()
    np.testing.assert_allclose(g["stats"][:3], stats64, rtol=1e-5)


def test_l1_dssim_training_reduces_loss():
    p, sh, cams, images, W, H, radius = config1_setup(n=8000)
    t = _trainer(p, sh, cams, images, W, H, radius, {}, shDeg=2, loss=gsabi.GS_LOSS_L1_DSSIM)
    first = None
    for k in range(60):
        t.stepOnce(0)
        if k == 4:
            first = t.readLoss()
    t.readLoss()
    for _ in range(5):
        t.stepOnce(0)
    last = t.readLoss()
    t.destroy()
    assert last < first


@pytest.mark.parametrize("gain", [6.0e4, 1.0e6])
def test_gradient_terms_beyond_the_fixed_point_clamp(gain):
    """An exposure gain of 6e4 brings single pixels' x16384 gradient terms
    past the +-1e9 clamp (the largest gain whose colour terms need none), one
    of 1e6 the colour terms too: sums and updates stay bit-exact."""
    print(f"gain {gain}", flush=True)
    params, sh, cams, images, W, H, radius, opts = rig_setup(3)
    # the camera struct holds the log gain in f32
    cams = [dict(c, g=float(np.float32(math.log(gain)))) for c in cams]
    _run_pair(params, sh, cams, images, W, H, radius, opts, 3, steps=2, start_iter=5000)


@pytest.mark.parametrize("precision", [gsabi.GS_PREC_F32, gsabi.GS_PREC_BF16, gsabi.GS_PREC_FP16])
@pytest.mark.parametrize("n,deg", [(1, 3), (32768, 0), (32769, 1), (11651, 3), (11650, 3), (600001, 2)])
def test_gaussians_read_in_blocks(n, deg, precision):
    """readGaussians hands 2 MB blocks of whole rows through a ring of 8: one
    row, one whole block (32768 rows of parameters; 11650 of degree 3), one
    row more, and several times around the ring. The rows are those set up
    (coefficients as the storage format rounds them, which the asynchronous
    read, a host loop over the planes, gives too)."""
    print(n, deg, precision, flush=True)
    rng = np.random.default_rng(n + deg)
    K = scenes.sh_k(deg)
    p = np.zeros((n, 16), np.float32)
    p[:, :14] = rng.normal(0, 1, (n, 14))
    sh = rng.normal(0, 1, (n, 3 * K)).astype(np.float32) if K else None
    cams = [{"imgIdx": 0, "R": [1, 0, 0, 0, 1, 0, 0, 0, 1], "t": [0, 0, 0], "f": 16.0, "cx": 8, "cy": 8, "w": 16, "h": 16}]
    images = [{"tw": 16, "th": 16, "rgb": np.full((256, 3), 0.5, np.float32)}]
    t = _trainer(p, sh, cams, images, 16, 16, 1.0, {}, shDeg=deg, precision=precision, maxSplats=n + 77)
    got, again, ref = t.readGaussians(), t.readGaussians(), t.read_gaussians_async().wait()
    t.destroy()
    for g in (got, again):
        np.testing.assert_array_equal(g["data"].view(np.uint32), p.view(np.uint32))
        if K:
            np.testing.assert_array_equal(g["sh"].view(np.uint32), ref["sh"].view(np.uint32))
            if precision == gsabi.GS_PREC_F32:
                np.testing.assert_array_equal(g["sh"], sh)


@pytest.mark.parametrize("W,H", [(1, 1), (512, 256), (257, 511), (1921, 1081)])
def test_view_read_in_blocks(W, H):
    """A rendered view comes in the same blocks: one pixel, one whole block,
    one pixel short of it, and several times around the ring; the image is
    the training forward's, which is read in one copy."""
    rng = np.random.default_rng(W)
    n, f = 500, float(W)
    p = np.zeros((n, 16), np.float32)
    z = rng.uniform(2.0, 4.0, n)
    p[:, 0] = rng.uniform(-0.5, 0.5, n) * W / f * z
    p[:, 1] = rng.uniform(-0.5, 0.5, n) * H / f * z
    p[:, 2] = z
    p[:, 3:6] = np.log(0.2)
    p[:, 6] = 1.0
    p[:, 10:14] = rng.normal(0, 1, (n, 4))
    cams = [{"imgIdx": 0, "R": [1, 0, 0, 0, 1, 0, 0, 0, 1], "t": [0, 0, 0], "f": f, "cx": W / 2, "cy": H / 2, "w": W, "h": H}]
    images = [{"tw": W, "th": H, "rgb": np.full((W * H, 3), 0.5, np.float32)}]
    t = _trainer(p, None, cams, images, W, H, 1.0, {}, shDeg=0)
    a, b = t.renderView(cams[0]), t.renderView(cams[0])
    ref = t.step_debug(0, want=("img",))["img"]
    t.destroy()
    for v in (a, b):
        np.testing.assert_array_equal(v.reshape(-1).view(np.uint32), ref.reshape(-1).view(np.uint32))


@pytest.mark.parametrize("tile,batch", [(16, 256), (16, 64), (32, 256), (8, 128)])
@pytest.mark.parametrize("n", [1, 63, 65, 127, 128, 129, 257, 385])
def test_backward_lists_at_the_edges_of_their_batches(n, tile, batch):
    """One view of 24x16 pixels: n faint splats, half of them inside one 4x4
    block, half over the whole view, so that the groups of a wave have lists
    of different lengths (none among them), over one batch of 128 keys, one
    key more or less, and several. Bit-exact against the restatement."""
    print(n, tile, batch, flush=True)
    rng = np.random.default_rng(n)
    W, H, f = 24, 16, 24.0
    p = np.zeros((n, 16), np.float32)
    z = rng.uniform(2.0, 4.0, n)
    wide = rng.random(n) < 0.5
    p[:, 0] = rng.uniform(-0.5, 0.5, n) * W / f * z
    p[:, 1] = rng.uniform(-0.5, 0.5, n) * H / f * z
    p[:, 2] = z
    p[:, 3:6] = np.where(wide, np.log(1.0), np.log(0.02))[:, None] + rng.normal(0, 0.1, (n, 3))
    p[:, 6] = 1.0
    p[:, 10:13] = rng.normal(0, 1, (n, 3))
    p[:, 13] = np.where(wide, -4.0, -1.0)
    cams = [{"imgIdx": 0, "R": [1, 0, 0, 0, 1, 0, 0, 0, 1], "t": [0, 0, 0], "f": f, "cx": W / 2, "cy": H / 2, "w": W, "h": H}]
    images = [{"tw": W, "th": H, "rgb": rng.random((H * W, 3)).astype(np.float32)}]
    t = _trainer(p, None, cams, images, W, H, 1.0, {}, shDeg=0, tile=tile, batch=batch)
    t.iter = 5000
    ref = OracleTrainer(p, None, cams, images, 1.0, opts={}, shDeg=0, tile=tile)
    ref.iter = 5000
    g, r = t.step_debug(0), ref.step(0)
    out = t.readGaussians()
    t.destroy()
    np.testing.assert_array_equal(g["accum"], r["accum"])
    np.testing.assert_array_equal(out["data"].view(np.uint32), ref.P.view(np.uint32))


@pytest.mark.parametrize("tile,batch", [(16, 256), (16, 64), (32, 256), (8, 128)])
@pytest.mark.parametrize("n", [1, 63, 65, 128, 129, 257])
@pytest.mark.parametrize("loss", ["charbonnier", "l1_dssim"])
def test_f32_sums_at_the_edges_of_their_batches(n, tile, batch, loss):
    """GS_ACCUM_F32 on the view above, both passes in one launch and in two:
    every per-pixel term is the restatement's for the same dL/dC, only the
    order of the sums differs. A sum of N f32 terms in
    any order is within (N - 1) 2^-24 of the sum of their magnitudes (and the
    terms' own sum in f64 is exact to 2^-53), here N = 384 pixels; the
    magnitudes come from the restatement, one pixel at a time."""
    print(n, tile, batch, loss, flush=True)
    rng = np.random.default_rng(n)
    W, H, f = 24, 16, 24.0
    p = np.zeros((n, 16), np.float32)
    z = rng.uniform(2.0, 4.0, n)
    wide = rng.random(n) < 0.5
    p[:, 0] = rng.uniform(-0.5, 0.5, n) * W / f * z
    p[:, 1] = rng.uniform(-0.5, 0.5, n) * H / f * z
    p[:, 2] = z
    p[:, 3:6] = np.where(wide, np.log(1.0), np.log(0.02))[:, None] + rng.normal(0, 0.1, (n, 3))
    p[:, 6] = 1.0
    p[:, 10:13] = rng.normal(0, 1, (n, 3))
    p[:, 13] = np.where(wide, -4.0, -1.0)
    cams = [{"imgIdx": 0, "R": [1, 0, 0, 0, 1, 0, 0, 0, 1], "t": [0, 0, 0], "f": f, "cx": W / 2, "cy": H / 2, "w": W, "h": H}]
    images = [{"tw": W, "th": H, "rgb": rng.random((H * W, 3)).astype(np.float32)}]
    t = _trainer(p, None, cams, images, W, H, 1.0, {}, shDeg=0, tile=tile, batch=batch, gradAccum=gsabi.GS_ACCUM_F32,
                 loss=gsabi.GS_LOSS_L1_DSSIM if loss == "l1_dssim" else gsabi.GS_LOSS_CHARBONNIER)
    out = t.step_debug(0, want=("accum", "gC"))
    t.destroy()
    g = out["accum"].view(np.float32).astype(np.float64)
    st = O.Stage(O.make_opts(shDeg=0), "f32")
    cam = O.make_cam(cams[0], tile=tile)
    proj, rect, cnt = st.project(cam, p, None)
    ids, ts, _ = st.bin_sort(cam, proj, rect, cnt)
    _, T, end = st.render_fwd(cam, proj, ids, ts)
    gC = np.ascontiguousarray(out["gC"][:, :3])
    valid = (out["gC"][:, 3] != 0).astype(np.uint8)
    ref = st.render_bwd(cam, proj, ids, ts, T, end, gC, valid, fixed=False)
    mag = np.zeros_like(ref)
    for px in range(W * H):
        one = np.zeros_like(valid)
        one[px] = valid[px]
        mag += np.abs(st.render_bwd(cam, proj, ids, ts, T, end, gC, one, fixed=False))
    assert mag.any()
    assert np.all(np.abs(g - ref) <= W * H * 2.0 ** -24 * mag + 1e-30)


def test_psnr_reads_start_from_cleared_statistics():
    """A PSNR read leaves its statistics cleared for the next one; a training
    view rendered in between adds to them. The sums' atomics come in any
    order, in f64: 1e-9 relative."""
    p, sh, cams, images, W, H, radius = config1_setup(n=3000)
    t = _trainer(p, sh, cams, images, W, H, radius, {}, shDeg=2)
    first = t.evalCamPsnr(0)
    again = t.evalCamPsnr(0)
    t.renderView(t.camMeta[0], 1, t.camMeta[0]["offset"])
    after = t.evalCamPsnr(0)
    t.stepOnce(0)
    assert t.readLoss() > 0.0
    assert t.readLoss() is None
    t.destroy()
    np.testing.assert_allclose([again, after], first, rtol=1e-9)
