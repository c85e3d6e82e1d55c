"""HairMSNN frame loop (render_hair_msnn.cu:699-771, cuda/hair_msnn.cu):
the truncated and training paths share the plain path tracer's random
streams, so with BETA >= path_v2 the short-path image equals the plain
path-traced pass bit for bit; with small BETA it matches the oracle's
msnnPathTrace restatement."""
import json
from pathlib import Path

import numpy as np
import pytest

from tests import oracle_lib as ol

pytestmark = pytest.mark.gpu
SCENES = Path(__file__).resolve().parent.parent / "hairmsnn_amd" / "scenes"


def cfg_small(w=64, h=64, records=1024, warmup=4):
    cfg = json.loads((SCENES / "c0_hairball.json").read_text())
    cfg["integrator"].update({"width": w, "height": h})
    cfg["hairmsnn"] = {"train_records": records, "warmup_steps": warmup, "learning_rate": 0.01}
    cfg["tcnn"] = {"config": "unused.json", "init_train": True}
    return cfg


def test_beta_beyond_depth_reproduces_plain_pass(gpu):
    cfg = cfg_small()
    with gpu.Scene(json_text=cfg) as sc:
        sc.pt_reset()
        sc.pt_passes(1)
        pt = sc.last_pass()[..., :3].copy()
        sc.msnn_begin(BETA=41)
        sc.msnn_frames(1)
        short = sc.msnn_image(1)[..., :3]
    ok = np.isfinite(pt).all(-1)
    np.testing.assert_array_equal(short[ok], pt[ok])


def test_truncated_pass_matches_oracle(gpu):
    cfg = cfg_small(records=128)  # 1 training pixel in 32
    cfg_trunc = json.loads(json.dumps(cfg))
    cfg_trunc["integrator"]["path_v2"] = 2  # vertices 0 and 1: the kernel-beta-0 truncated path
    with gpu.Scene(json_text=cfg_trunc) as st:
        st.pt_reset()
        st.pt_passes(1)
        pt_trunc = st.last_pass()[..., :3].astype(np.float64)
    with gpu.Scene(json_text=cfg) as sc:
        sc.pt_reset()
        sc.pt_passes(1)
        pt_full = sc.last_pass()[..., :3].astype(np.float64)  # every pixel's full path, frame 0's seeds
        sc.msnn_begin(BETA=1)
        sc.msnn_frames(1)
        short = sc.msnn_image(1)[..., :3].astype(np.float64)
        osc = ol.OracleScene(sc.info, sc.segments(), sc.env())
    o_short, _, hit = osc.render(0, 0, 64, 64, spp=1, accum_id0=0, mode=1, kbeta=0, prec=1)
    o_full, o_s2, _ = osc.render(0, 0, 64, 64, spp=1, accum_id0=0, mode=2, kbeta=0, prec=1)
    # a pixel is either a truncated path or a training path (full colour kept)
    close_short = (np.abs(short - o_short) <= 1e-3 * np.maximum(np.abs(o_short), 1e-2)).all(-1)
    close_full = (np.abs(short - o_full) <= 1e-3 * np.maximum(np.abs(o_full), 1e-2)).all(-1)
    frac = (close_short | close_full).mean()
    print(f"truncated-pass agreement {frac:.4f}; training-like pixels {np.mean(close_full & ~close_short):.4f}")
    assert frac >= 0.95
    # GPU against GPU, bit for bit: every pixel of the short image is its
    # truncated path, except the training pixels (one per 32, traced in full
    # by their batch pass), which carry their full path
    diff = ~(short == pt_trunc).all(-1)
    full = (short == pt_full).all(-1)
    print(f"pixels differing from the truncated pass: {diff.sum()} (training records 128), all full paths: "
          f"{bool(full[diff].all())}")
    assert full[diff].all()
    assert 0 < diff.sum() <= 128
    # the truncated path is never brighter than the full path on average
    assert o_short.mean() <= o_full.mean() + 1e-6


def test_render_composes_short_path_and_cache(gpu):
    """RENDER composite (cuda/hair_msnn.cu:314-331): on a hair primary hit the
    final colour is short path + network output; escaped and surface pixels
    keep the short path, and their network image is the short path too. After
    one frame the averages are the frame's values, so the relation is exact
    (one FP32 addition)."""
    cfg = cfg_small(records=2048, warmup=16)
    cfg["surface"] = {"sphere": {"center": [0, 0, 0], "radius": 1.0, "albedo": [0.3, 0.3, 0.3], "alpha": 0.5}}
    with gpu.Scene(json_text=cfg) as sc:
        sc.msnn_begin(BETA=1)
        st = sc.msnn_frames(1)
        final = sc.msnn_image(0)[..., :3].reshape(-1, 3)
        short = sc.msnn_image(1)[..., :3].reshape(-1, 3)
        net = sc.msnn_image(2)[..., :3].reshape(-1, 3)
        hit = sc.msnn_buffer("gb_hit")
        nn_out = sc.msnn_buffer("nn_output")
        gb_color = sc.msnn_buffer("gb_color")[:, :3]
        st8 = sc.msnn_frames(7)
        final8 = sc.msnn_image(0)[..., :3]
        ref = sc.render_path_tracing(64)[..., :3]
    assert st["frames"] == 1 and st["train_steps"] == 16 + 1 and st8["train_steps"] == 16 + 8
    hair = (hit & 1).astype(bool) & ~(hit & 2).astype(bool)
    other = ~hair
    print(f"hair pixels {hair.mean():.3f}, surface {((hit & 2) > 0).mean():.3f}, escaped {((hit & 1) == 0).mean():.3f}")
    assert 0.05 < hair.mean() < 0.95 and ((hit & 2) > 0).any() and ((hit & 1) == 0).any()
    ok = np.isfinite(gb_color).all(-1) & np.isfinite(nn_out).all(-1)
    assert ok.mean() > 0.999
    h, o = hair & ok, other & ok
    np.testing.assert_array_equal(short[ok], gb_color[ok])
    np.testing.assert_array_equal(net[h], nn_out[h])
    np.testing.assert_array_equal(final[h], (gb_color[h] + nn_out[h]).astype(np.float32))
    np.testing.assert_array_equal(final[o], gb_color[o])
    np.testing.assert_array_equal(net[o], gb_color[o])
    assert (nn_out[h] > 0).all()  # exp activation
    # after 8 frames: finite, and within a loose bias band of the reference
    assert np.all(np.isfinite(final8))
    assert final8.mean() == pytest.approx(ref.mean(), rel=0.25)


def test_training_records_match_oracle(gpu):
    """The frame's training records (cuda/hair_msnn.cu:203-276): network
    input at the training pixel's primary hit and target full - short after
    the reference's NaN / Inf scrub, against the oracle's restatement of the
    training path on the same random stream (FP32). Records of pixels that
    miss are zero targets exactly; the input record of each training pixel
    equals the frame pass's record of that pixel bit for bit (the batch pass
    traces the same camera ray)."""
    cfg = cfg_small(records=1024, warmup=2)
    with gpu.Scene(json_text=cfg) as sc:
        sc.msnn_begin(BETA=1)
        sc.msnn_frames(1)
        z = sc.msnn_sizes()
        pix = sc.msnn_buffer("train_pixel")
        tin = sc.msnn_buffer("train_input")
        tgt = sc.msnn_buffer("train_target").astype(np.float64)
        gin = sc.msnn_buffer("gb_input")
        ghit = sc.msnn_buffer("gb_hit")
        scale = float(sc.info["scene_scale"])
        osc = ol.OracleScene(sc.info, sc.segments(), sc.env())
    n, nth = z["train_records"], z["every_nth"]
    assert n == 1024 and nth == 4 and z["frames"] == 1
    # one training pixel per block of every_nth pixels (hair_msnn.cu:206-209)
    np.testing.assert_array_equal(pix // nth, np.arange(n))
    np.testing.assert_array_equal(tin, gin[pix])
    rec = osc.msnn_records(0, 0, pix, scale, prec=1)
    hit_g, hit_o = ghit[pix], rec["hit"]
    assert (hit_g == hit_o).mean() >= 0.99
    both = (hit_g & 1).astype(bool) & (hit_o & 1).astype(bool)
    miss = ((hit_g & 1) == 0) & ((hit_o & 1) == 0)
    print(f"training records: {both.sum()} hits, {miss.sum()} misses")
    assert both.sum() > 200 and miss.sum() > 50
    np.testing.assert_array_equal(tgt[miss], 0.0)
    np.testing.assert_allclose(tin[both, 0:3], rec["input"][both, 0:3], rtol=0, atol=2e-5)
    np.testing.assert_allclose(tin[both, 3:9], rec["input"][both, 3:9], rtol=0, atol=2e-5)
    np.testing.assert_array_equal(tin[both, 9:12], rec["input"][both, 9:12])
    # the target is the difference of two path colours, so its rounding error
    # scales with the full colour, not with the difference
    ot = rec["target"][both]
    of = rec["full"][both]
    close = (np.abs(tgt[both] - ot) <= 1e-3 * np.maximum(np.abs(of), 1e-2)).all(-1)
    print(f"training targets agreeing with the oracle: {close.mean():.3f}")
    # full-depth paths: FP32 rounding that flips one sampling decision makes a
    # path diverge; a target agrees only if both its full path (about 0.9 of
    # C0 pixels at 40 vertices) and its short path agree
    assert close.mean() >= 0.80
    # the target is full - short: never negative in expectation
    assert tgt[both].mean() >= -1e-6 and ot.mean() >= -1e-6


@pytest.mark.parametrize("warmup", [6, 40])
def test_job_schedule_equals_per_pass_schedule(gpu, warmup):
    """Warm-up records traced on the job schedule (the default: a compacted
    wavefront refilled with new records as paths finish) are the per-pass
    schedule's bit for bit, and so are the network they train and the
    frames' records and images. 40 warm-up steps of 1024 records are two
    runs (32 + 8 steps) of more records than the slot's 4096 paths, so the
    wavefront is refilled and the second run traces while the first one's
    steps train."""
    cfg = cfg_small(records=1024, warmup=warmup)
    out = []
    for sched in ("stream", "passes"):
        with gpu.Scene(json_text=cfg) as sc:
            sc.set_pt_schedule(sched)
            sc.msnn_begin(BETA=2)
            sc.msnn_frames(10)
            got = {k: sc.msnn_buffer(k) for k in ("train_input", "train_target", "train_pixel", "nn_output",
                                                   "gb_color")}
            got["final"] = sc.msnn_image(0)
            got["short"] = sc.msnn_image(1)
            out.append(got)
    assert np.isfinite(out[0]["final"]).all() and (out[0]["train_target"] != 0).any()
    for k in out[0]:
        np.testing.assert_array_equal(out[0][k], out[1][k], err_msg=k)


def test_split_calls_equal_one_call(gpu):
    """Frames rendered in several calls, with a per-strand absorption upload
    between them (equal to the global value), give the image of one call bit
    for bit: every training batch a call starts is finished inside it."""
    cfg = cfg_small(records=1024, warmup=4)
    with gpu.Scene(json_text=cfg) as sc:
        sc.msnn_begin(BETA=1)
        sc.msnn_frames(10)
        one = sc.msnn_image(0)
    with gpu.Scene(json_text=cfg) as sc:
        sig = np.tile(np.asarray(sc.info["sigma_a"], np.float32), (int(sc.info["num_strands"]), 1))
        sc.msnn_begin(BETA=1)
        sc.msnn_frames(1)
        sc.set_strand_sigma_a(sig)
        sc.msnn_frames(6)
        sc.msnn_frames(3)
        split = sc.msnn_image(0)
    np.testing.assert_array_equal(split, one)


def test_trained_cache_gains_over_method_without_it(gpu):
    """What the trained network gains: at BETA 1 the truncated paths alone
    (the short image) miss all light past the second vertex; adding the
    cache's estimate brings the image closer to a 1024-spp path-traced
    reference than the short paths alone and than plain path tracing with
    the same number of samples per pixel. Wall times are printed."""
    import time
    cfg = cfg_small(records=1024, warmup=64)
    frames = 32
    with gpu.Scene(json_text=cfg) as sc:
        sc.set_seed_offset(1 << 20)
        ref = sc.render_path_tracing(1024)[..., :3].astype(np.float64)
        sc.set_seed_offset(0)
        sc.synchronize()
        t0 = time.perf_counter()
        pt = sc.render_path_tracing(frames)[..., :3].astype(np.float64)
        t_pt = time.perf_counter() - t0
        t0 = time.perf_counter()
        sc.msnn_begin(BETA=1)
        sc.msnn_frames(frames)
        t_ms = time.perf_counter() - t0
        final = sc.msnn_image(0)[..., :3].astype(np.float64)
        short = sc.msnn_image(1)[..., :3].astype(np.float64)
        hit = sc.msnn_buffer("gb_hit").reshape(final.shape[:2])

    def rmse(a):
        return float(np.sqrt(np.mean((a - ref) ** 2)))

    r_final, r_short, r_pt = rmse(final), rmse(short), rmse(pt)
    # the truncated paths miss the light beyond the second vertex: their
    # image is darker than the reference; the cache restores most of it
    hair = (hit & 1).astype(bool) & ~(hit & 2).astype(bool)
    b_short = short[hair].mean() / ref[hair].mean() - 1
    b_final = final[hair].mean() / ref[hair].mean() - 1
    print(f"RMSE vs 1024 spp after {frames} frames: cache {r_final:.4f}, short paths alone {r_short:.4f}, "
          f"plain PT {r_pt:.4f}; relative bias: short {b_short:+.4f}, with the cache {b_final:+.4f}; "
          f"wall time HairMSNN {t_ms:.3f} s (incl. warm-up) vs PT {t_pt:.3f} s")
    assert b_short < -0.05
    assert abs(b_final) < 0.5 * abs(b_short)
    assert r_final < r_short
    assert r_final < r_pt


def test_beta_zero_equals_beta_one(gpu):
    """Kernel beta = BETA - 1 and the break test `bounces > beta` after the
    second vertex's light make BETA 0 and BETA 1 the same truncation
    (render_hair_msnn.cu:1170, hair_msnn.cu:166-179): identical frames."""
    cfg = cfg_small(records=1024, warmup=4)
    imgs = []
    for beta in (0, 1):
        with gpu.Scene(json_text=cfg) as sc:
            sc.msnn_begin(BETA=beta)
            sc.msnn_frames(3)
            imgs.append((sc.msnn_image(0), sc.msnn_image(1)))
    np.testing.assert_array_equal(imgs[0][1], imgs[1][1])
    np.testing.assert_array_equal(imgs[0][0], imgs[1][0])


def test_init_weights_from_scene(gpu, tmp_path):
    """tcnn.init_weights (scene.cpp:330-331 -> render_hair_msnn.cu:109-110):
    a network saved from one HairMSNN run is loaded by the next scene that
    names it, before its warm-up; with no warm-up and no training the second
    run's cache is that network exactly, and its frames match a run whose
    network was set the same way."""
    cfg = cfg_small(records=1024, warmup=8)
    path = tmp_path / "cache.json"
    with gpu.Scene(json_text=cfg) as sc:
        sc.msnn_begin(BETA=1)
        sc.msnn_frames(2)
        sc.msnn_save_weights(str(path))
    import json
    saved = json.loads(path.read_text())["params"]
    cfg2 = json.loads(json.dumps(cfg))
    cfg2["hairmsnn"]["warmup_steps"] = 0
    cfg2["tcnn"] = {"config": "unused.json", "init_train": False, "init_weights": str(path)}
    with gpu.Scene(json_text=cfg2) as sc:
        sc.msnn_begin(BETA=1)
        sc.msnn_frames(1)
        sc.msnn_save_weights(str(tmp_path / "again.json"))
        net = sc.msnn_image(2)
    again = json.loads((tmp_path / "again.json").read_text())["params"]
    assert again == saved
    assert np.isfinite(net).all()
    cfg3 = json.loads(json.dumps(cfg2))
    cfg3["tcnn"]["init_weights"] = str(tmp_path / "missing.json")
    with gpu.Scene(json_text=cfg3) as sc:
        with pytest.raises(gpu.HmsnnError):
            sc.msnn_begin(BETA=1)


def test_training_pixel_shuffles(gpu):
    """The per-frame shuffle of trainIdxs (render_hair_msnn.cu:712-714) picks
    pixel i * every_nth + trainIdxs[i] % every_nth as training record i
    (hair_msnn.cu:206-209). trainIdxs is a permutation of 0..n-1, so over a
    frame every residue mod every_nth occurs exactly n / every_nth times;
    consecutive frames draw different permutations; the same seed draws the
    same sequence in a second context."""
    cfg = cfg_small(records=1024, warmup=2)

    def residues(frames):
        out = []
        with gpu.Scene(json_text=cfg) as sc:
            sc.msnn_begin(BETA=1)
            for _ in range(frames):
                sc.msnn_frames(1)
                z = sc.msnn_sizes()
                pix = sc.msnn_buffer("train_pixel")
                n, nth = z["train_records"], z["every_nth"]
                np.testing.assert_array_equal(pix // nth, np.arange(n))
                out.append(pix % nth)
        return out, n, nth

    a, n, nth = residues(4)
    for r in a:
        np.testing.assert_array_equal(np.bincount(r, minlength=nth), np.full(nth, n // nth))
    assert all((a[k] != a[k + 1]).mean() > 0.5 for k in range(3))
    b, _, _ = residues(4)
    for x, y in zip(a, b):
        np.testing.assert_array_equal(x, y)


def test_second_run_on_a_scene_equals_the_first(gpu):
    """hmsnn_msnn_begin keeps the buffers of an earlier run on the same scene:
    a second render, after one with another BETA and more frames than a
    training batch holds, is the first one bit for bit."""
    cfg = cfg_small(records=1024, warmup=40)
    with gpu.Scene(json_text=cfg) as sc:
        a = sc.render_hair_msnn(1, 11)
        sc.render_hair_msnn(3, 5)
        b = sc.render_hair_msnn(1, 11)
    np.testing.assert_array_equal(a, b)
