"""Neural radiance caching on the GPU (render_nrc.cu:640-701, cuda/nrc.cu):
the G_BUFFER pass against the oracle's nrcTracePaths restatement per pixel,
the c = 0 case against the plain path tracer bit for bit, the RENDER
composite and the training targets."""
import json
from pathlib import Path

import numpy as np
import pytest

from tests import oracle_lib as ol

pytestmark = pytest.mark.gpu
SCENES = Path(__file__).resolve().parent.parent / "hairmsnn_amd" / "scenes"


def cfg_small(w=64, h=64, records=2560, c=0.01, all_unbiased=False, path_v2=40):
    cfg = json.loads((SCENES / "c0_hairball.json").read_text())
    cfg["integrator"].update({"width": w, "height": h, "path_v1": 1, "path_v2": path_v2})
    cfg["nrc"] = {"train_records": records, "c": c, "all_unbiased": all_unbiased}
    cfg["tcnn"] = {"config": "unused.json", "init_train": True}
    return cfg


def pixel_flags(idx, every_nth, npx, all_unbiased=False):
    """Training / unbiased flags per pixel (cuda/nrc.cu:371-377)."""
    flags = np.zeros(npx, np.uint8)
    px = np.arange(npx)
    tr = px // every_nth
    ok = tr < len(idx)
    train = np.zeros(npx, bool)
    train[ok] = (px[ok] % every_nth) == (idx[tr[ok]] % every_nth)
    flags[train] |= 1
    unb = train & ((tr % 16 == 0) | all_unbiased)
    flags[unb] |= 2
    return flags


def close(a, b, rtol=1e-3, floor=1e-2):
    return (np.abs(a - b) <= rtol * np.maximum(np.abs(b), floor)).all(-1)


def record_close(a, b):
    """Cache-query / training records: position / scene scale and wo to 1e-4;
    the shading normal to 2e-2, since an FP32 hit point on a 0.005-radius
    fibre is uncertain by ~1e-5 and the normal by ~1e-5 / r (the oracle's own
    FP32 and FP64 runs differ that much)."""
    return (np.abs(a[..., :6] - b[..., :6]) <= 1e-4).all(-1) & (np.abs(a[..., 6:9] - b[..., 6:9]) <= 2e-2).all(-1)


def test_c_zero_gbuffer_is_first_vertex_pass(gpu):
    with gpu.Scene(json_text=cfg_small(path_v2=1)) as st:
        st.pt_reset()
        st.pt_passes(1)
        first = st.last_pass()[..., :3].reshape(-1, 3).copy()
    with gpu.Scene(json_text=cfg_small(c=0.0)) as sc:
        sc.nrc_begin()
        sc.nrc_frames(1)
        rad = sc.nrc_buffer("gb_radiance")[:, :3]
        beta = sc.nrc_buffer("gb_beta")[:, :3]
        hit = sc.nrc_buffer("gb_hit")
    ok = np.isfinite(first).all(-1)
    np.testing.assert_array_equal(rad[ok], first[ok])
    queried = np.abs(beta).sum(-1) > 0
    print(f"c = 0: {hit.sum()} hits, {queried.sum()} cache queries at the second vertex")
    assert queried.sum() > 0.2 * hit.sum()
    assert not queried[hit == 0].any()


# Thresholds: the oracle's FP32 and FP64 runs of the same frame agree on
# 0.963 (c = 0.01) and 0.887 (c = 1, every suffix unbiased) of the pixels at
# these tolerances; longer paths leave more room for FP32 chaos.
@pytest.mark.parametrize("c,all_unbiased,min_agree", [(0.01, False, 0.93), (1.0, True, 0.82)])
def test_gbuffer_matches_oracle(gpu, c, all_unbiased, min_agree):
    cfg = cfg_small(c=c, all_unbiased=all_unbiased, records=10240)  # 256 training pixels, one in 16
    with gpu.Scene(json_text=cfg) as sc:
        sc.nrc_begin()
        sc.nrc_frames(1)
        z = sc.nrc_sizes()
        b = {k: sc.nrc_buffer(k) for k in ("gb_radiance", "gb_beta", "gb_hit", "query", "train_idx",
                                           "train_bounces", "train_hit", "train_input", "train_target", "cache")}
        osc = ol.OracleScene(sc.info, sc.segments(), sc.env())
        scale = float(sc.info["scene_scale"])
    npx = 64 * 64
    assert z["train_pixels"] == 10240 // 40 and z["every_nth"] == npx // z["train_pixels"]
    flags = pixel_flags(b["train_idx"], z["every_nth"], npx, all_unbiased)
    o = osc.nrc_gbuffer(0, flags, c=c, scene_scale=scale, prec=1)
    assert (b["gb_hit"] == o["gb_hit"]).mean() > 0.999
    agree = close(b["gb_radiance"][:, :3], o["rad"]) & close(b["gb_beta"][:, :3], o["beta"])
    agree &= record_close(b["query"][:npx, :9], o["q"])
    frac = agree.mean()
    nq = (o["query"] == 1).sum()
    print(f"c={c}: per-pixel G-buffer agreement {frac:.4f}; oracle queries {nq}, GPU queries "
          f"{(np.abs(b['gb_beta'][:, :3]).sum(-1) > 0).sum()}")
    assert frac >= min_agree
    assert nq > 100
    # training pixels: bounce counts, suffix queries, inputs and targets (with
    # the GPU's network outputs as the cache values)
    tpx = np.flatnonzero(flags & 1)
    tr = tpx // z["every_nth"]
    same_b = (b["train_bounces"][tr] == o["bounces"][tpx]) & (b["train_hit"][tr] == o["tb_hit"][tpx])
    print(f"training pixels {len(tpx)}: bounce/suffix agreement {same_b.mean():.4f}")
    assert same_b.mean() >= 0.9
    checked = candidates = 0
    for k, (t, p) in enumerate(zip(tr, tpx)):
        B = int(o["bounces"][p])
        # records beyond the path stay zero
        assert not b["train_target"][t * 40 + max(B, 0):(t + 1) * 40].any() or not same_b[k]
        if not (agree[p] and same_b[k] and o["gb_hit"][p] and B > 0):
            continue
        candidates += 1
        rec = o["rec"][p]
        unbiased = (t % 16 == 0) or all_unbiased
        cr = b["cache"][npx + t] if (o["tb_hit"][p] and not unbiased) else np.zeros(3)
        want = []
        for bb in range(B):
            color, beta = np.zeros(3), np.ones(3)
            for sub in range(bb, B):
                color = color + beta * rec[sub, 9:12]
                beta = beta * rec[sub, 12:15]
            want.append(color + beta * cr)
        got = b["train_target"][t * 40:t * 40 + B]
        gin = b["train_input"][t * 40:t * 40 + B, :9]
        if close(got, np.array(want), 2e-3, 1e-2).all() and record_close(gin, rec[:B, :9]).all():
            checked += 1
    print(f"training targets reproduced for {checked} of {candidates} pixels with recorded vertices")
    assert candidates >= 10
    assert checked >= 0.8 * candidates


def test_render_composite_and_frame_stats(gpu):
    cfg = cfg_small()
    with gpu.Scene(json_text=cfg) as sc:
        sc.nrc_begin()
        st = sc.nrc_frames(1)
        img1 = sc.nrc_image()[..., :3].reshape(-1, 3).astype(np.float64)
        rad = sc.nrc_buffer("gb_radiance")[:, :3].astype(np.float64)
        beta = sc.nrc_buffer("gb_beta")[:, :3].astype(np.float64)
        cache = sc.nrc_buffer("cache")[:64 * 64].astype(np.float64)
        st8 = sc.nrc_frames(8)
        img9 = sc.nrc_image()
    cache = np.where(np.isnan(cache).any(-1, keepdims=True), 0.0, np.maximum(cache, 0.0))
    want = rad + beta * cache
    want[np.isnan(want).any(-1)] = 0.0
    np.testing.assert_allclose(img1, want, rtol=2e-6, atol=1e-7)
    print(st, st8)
    assert st["frames"] == 1 and st["train_steps"] == 1 and st8["train_steps"] == 9
    assert st["cache_queries"] > 0 and st["train_records_used"] > 0
    assert np.isfinite(img9).all()


def test_second_run_on_a_scene_equals_the_first(gpu):
    """hmsnn_nrc_begin keeps the buffers of an earlier run on the same scene:
    image and trained weights of a second run, after one with other
    parameters, are the first one's bit for bit."""
    out = []
    with gpu.Scene(json_text=cfg_small()) as sc:
        for c in (None, 0.5, None):
            sc.nrc_begin()
            if c is not None:
                sc.nrc_set_params(c, True)
            sc.nrc_frames(7)
            out.append((sc.nrc_image(), sc.nrc_weights()))
    np.testing.assert_array_equal(out[0][0], out[2][0])
    np.testing.assert_array_equal(out[0][1], out[2][1])


@pytest.mark.parametrize("frames", [2, 16, 17, 35])
def test_frames_of_one_call_equal_frames_of_many(gpu, frames):
    """A call traces up to 16 frames as one pass, in batches of like sizes on
    two sets of buffers; image, weights and the last frame's buffers are those
    of single-frame calls bit for bit, also on buffers that grew meanwhile."""
    names = ("train_idx", "query", "gb_radiance", "gb_beta", "gb_hit", "train_input", "train_target", "train_bounces")

    def result(sc):
        return [sc.nrc_image(), sc.nrc_weights()] + [sc.nrc_buffer(n) for n in names]

    with gpu.Scene(json_text=cfg_small(w=40, h=32, records=1280)) as sc:
        sc.nrc_begin()
        for _ in range(frames):
            one = sc.nrc_frames(1)
        single = result(sc)
        sc.nrc_begin()
        all_ = sc.nrc_frames(frames)
        whole = result(sc)
        sc.nrc_begin()
        sc.nrc_frames(frames // 2)
        sc.nrc_frames(frames - frames // 2)
        halves = result(sc)
    assert one["train_steps"] == all_["train_steps"] == frames
    assert one["cache_queries"] == all_["cache_queries"] and one["train_records_used"] == all_["train_records_used"]
    for a, b, c in zip(single, whole, halves):
        np.testing.assert_array_equal(a, b)
        np.testing.assert_array_equal(a, c)
