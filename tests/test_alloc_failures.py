"""What the contexts do with their buffers and streams, on the CPU: when the
device has no memory left, after a begin that failed, when they grow. The
library runs on tests/fake_hip.c (host memory, launches that do nothing), which
fails allocations on request and counts them. Each script runs in a process of
its own."""
import json
import subprocess
import sys
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent

PRELUDE = '''
import ctypes as C, json, sys
fake = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)  # before the library: its symbols are found first
fake.fake_bytes.restype = C.c_size_t
fake.fake_limit.argtypes = [C.c_size_t]
fake.fake_live.restype = C.c_long
sys.path.insert(0, sys.argv[2])
import hairmsnn_amd as hm
from hairmsnn_amd._lib import load
lib = load()
cfg = json.load(open(sys.argv[2] + "/hairmsnn_amd/scenes/c0_hairball.json"))
cfg["integrator"].update(width=16, height=8)
cfg["hair"]["procedural"].update(strands=1, segments=1)  # a tree of one leaf needs no kernel's output
def scene(w=16, h=8, **hair):
    cfg["integrator"].update(width=w, height=h)
    return hm.Scene(json_text=cfg)
def call(f, *a):
    try:
        f(*a)
        return ""
    except hm._lib.HmsnnError as e:
        return str(e)
'''


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    so = tmp_path_factory.mktemp("fake") / "libfakehip.so"
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-o", str(so), str(ROOT / "tests" / "fake_hip.c")], check=True)

    def run(script: str):
        r = subprocess.run([sys.executable, "-c", PRELUDE + script, str(so), str(ROOT)], capture_output=True, text=True,
                           timeout=300)
        assert r.returncode == 0, r.stderr[-2000:]
        return json.loads(r.stdout.strip().splitlines()[-1])
    return run


@pytest.mark.parametrize("entry", ["trace_stats", "pt_passes"])
def test_failed_allocation_leaves_no_partial_buffers(fake, entry):
    """Every allocation of a first render fails in turn: the call reports it,
    and the same call afterwards makes everything that was missing (a set of
    path buffers with null arrays would fault in the kernels). The launches do
    nothing here, so a streamed call ends by reporting that no pass was
    accumulated."""
    out = fake(f'''
done = "" if "{entry}" == "trace_stats" else "0 of 1 passes accumulated"
base = scene(); before = fake.fake_live(); e = call(base.{entry}, 1); whole = fake.fake_live() - before
assert (done in e) if done else not e, e
base.close()
bad = []
for k in range(whole):
    sc = scene(); before = fake.fake_live()
    fake.fake_fail_after(k)
    first = call(sc.{entry}, 1)
    fake.fake_fail_after(-1)
    again = call(sc.{entry}, 1)
    got = fake.fake_live() - before
    if "ENOMEM" not in first or ((done not in again) if done else again) or got != whole: bad.append([k, first, again, got])
    sc.close()
print(json.dumps(dict(whole=whole, bad=bad, left=fake.fake_live())))
''')
    assert out["whole"] > 40
    assert out["bad"] == []
    assert out["left"] == 0


def test_path_buffers_follow_the_call_and_the_memory(fake):
    """A call of one pass makes buffers for a frame's paths, not for the ring's
    16 passes, in either schedule; a longer call grows them; and where memory
    is short it takes fewer paths (half as many, down to a frame's) instead of
    failing. Per path the buffers are 300 to 400 bytes, the ring and the image
    288 bytes a pixel."""
    out = fake('''
n = 256 * 128
def used(sc, passes):
    e = call(sc.pt_passes, passes)
    assert "of %d passes accumulated" % passes in e, e
    return (fake.fake_bytes() - base) / n
r = {}
sc = scene(256, 128); base = fake.fake_bytes(); r["one"] = used(sc, 1); r["all"] = used(sc, 40); r["again"] = used(sc, 1); sc.close()
sc = scene(256, 128); base = fake.fake_bytes(); sc.set_pt_schedule("passes"); sc.set_pass_concurrency(1); sc.pt_passes(1)
r["passes"] = (fake.fake_bytes() - base) / n; sc.close()
sc = scene(256, 128); base = fake.fake_bytes(); sc.trace_stats(1); spill = fake.fake_bytes() - base
fake.fake_limit(fake.fake_bytes() + n * (288 + 400 * 5)); r["short"] = used(sc, 16); fake.fake_limit(0); r["kept"] = used(sc, 16); sc.close()
r["left"] = fake.fake_live()
print(json.dumps(r))
''')
    print(out)
    assert out["left"] == 0
    assert out["one"] < 288 + 400 + 400 and out["passes"] < 32 + 400 + 400
    assert out["all"] > out["one"] + 15 * 300 and out["again"] == out["all"]
    assert out["one"] < out["short"] < out["all"] / 2 and out["kept"] == out["short"]


@pytest.mark.parametrize("kind", ["msnn", "nrc"])
def test_failed_begin_shows_no_earlier_image(fake, kind):
    """The renderers keep their buffers from one begin to the next. A begin that
    fails (the weight file is gone) refuses the image afterwards, as on a new
    context, instead of returning the earlier run's; the next good one works."""
    begin = "sc.msnn_begin(1)" if kind == "msnn" else "sc.nrc_begin()"
    out = fake(f'''
import os, tempfile
w = os.path.join(tempfile.mkdtemp(), "w.json")
sc = scene(); {begin}; sc.{kind}_save_weights(w); sc.close()
cfg["tcnn"] = {{"config": "unused.json", "init_train": False, "init_weights": w}}
sc = scene(); {begin}; first = call(sc.{kind}_image)
os.rename(w, w + "x")
bad = call(lambda: {begin}); image = call(sc.{kind}_image)
os.rename(w + "x", w); {begin}; last = call(sc.{kind}_image); sc.close()
print(json.dumps(dict(first=first, bad=bad, image=image, last=last, left=fake.fake_live())))
''')
    print(out)
    assert not out["first"] and not out["last"] and out["left"] == 0
    assert "EIO" in out["bad"] and "EINVAL" in out["image"]


def test_nrc_slots_keep_their_stream_when_they_grow(fake):
    """Calls of more frames make larger slots. They stay on the streams made at
    the begin, which mostly have a hardware queue each. A growth that finds no
    memory leaves the slot and its stream as they were."""
    out = fake('''
sc = scene(); sc.nrc_begin(); sc.nrc_frames(1); a = fake.fake_streams()
sc.nrc_frames(3); sc.nrc_frames(9); b = fake.fake_streams()
fake.fake_fail_after(5); sc.nrc_frames(16); fake.fake_fail_after(-1); sc.nrc_frames(2); sc.close()
print(json.dumps(dict(a=a, b=b, left=fake.fake_live())))
''')
    assert out["a"] == out["b"] and out["left"] == 0
