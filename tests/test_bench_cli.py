"""bench.py's command-line contract on the CPU: one GPU only, and no GPU work before the check."""
import glob
import json
import os
import re
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_more_than_one_gpu_is_refused_with_a_message():
    r = subprocess.run([sys.executable, os.path.join(ROOT, "bench.py"), "--gpus", "2"], capture_output=True,
                       text=True, timeout=120)
    assert r.returncode != 0
    assert "one GPU" in (r.stdout + r.stderr)
    assert r.stdout.strip() == "" or not r.stdout.lstrip().startswith("{")  # no result line


def test_world_size_above_one_is_refused():
    env = dict(os.environ, WORLD_SIZE="2")
    r = subprocess.run([sys.executable, os.path.join(ROOT, "bench.py")], capture_output=True, text=True,
                       timeout=120, env=env)
    assert r.returncode != 0
    assert "one GPU" in (r.stdout + r.stderr)


def bench():
    sys.path.insert(0, ROOT)
    try:
        import bench as b
    finally:
        sys.path.pop(0)
    return b


def test_kernel_of_a_launch_label():
    b = bench()
    report = ["march_frame 1920x1080 level=10 beam=1: one-ray-per-lane 0.15 ms refill 0.16 ms -> one-ray-per-lane-8x8-bands",
              "march_frame_batch S=4 64x64 beam=1: 16x16 0.1 ms -> 8x8", "march_rays variant=0 level=10 R~2^4: -> one-ray-per-lane",
              "march_rays variant=1 level=10 R~2^20: one-ray-per-lane 0.3 ms refill 0.2 ms -> refill"]
    assert b.kernel_of("march_frame", report) == "march_frame_kernel<1u,1u,true>"
    assert b.kernel_of("march_frame", []) == "march_frame_kernel<1u,1u,false>"
    assert b.kernel_of("march_rays5", report) == "march_pool<1,256u,ExplicitRays>"
    assert b.kernel_of("march_rays5", report[:3]) == "march_rays_kernel<1>"
    assert b.kernel_of("march_rays6", report) == "march_rays_kernel<0>"
    assert b.kernel_of("vox_fill", report) == "vox_fill"


def test_counters_are_those_of_the_kernel_that_runs(tmp_path, monkeypatch):
    b = bench()
    monkeypatch.setattr(b, "ROOT", str(tmp_path))
    os.makedirs(tmp_path / "profiles")
    with open(tmp_path / "profiles" / "traffic_march_rays5_c2.json", "w") as f:
        json.dump({"rocprof_name": "march_pool<1,256u,ExplicitRays>", "bytes_per_launch": 7}, f)
    assert b.counter("traffic", "march_rays5", 2, "march_pool<1,256u,ExplicitRays>", "bytes_per_launch") == 7
    assert b.counter("traffic", "march_rays5", 2, "march_rays_kernel<1>", "bytes_per_launch") is None
    assert b.counter("traffic", "march_rays5", 3, "march_pool<1,256u,ExplicitRays>", "bytes_per_launch") is None


def test_recorded_counters_name_kernels_of_the_sources():
    csrc = os.path.join(ROOT, "sparsevoxeloctree_amd", "csrc")
    text = "".join(open(os.path.join(csrc, f)).read() for f in os.listdir(csrc))
    for path in glob.glob(os.path.join(ROOT, "profiles", "*_c[0-9].json")):
        name = json.load(open(path))["rocprof_name"].split("<")[0]
        assert re.search(r"\b%s\(" % name, text), "%s: no kernel %s" % (os.path.basename(path), name)
