"""The benchmark's command line on the CPU: a request for more than one GPU
ends with a message and exit status 2 before anything touches a device, and
the options parse.  (The GPU legs themselves run in the benchmark.)"""
import json
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def run_bench(*args):
    return subprocess.run([sys.executable, os.path.join(ROOT, "bench.py"), *args], capture_output=True, text=True,
                          timeout=120, cwd=ROOT)


def test_more_than_one_gpu_is_refused():
    r = run_bench("--gpus", "2")
    assert r.returncode == 2
    line = json.loads(r.stdout.strip().splitlines()[-1])
    assert line["n_gpus"] == 2 and "one MI355X" in line["error"]


def test_options_parse():
    sys.path.insert(0, ROOT)
    import bench
    argv = sys.argv
    try:
        sys.argv = ["bench.py", "--only-c4", "--c4-eager", "eager_single", "--steps", "2", "--no-cpu"]
        a = bench.parse()
    finally:
        sys.argv = argv
    assert a.only_c4 and a.c4_eager == "eager_single" and a.steps == 2 and a.no_cpu and a.gpus == 1


def test_traffic_of_another_kernel_is_not_reported(tmp_path):
    """the committed counter summary is printed only for the kernel it was
    measured on: no figure once the deposit's source is another, or the
    summary does not say which it was; comments do not matter"""
    sys.path.insert(0, ROOT)
    import bench
    src = tmp_path / "qpad_amd" / "csrc"
    src.mkdir(parents=True)
    for name in ("k_plasma.hip", "wave_reduce.h", "conv.h", "qpad_internal.h"):
        (src / name).write_text("int kernel;  // " + name + "\n")
    (tmp_path / "profiles").mkdir()
    summary = tmp_path / "profiles" / "k_amjdeposit_c2_hbm_traffic.txt"
    head = "of k_amjdeposit<2, false, 4>\n"
    assert bench.measured_traffic("c2", 2, str(tmp_path)) is None
    summary.write_text(head + "traffic_bytes_per_launch: 41387494\n")
    assert bench.measured_traffic("c2", 2, str(tmp_path)) is None
    summary.write_text(head + f"kernel_source: {bench.kernel_source_hash(str(tmp_path))}\n"
                       "traffic_bytes_per_launch: 41387494\n")
    assert bench.measured_traffic("c2", 2, str(tmp_path)) == 41387494.0
    assert bench.measured_traffic("c2", 4, str(tmp_path)) is None and bench.measured_traffic("c3", 2, str(tmp_path)) is None
    (src / "k_plasma.hip").write_text("// another comment\nint kernel;\n")
    assert bench.measured_traffic("c2", 2, str(tmp_path)) == 41387494.0
    (src / "k_plasma.hip").write_text("int kernel = 1;\n")
    assert bench.measured_traffic("c2", 2, str(tmp_path)) is None
