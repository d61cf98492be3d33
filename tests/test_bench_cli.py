"""bench.py's command line on the CPU: the one-GPU contract (no GPU needed,
the checks run before anything touches the device)."""
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _bench(*args):
    return subprocess.run([sys.executable, os.path.join(ROOT, "bench.py"), *args], cwd=ROOT,
                          capture_output=True, text=True, timeout=120)


def test_more_than_one_gpu_is_refused():
    r = _bench("--gpus", "2")
    assert r.returncode == 2
    assert "one GPU" in r.stderr
    assert r.stdout == ""  # no JSON line


def test_help_lists_the_contract_flags():
    r = _bench("--help")
    assert r.returncode == 0
    for flag in ("--gpus", "--steps", "--warmup", "--serve-lanes", "--serve-path-split"):
        assert flag in r.stdout


def test_roofline_names_the_profiled_kernel():
    """The roofline's counters are those of the kernel it names: the profile
    that it cites names that kernel, and at the 32.0 ms the launch took under
    the counters its instructions stay below the nominal issue rate."""
    import bench
    r = bench.lookup_roofline(4096, 131072, 12, 890.85, [6.2, 32.0, 8.0])
    text = open(os.path.join(ROOT, r["counters_profile"])).read()
    assert r["kernel"] in text
    assert 0.5 < r["issue"]["frac"] < 1.0
    assert r["hbm"]["unique_bytes"] < r["hbm"]["measured_bytes"]
    assert bench.lookup_roofline(64, 2048, 12, 890.85, [6.2, 32.0, 8.0])["counters_profile"] is None
