"""bench.py's options and the traffic figure it takes from the profiles."""
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_lds_option_is_accepted():
    """Refused for its value of --gpus, not for --lds."""
    r = subprocess.run([sys.executable, os.path.join(ROOT, "bench.py"), "--lds", "0", "--gpus", "2"],
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 2 and "one GPU" in r.stderr


def test_traffic_only_for_the_steps_it_was_measured_over():
    sys.path.insert(0, ROOT)
    import bench
    shape = {"zm": 16, "rows": 8, "xcd": 0}
    assert bench.measured_traffic("256x256x512", shape, 5000, 50) > 1.0e9
    for steps, warmup in ((20, 50), (5000, 5)):
        assert bench.measured_traffic("256x256x512", shape, steps, warmup) is None
    # FP32-deviation steps write the same at any state
    assert bench.measured_traffic("256x256x512", shape, 20, 5, "fp32") > 1.0e9
