"""bench.py without a GPU."""
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_lds_option_is_accepted():
    """Refused for its value of --gpus, not for --lds."""
    r = subprocess.run([sys.executable, os.path.join(ROOT, "bench.py"), "--lds", "0", "--gpus", "2"],
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 2 and "one GPU" in r.stderr
