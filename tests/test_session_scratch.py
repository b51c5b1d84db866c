"""What a session takes beside its caches: Q slots for the layers that are launched
together, where there is memory for them."""

import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))


def test_session_creation_with_little_memory():
    program = os.path.join(HERE, "native", "session_scratch")
    if not os.path.exists(program):
        subprocess.run([sys.executable, os.path.join(HERE, "native", "build.py")], check=True, timeout=120)
    res = subprocess.run([program], capture_output=True, text=True, timeout=60)
    assert res.returncode == 0, res.stdout + res.stderr
