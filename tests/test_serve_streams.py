"""Which stream the serving loop puts its work on (no GPU): tests/cpp/serve_streams_check.cpp runs the loop over the CPU
stand-in for the device with its launches and runtime calls recorded, under the address sanitizer."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
OUT = os.path.join(ROOT, "hypercraft_amd", "_build", "sanitize", "serve_streams_check")


def test_streams_of_the_serving_loop():
    subprocess.run(["make", "-s", "-C", os.path.join(ROOT, "tests", "cpp"), OUT], check=True, timeout=600)
    p = subprocess.run([OUT], capture_output=True, text=True, timeout=120)
    assert p.returncode == 0 and "all checks passed" in p.stdout, (p.stdout + p.stderr)[-4000:]
