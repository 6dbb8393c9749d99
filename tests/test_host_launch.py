"""What the library's entry points launch, and how they hold their workspaces,
checked without a GPU: tests/cpp/host_launch (built by
tests/cpp/build_sanitize.py) links the library's host code, launchers included,
under AddressSanitizer and UndefinedBehaviorSanitizer against a stand-in for the
HIP host calls that records launches.  Each check says in
tests/cpp/host_launch.cpp what it holds the library to."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
BINARY = os.path.join(HERE, "cpp", "host_launch")


def _binary():
    if not os.path.exists(BINARY):
        sys.path.insert(0, os.path.join(HERE, "cpp"))
        import build_sanitize

        build_sanitize.build()
    return BINARY


@pytest.mark.parametrize("check", ["f32_offsets", "graph_workspace", "stream_locks", "grid_limits",
                                   "overlapping_outputs", "mlp_wrappers"])
def test_host_launch(check, tmp_path):
    if subprocess.run(["g++", "--version"], capture_output=True).returncode != 0:
        pytest.skip("no g++")
    env = dict(os.environ)
    env["ASAN_OPTIONS"] = "detect_leaks=0:halt_on_error=1"  # workspaces live until the process ends
    env["UBSAN_OPTIONS"] = "halt_on_error=1:print_stacktrace=1"
    r = subprocess.run([_binary(), check], capture_output=True, text=True, env=env, cwd=tmp_path, timeout=300)
    out = r.stdout + r.stderr
    assert "AddressSanitizer" not in out and "runtime error" not in out, out[-4000:]
    assert r.returncode == 0 and f"{check} ok" in r.stdout, out[-4000:]
