"""Copies through the pinned ring on the CPU, over a stand-in for the HIP runtime
whose stream runs its copies late and whose hipHostFree waits for nothing: a
download that needs a larger ring than the upload queued before it must not give
the ring back while the upload's copies still read it."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
KB, MB = 1 << 10, 1 << 20


@pytest.fixture(scope="module")
def host_copies(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("copies") / "host_copies")
    src = os.path.join(HERE, "hip_stub", "host_copies.cpp")
    subprocess.run([shutil.which("g++") or "g++", "-std=c++17", "-O1", "-Wall", "-pthread",
                    "-I", os.path.dirname(src), src, "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("up,down", [
    (32, 16), (32, MB), (64 * KB, 8 * MB), (64 * KB + 1, MB - 1), (200 * KB, 20 * MB),
    (MB + 5, 9 * MB + 3), (5 * MB, 5 * MB), (40 * MB + 7, 2 * MB), (3 * MB, 64 * MB + 11)])
def test_download_after_upload(host_copies, up, down):
    r = subprocess.run([host_copies, str(up), str(down)], capture_output=True, text=True,
                       timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr


@pytest.mark.parametrize("up,down", [(32, 16), (32, MB), (200 * KB, 20 * MB), (40 * MB + 7, 2 * MB)])
def test_without_pinned_memory(host_copies, up, down):
    """The same answers, through ordinary memory."""
    r = subprocess.run([host_copies, str(up), str(down), "nopin"], capture_output=True, text=True,
                       timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
