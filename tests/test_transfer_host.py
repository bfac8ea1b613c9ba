"""Host logic of the large transfers (csrc/lbm_transfer.hip) over a stand-in
for the HIP runtime (tests/cpp/transfer_fake.cpp): CPU only."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT

ROCM = "/opt/rocm/include"


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    if shutil.which("g++") is None or not os.path.exists(os.path.join(ROCM, "hip", "hip_runtime.h")):
        pytest.skip("needs g++ and the HIP headers")
    exe = str(tmp_path_factory.mktemp("transfer") / "transfer_fake")
    r = subprocess.run(["g++", "-std=c++20", "-O1", "-g", "-D__HIP_PLATFORM_AMD__", f"-I{ROCM}", "-x", "c++",
                        os.path.join(ROOT, "tests", "cpp", "transfer_fake.cpp"), "-o", exe, "-pthread"],
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-3000:]
    return exe


def _holds(driver, scenario):
    r = subprocess.run([driver, scenario], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr


def test_bytes(driver):
    """Whole chunks and a remainder, both directions."""
    _holds(driver, "bytes")


def test_lanes_start_behind_earlier_work(driver):
    """The threads start once the stream has reached the copy: they do not
    wait for the steps queued before it."""
    _holds(driver, "earlier")


def test_failed_lane_leaves_nothing_in_flight(driver):
    """After a lane has failed, the copies of all lanes are waited for before
    the chunks can be taken by another call or freed."""
    _holds(driver, "failure")


def test_device_view_covers_the_whole_range(driver):
    """A kernel may write host memory only if all of it is page-locked."""
    _holds(driver, "view")


def test_small_uploads_are_queued(driver):
    """The caller queues the kernel that reads them and waits once, behind it."""
    _holds(driver, "queued")


def test_uploads_take_threads_where_they_are_faster(driver):
    _holds(driver, "thresholds")
