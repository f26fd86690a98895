"""The host layer's pools of device blocks, events and result blocks with two devices, and the limit of a download's wait:
tests/native/two_devices.cpp, a program with stand-ins for the HIP calls.  Host only."""
import os
import subprocess

import selftest_lib


def test_blocks_and_events_go_back_to_their_own_device():
    selftest_lib.lib()
    exe = os.path.join(os.path.dirname(os.path.abspath(__file__)), "native", "two_devices")
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stderr


def test_masked_streams_that_cannot_be_made():
    """tests/native/lane_streams.cpp: every call that makes a group of streams fails in turn; nothing is left behind, and nothing is tried again."""
    selftest_lib.lib()
    exe = os.path.join(os.path.dirname(os.path.abspath(__file__)), "native", "lane_streams")
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stderr


def test_staging_matrices_of_sparse_blocks():
    """tests/native/sparse_block.cpp: two matrices take turns; one does where the device has no room for the second, and where it is so large that
    a second would take gigabytes.  Every block is what its rows' products are, and every matrix empty when it is used."""
    selftest_lib.lib()
    exe = os.path.join(os.path.dirname(os.path.abspath(__file__)), "native", "sparse_block")
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stderr
