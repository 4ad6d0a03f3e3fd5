"""The copies between caller memory and the device (convector_amd/csrc/
copies.hip), compiled for the host against a HIP runtime of plain host memory
(tests/host_hip) whose streams run their work as early or as late as they may:
tests/copies_check.cpp holds the checks, one test here per check."""
import os
import subprocess

import pytest

TESTS = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("copies") / "copies_check")
    r = subprocess.run(["g++", "-O2", "-g", "-std=c++17", "-Wall", "-Wno-unused-function", "-pthread",
                        "-I", os.path.join(TESTS, "host_hip"),
                        os.path.join(TESTS, "copies_check.cpp"), "-o", exe],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr

    def run(name):
        r = subprocess.run([exe, name], capture_output=True, text=True, timeout=100)
        assert r.returncode == 0, r.stdout + r.stderr

    return run


def test_pieces_and_boundaries(check):
    check("shapes")


def test_pieces_are_coherent(check):
    check("coherent")


def test_any_current_device(check):
    check("devices")


@pytest.mark.parametrize("name", ["threads", "crowd", "settled"])
def test_concurrent_copies(check, name):
    check(name)


def test_neighbours_share_transfers(check):
    check("many")
