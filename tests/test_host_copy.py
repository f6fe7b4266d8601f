"""channel_amd/csrc/host_copy.hip on the CPU against a stand-in for the HIP runtime
(tests/fake_hip): which transfers are staged, that their chunks arrive whole, that the
slots are kept and given back, and that an owner that could not pin its slots goes on
without them.  Once plain, once under ThreadSanitizer."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "channel_amd", "csrc")
MB = 1 << 20
CHUNK, SLOTS = 2 * MB, 16


@pytest.fixture(scope="module", params=["plain", "threads"])
def driver(request, tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ is not installed")
    out = str(tmp_path_factory.mktemp("host_copy") / "driver")
    cmd = [gxx, "-std=c++17", "-O2", "-g", "-pthread", "-I" + os.path.join(HERE, "fake_hip"), "-I" + CSRC, "-x", "c++",
           os.path.join(CSRC, "host_copy.hip"), os.path.join(HERE, "host_copy_driver.cpp"), "-o", out]
    if request.param == "threads":
        cmd.insert(1, "-fsanitize=thread")
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr

    def run(*args):
        env = dict(os.environ)
        env.pop("LD_PRELOAD", None)  # the sanitizer's runtime comes first
        r = subprocess.run([out] + list(args), capture_output=True, text=True, env=env)
        assert r.returncode == 0, r.stdout + r.stderr[-4000:]
        return [ln.split() for ln in r.stdout.splitlines()]

    return run


def chunks(n):
    return -(-n // CHUNK)


def test_small_transfers_go_directly(driver):
    for row in driver("h%d" % (8 * MB - 4), "d%d" % (96 * MB - 4), "p%d" % (40 * MB)):
        assert row == ["1", "0", "1", "0", "0"]


@pytest.mark.parametrize("n", [8 * MB, 8 * MB + 4, 31 * MB + 20, 32 * MB, 40 * MB + 8])
def test_to_host_is_staged_once_it_has_moved_the_slots_size(driver, n):
    rows = driver(*(["h%d" % n] * 6))
    moved, held = 0, 0
    for row in rows:
        moved += n
        assert row[0] == "1"
        if moved <= SLOTS * CHUNK:
            assert row[1:] == ["0", "1", "0", "0"]
            continue
        want = min(chunks(n), SLOTS)
        assert row[1:] == [str(chunks(n)), "0", str(want), str(want - held)]
        held = want


def test_to_device_is_staged_once_the_slots_pay(driver):
    n = 97 * MB + 12  # a sixth of what goes to the device counts
    rows = driver("d%d" % n, "d%d" % n, "g")
    assert rows[0] == ["1", "0", "1", "0", "0"]
    assert rows[1] == ["1", str(chunks(n)), "0", str(SLOTS), str(SLOTS)]
    assert rows[2] == ["held", "0", "0"]
    n = 193 * MB  # a first one as large as that
    rows = driver("d%d" % n, "d%d" % (97 * MB), "d%d" % (96 * MB - 4))
    assert rows[0] == ["1", str(chunks(n)), "0", str(SLOTS), str(SLOTS)]
    assert rows[1] == ["1", str(chunks(97 * MB)), "0", str(SLOTS), "0"]
    assert rows[2] == ["1", "0", "1", str(SLOTS), "0"]


@pytest.mark.parametrize("slots", [0, 1, 9])
def test_an_owner_without_slots_goes_on(driver, slots):
    n, m = 193 * MB, 40 * MB
    first, second, third = driver("f%d" % slots, "d%d" % n, "d%d" % n, "h%d" % m)
    assert first[0] == "1" and first[2] == "1"  # the plain copy brought it all
    assert first[3] == "0"  # the slots it had are given back
    assert second == ["1", "0", "1", "0", "0"]  # and it does not try again
    assert third == ["1", "0", "1", "0", "0"]
