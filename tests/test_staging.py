"""The staging buffer's layout and the sharing of its packing
(cable_amd/csrc/staging.h), on the CPU."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not found")


@pytest.fixture(scope="module")
def lines(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("staging") / "s")
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", os.path.join(HERE, "host_staging.cpp"), "-o", exe],
                   check=True, capture_output=True)
    out = subprocess.run([exe], check=True, capture_output=True, text=True, timeout=60).stdout
    return [(x.split()[0], [int(v) for v in x.split()[1:]]) for x in out.splitlines()]


def test_every_array_starts_at_the_alignment(lines):
    assert dict(lines)["offsets"] == [0, 0, 0, 0]


def test_every_byte_is_handed_out_once_in_pieces_within_a_unit(lines):
    got = [v for k, v in lines if k == "pieces"]
    assert len(got) == 14 and all(n == once and beyond == 0 for n, once, beyond, _ in got)


def test_a_large_buffer_is_not_shared_within_a_huge_page(lines):
    """From 16 MiB on, but for the last 4 to 6 MiB: else the threads that touch a
    page of a new array first wait for each other."""
    assert all(most == 1 for k, v in lines if k == "pieces" for most in v[3:])


def test_chunks_through_two_halves(lines):
    """Each closed once and in its half's turn, and all bytes arrive."""
    got = [v for k, v in lines if k == "chunks"]
    assert len(got) == 3 and all(n == 11 and closed == 11 and early == 0 and same for n, closed, early, same in got)


def test_no_data_race(tmp_path):
    """The same program under the thread sanitizer."""
    exe = str(tmp_path / "s")
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=thread", "-pthread",
                        os.path.join(HERE, "host_staging.cpp"), "-o", exe], capture_output=True, text=True)
    if r.returncode != 0:
        pytest.skip("sanitizer build unavailable: " + r.stderr[-300:])
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and "WARNING: ThreadSanitizer" not in r.stderr, r.stderr[-3000:]


def test_a_small_context_pins_once(lines):
    assert [v for k, v in lines if k == "pins"] == [[77, 1], [1000, 1], [4093, 2], [20011, 2]]
