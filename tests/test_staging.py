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


def test_a_small_context_pins_once(lines):
    assert [v for k, v in lines if k == "pins"] == [[77, 1], [1000, 1], [4093, 2], [20011, 2]]
