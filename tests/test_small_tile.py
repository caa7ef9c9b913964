"""LDS bounds of the small-output GEMM's staged result tile, on the CPU."""
import os
import re
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = os.path.join(HERE, "native", "small_tile_check.cpp")
HIP = os.path.join(HERE, "..", "flashvsr-sm89-ops_amd", "csrc", "gemm_fp8.hip")


def _run(tmp_path, *flags):
    exe = str(tmp_path / "small_tile_check")
    subprocess.run(["g++", "-std=c++17", "-O1", *flags, "-o", exe, SRC], check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    return r.returncode, dict(line.split() for line in r.stdout.splitlines())


def test_staged_rows_lie_within_their_slots(tmp_path):
    rc, bad = _run(tmp_path)
    assert rc == 0 and set(bad.values()) == {"0"}, bad
    # the tiles walked are the ones the kernel is built for
    built = re.findall(r"gemm_fp8_small<EPI, (\d), (\d), (\d), \d>", open(HIP).read())
    walked = re.findall(r"check<SmallTile<(\d), (\d), (\d)>", open(SRC).read())
    assert sorted(built) == sorted(walked)


def test_a_tile_larger_than_its_slot_is_reported(tmp_path):
    """128 x 256 is 64 KB of bf16 in slots of 48 KB: its last 32 rows would lie
    past slot 0; the other tiles fit into it."""
    rc, bad = _run(tmp_path, "-DONE_SLOT")
    assert rc == 1 and bad == {"64x64": "0", "64x128": "0", "128x128": "0", "128x256": "32"}
