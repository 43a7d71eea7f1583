"""Index arithmetic of the sparse products at the limits of int32 sizes: the
offset type chosen for a vector's gathers reaches its last element (a
multi-right-hand-side CG of more than 2^29 rows gathers past 4 GiB), and
loops over a block's entries end and stay in bounds for entry counts up to
INT_MAX - 1.  Host build of hala_amd/csrc/gather.hpp under
UndefinedBehaviorSanitizer; the products take both from there."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "hala_amd", "csrc")


def test_gather_limits(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("no g++")
    exe = tmp_path / "gather_limits"
    flags = ["-fsanitize=undefined", "-fno-sanitize-recover=all"]
    src = os.path.join(ROOT, "tests", "cpp", "gather_limits.cpp")
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", *flags, src, "-o", str(exe)], capture_output=True, text=True)
    if r.returncode != 0 and "cannot find" in r.stderr:
        r = subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", src, "-o", str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    bad = [l for l in r.stdout.splitlines() if not l.startswith("ok")]
    assert r.returncode == 0 and not bad, (bad, r.stderr)


def test_tile_tickets(tmp_path):
    # the grid sweeps' tiles, in an order in which a tile only waits for earlier tickets
    if shutil.which("g++") is None:
        pytest.skip("no g++")
    exe = tmp_path / "tile_order"
    src = os.path.join(ROOT, "tests", "cpp", "tile_order.cpp")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", src, "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout


def test_offset_products_choose_the_width():
    # whoever instantiates the offset gathers with 32 bits also asks gather_wide
    users = [f for f in os.listdir(CSRC) if f.endswith(".hip") and "csr_block_rowsums<" in open(os.path.join(CSRC, f)).read()]
    assert sorted(users) == ["cgbatch.hip", "spmm.hip"]
    for f in users:
        text = open(os.path.join(CSRC, f)).read()
        assert "gather_wide(" in text, f
        for call in re.findall(r"csr_block_rowsums<([^;]*?)>\(", text):
            assert call.split(",")[4].strip() == "TO", (f, call)


def test_tile_loops_step_in_bounds():
    # a loop over int entry positions steps by tile_next: base += TILE overflows within a tile of INT_MAX
    for f in ("spmv.hpp", "spmv.hip", "spmm.hpp", "spmm.hip"):
        for loop in re.findall(r"for \(int base = [^;]*;[^;]*;([^)]*\)?)\)", open(os.path.join(CSRC, f)).read()):
            assert "tile_next(base" in loop, (f, loop)
