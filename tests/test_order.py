"""The host side of bh_batch_order_by_cost (csrc/bh_order.h): the same costs and order as a sort of
(cost, entry) pairs with a search for every wave's entry, and not slower than that sort was on half
as many entries, which it had when an entry held 128 sinks."""
import os
import subprocess
import tempfile

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_order_by_cost_host():
    with tempfile.TemporaryDirectory() as d:
        exe = os.path.join(d, "order_check")
        subprocess.run(["g++", "-std=c++17", "-O2", os.path.join(ROOT, "tests", "order_check.cpp"),
                        "-o", exe], check=True)
        r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0 and r.stdout.startswith("OK"), r.stdout + r.stderr
    former, now = map(float, r.stdout.split()[1:])
    assert now <= former, r.stdout
