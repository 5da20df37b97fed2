"""The work lists' load estimate (yaxus_amd/csrc/deal.hpp) against a sort and a heap, natively
(tests/native/deal_check.cpp): the same results, in a fraction of the host time, which every
yx_pass_begin of many sequences pays several times. CPU only."""

import json
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_deal_matches_a_heap(tmp_path):
    exe = str(tmp_path / "deal_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Wextra", os.path.join(HERE, "native", "deal_check.cpp"),
                    "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    d = json.loads(r.stdout.strip().splitlines()[-1])
    print(d)
    assert d["deal_us"] < 0.6 * d["heap_us"]
