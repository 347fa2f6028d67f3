"""The public kernel timers against the host code that records them: a timer
that nothing begins is marked so in the header, and the bench has byte counts
for recorded ones alone."""
import os
import re

import bench

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HOST = os.path.join(ROOT, "parties-vof-ibm_amd", "host")


def timers():
    """name -> comment of the header's enum, in its order"""
    src = open(os.path.join(ROOT, "include", "parties_vof.h")).read()
    return dict(re.findall(r"PV_T_(\w+)(?: = 0)?,\s*/\*(.*?)\*/", src, flags=re.S))


def recorded():
    src = "".join(open(os.path.join(HOST, f)).read() for f in sorted(os.listdir(HOST)) if f.endswith(".c"))
    return set(re.findall(r"\bPV_T_(\w+)", src))


def test_unrecorded_timers_are_marked():
    t, used = timers(), recorded()
    assert list(t) == bench.TIMERS and used <= set(t)
    for name, comment in t.items():
        assert ("not recorded" in comment) == (name not in used), name


def test_bench_has_byte_counts_for_recorded_timers():
    for table in (bench.BYTES_PER_CELL, bench.BYTES_PER_CELL_FFT, bench.BYTES_PER_CELL_MG, bench.BYTES_PER_CELL_MG32):
        assert set(table) <= recorded(), set(table) - recorded()
