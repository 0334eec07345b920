"""The units of the prefill's two segment launches (csrc/gdn_prefill_segments.h)
on the host: which state blocks each one reads and writes, in place too."""

from __future__ import annotations

import ctypes
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "flashinfer_competition_codebase_amd" / "csrc"
NONE, IDENTITY, STATE, NEW_STATE, START, ZERO_END, TRANSITION = range(7)


@pytest.fixture(scope="module")
def seg_unit(tmp_path_factory):
    """(out, nseg, u, in_place) -> (segment, from, to, to's segment, keep_start)."""
    d = tmp_path_factory.mktemp("segments")
    (d / "unit.cpp").write_text(
        '#include "gdn_prefill_segments.h"\n'
        'extern "C" void unit(int out, int nseg, int u, int in_place, int* r) {\n'
        '  const gdn_pf::SegUnit s = gdn_pf::seg_unit(out != 0, nseg, u, in_place != 0);\n'
        '  r[0] = s.seg; r[1] = static_cast<int>(s.from); r[2] = static_cast<int>(s.to);\n'
        '  r[3] = s.to_seg; r[4] = s.keep_start;\n}\n')
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-Wall", "-Werror",
                    f"-I{CSRC}", str(d / "unit.cpp"), "-o", str(d / "unit.so")], check=True)
    lib = ctypes.CDLL(str(d / "unit.so"))

    def call(out, nseg, u, in_place):
        r = (ctypes.c_int * 5)()
        lib.unit(int(out), nseg, u, int(in_place), r)
        return tuple(r)
    return call


def _accesses(unit, in_place):
    """(blocks read, blocks written) of a unit; in place, the caller's state and
    new state are one block."""
    seg, frm, to, to_seg, keep = unit

    def block(kind, s):
        if kind in (STATE, NEW_STATE):
            return ("caller", STATE if in_place else kind)
        return (kind, s)
    reads = set() if frm in (NONE, IDENTITY) else {block(frm, seg)}
    writes = set() if to == NONE else {block(to, to_seg)}
    if keep:
        writes.add(block(START, seg))
    return reads, writes


@pytest.mark.parametrize("in_place", [False, True])
@pytest.mark.parametrize("nseg", [1, 2, 3, 4, 7, 32, 33])
def test_no_unit_reads_what_another_of_its_launch_writes(nseg, in_place, seg_unit):
    """The workgroups of a launch run in any order, so a block that one unit
    writes is neither read nor written by another of the same launch -- the
    last segment's end and the first one's start are one block in place."""
    written = {("caller", STATE)}                   # before the first launch
    for out, units in ((False, 2 * nseg - 3 if nseg >= 2 else 0), (True, nseg)):
        acc = [_accesses(seg_unit(out, nseg, u, in_place), in_place) for u in range(units)]
        for u, (_, writes) in enumerate(acc):
            for w, (reads, other) in enumerate(acc):
                if w != u:
                    assert not writes & (reads | other), (out, u, w)
        for u, (reads, _) in enumerate(acc):        # nothing unwritten is read
            assert reads <= written, (out, u, reads - written)
        for _, writes in acc:
            written |= writes
        if not out:                                 # the combine between the launches:
            if nseg >= 3:                           # starts 2 .. from start 1 and each
                assert (START, 1) in written        # middle segment's transition and end
                for j in range(1, nseg - 1):
                    assert {(TRANSITION, j), (ZERO_END, j)} <= written
            written |= {(START, j) for j in range(2, nseg)}
    assert ("caller", STATE if in_place else NEW_STATE) in written


@pytest.mark.parametrize("nseg", [1, 2, 3, 8, 33])
def test_every_segment_is_scanned_with_its_outputs_once(nseg, seg_unit):
    assert [seg_unit(True, nseg, u, False)[0] for u in range(nseg)] == list(range(nseg))
    if nseg >= 2:
        first = [seg_unit(False, nseg, u, False) for u in range(2 * nseg - 3)]
        assert first[0][:4] == (0, STATE, START, 1)
        middle = list(range(1, nseg - 1))
        assert [u[:4] for u in first[1:]] == (
            [(j, NONE, ZERO_END, j) for j in middle] +
            [(j, IDENTITY, TRANSITION, j) for j in middle])
