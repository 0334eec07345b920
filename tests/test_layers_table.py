"""The grouped-layers kernel has an instance for every row of the single-token
launch tables (csrc/gdn_decode.hip), whatever rows these hold."""

from __future__ import annotations

import re
import subprocess

import pytest

from flashinfer_competition_codebase_amd.build import CSRC, INCLUDE_DIR, hipcc_path

TABLES = {"kShapeFp32": "false", "kShapeBf16": "true"}


def _rows(text, table):
    body = re.search(rf"constexpr ShapeRow {table}\[\] = \{{(.*?)\}};", text, re.S).group(1)
    return [(int(ns), int(w)) for ns, w in re.findall(r"\{-?\d+, (\d+), (\d+)\}", body)]


@pytest.mark.parametrize("edit", [None, ("kShapeFp32", 8, 2), ("kShapeBf16", 8, 1)])
def test_every_table_row_has_a_layers_kernel(edit, tmp_path):
    """Host code only.  With a row changed to a shape the tables did not hold,
    its instances come with it: a launch of that shape finds a kernel."""
    text = CSRC.read_text()
    if edit is not None:
        table, ns, w = edit
        assert (ns, w) not in _rows(text, table)
        text = re.sub(rf"(constexpr ShapeRow {table}\[\] = \{{\s*\{{-?\d+), \d+, \d+\}}",
                      rf"\g<1>, {ns}, {w}}}", text, count=1)
        assert (ns, w) in _rows(text, table)
    src = tmp_path / "gdn_decode.hip"
    src.write_text(text)
    obj = tmp_path / "gdn_decode.o"
    subprocess.run([hipcc_path(), "--offload-arch=gfx950", "--offload-host-only", "-O0",
                    "-std=c++17", f"-I{CSRC.parent}", f"-I{INCLUDE_DIR}", "-c", str(src),
                    "-o", str(obj)], check=True)
    symbols = subprocess.run(["nm", "-C", str(obj)], check=True, capture_output=True,
                             text=True).stdout
    for table, bf16 in TABLES.items():
        for ns, w in _rows(text, table):
            for l2 in ("true", "false"):
                assert f"gdn_decode_layers_k128<{ns}, {w}, {l2}, {bf16}>" in symbols, (table, ns, w)
