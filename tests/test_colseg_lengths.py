"""Every nz from 16 to 1024 has a cut into segments that the column pass takes
(csrc/sparc_launch.h, SPARC_COLSEG_SIZES): whole row pairs, at most 64 segments, at
least three real rows in the last."""
import re
from pathlib import Path

HEADER = Path(__file__).resolve().parent.parent / "sparc_flows_amd" / "csrc" / "sparc_launch.h"


def test_every_nz_has_a_cut():
    line = re.search(r"#define SPARC_COLSEG_SIZES\(X\)(.*)", HEADER.read_text()).group(1)
    sizes = [int(v) for v in re.findall(r"X\((\d+)\)", line)]
    assert sizes and all(v % 2 == 0 for v in sizes)
    for nz in range(16, 1025):
        assert any(-(-nz // m) <= 64 and nz - (-(-nz // m) - 1) * m >= 3 for m in sizes), nz
