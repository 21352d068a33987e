"""The segmented z-derivatives that run, on the CPU from the kernels' own source:
tests/seg_rows_emul.cpp drives the column pass's interface rows by kind
(build_seg_rows, seg_correct_rows) for every segment length of SPARC_COLSEG_SIZES,
and the z kernels' banded inverse (build_zseg, seg_correct) at the length that
zseg_length gives, against the oracle's dbyd2 (bit-identical to the reference's
dbyd2.f + mtridag.f).

The segmented solve differs from the Thomas sweep by rounding only: 1e-12 relative
(max norm) on smooth columns and 1e-10 on white noise, whose boundary closure
amplifies rounding."""
import ctypes
import re
import shutil
import subprocess
from pathlib import Path

import numpy as np
import pytest

import oracle

ROOT = Path(__file__).resolve().parents[1]
CSRC = ROOT / "sparc_flows_amd" / "csrc"
DP = ctypes.POINTER(ctypes.c_double)


def colseg_sizes():
    line = re.search(r"#define SPARC_COLSEG_SIZES\(X\)(.*)", (CSRC / "sparc_launch.h").read_text()).group(1)
    return [int(v) for v in re.findall(r"X\((\d+)\)", line)]


SIZES = colseg_sizes()


def usable(nz, ms):
    p = -(-nz // ms)
    return p <= 64 and nz - (p - 1) * ms >= 3


@pytest.fixture(scope="module")
def emul(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    out = tmp_path_factory.mktemp("seg") / "libsegrows.so"
    sizes = " ".join(f"X({v})" for v in SIZES)
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wno-unknown-pragmas", f"-I{CSRC}",
                    f"-DCOLSEG_SIZES(X)={sizes}", str(ROOT / "tests" / "seg_rows_emul.cpp"),
                    str(CSRC / "sparc_segtab.cpp"), "-o", str(out)], check=True, capture_output=True)
    L = ctypes.CDLL(str(out))
    i, d = ctypes.c_int, ctypes.c_double
    L.colseg_column.argtypes = [i, i, i, i, DP, d, d, DP]
    L.zseg_column.argtypes = [i, i, DP, d, d, DP]
    L.zseg_length_of.argtypes = [i]
    L.colseg_shape.argtypes = [i, i, ctypes.POINTER(i)]
    return L


def columns(nz):
    z = np.linspace(0.0, 1.0, nz)
    return (("smooth", np.sin(2.3 * np.pi * z + 0.4) + 0.3 * z ** 3, 1e-12),
            ("noise", np.random.default_rng(nz).standard_normal(nz), 1e-10))


def presets(ibc):
    return (0.7 if ibc == 2 else 0.0), (-1.3 if ibc == 3 else 0.0)


def check(nz, ibc, B, tol, run, what):
    pre0, preN = presets(ibc)
    A = np.zeros((nz, 1))
    A[0, 0], A[-1, 0] = pre0, preN
    ref = oracle.dbyd2(B[:, None], ibc, A)[:, 0]
    got = np.full(nz, np.nan)
    assert run(np.ascontiguousarray(B), pre0, preN, got) == 0, what
    err = np.abs(got - ref).max() / np.abs(ref).max()
    assert err < tol, (what, err)          # a NaN is not below tol either


@pytest.mark.parametrize("nz", [16, 17, 23, 40, 60, 97, 121, 150, 255, 300, 301, 384, 512, 721, 722, 1023, 1024])
def test_column_pass_rows_match_oracle(emul, nz):
    for ms in [m for m in SIZES if usable(nz, m)]:
        for unroll in (1, 2):
            for ibc in (1, 2, 3):
                for name, B, tol in columns(nz):
                    check(nz, ibc, B, tol,
                          lambda b, p0, pN, o: emul.colseg_column(nz, ms, unroll, ibc, b.ctypes.data_as(DP), p0, pN,
                                                                  o.ctypes.data_as(DP)), (nz, ms, unroll, ibc, name))


@pytest.mark.parametrize("nz", [60, 303])
def test_each_row_of_the_column_enters(emul, nz):
    """A column with one nonzero value at every row in turn: a wrong one-sided row, or
    a repeated interior pair that is not its segment's own, cannot hide."""
    for ms in (6, 10):
        for ibc in (1, 2, 3):
            for r in range(nz):
                B = np.zeros(nz)
                B[r] = 1.0
                ref = oracle.dbyd2(B[:, None], ibc, np.zeros((nz, 1)))[:, 0]
                got = np.full(nz, np.nan)
                assert emul.colseg_column(nz, ms, 2, ibc, B.ctypes.data_as(DP), 0.0, 0.0, got.ctypes.data_as(DP)) == 0
                assert np.abs(got - ref).max() < 1e-12 * max(np.abs(ref).max(), 1.0), (ms, ibc, r)


@pytest.mark.parametrize("nz", [16, 17, 35, 63, 121, 160, 161, 300, 301, 323, 512, 700, 1024])
def test_z_kernel_tables_match_oracle(emul, nz):
    for ibc in range(4):
        for name, B, tol in columns(nz):
            check(nz, ibc, B, tol, lambda b, p0, pN, o: emul.zseg_column(nz, ibc, b.ctypes.data_as(DP), p0, pN,
                                                                         o.ctypes.data_as(DP)), (nz, ibc, name))


def test_depths_without_a_cut_of_the_z_kernels(emul):
    """The depths that run the one-lane forms, as sparc_seg.h and sparc_zseg.h name them."""
    length = {nz: emul.zseg_length_of(nz) for nz in range(16, 1026)}
    none = [nz for nz, m in length.items() if m == 0]
    assert none == [673, 674, 897, 898, 929, 930, 961, 962, 993, 994, 1025]
    long3d = [nz for nz, m in length.items() if nz <= 512 and (m == 0 or m > 16)]
    assert long3d == [337, 338, 449, 450, 465, 466, 481, 482, 497, 498]
    assert all(m == 0 or m > 16 for nz, m in length.items() if nz > 512)
    # the lengths whose 3D velocity pass keeps registers in scratch
    assert [nz for nz, m in length.items() if nz <= 320 and m in (12, 14, 16)] == [
        121, 122, 131, 132, 141, 142, 151, 152, 241, 242, 261, 262, 271, 272, 281, 282, 291, 292, 301, 302, 311, 312]


def test_column_pass_lds_up_to_nz_1024(emul):
    """Some segment length fits each form of the column pass (TC = 1, 40 PML rows) in
    gfx950's 160 KB at every nz, by colsplit_lds_bytes and colone_lds_bytes."""
    kzs, kzf, kcb, kpl, nzpml = 15, 6, 12, 7, 40
    shape = (ctypes.c_int * 4)()
    for nz in list(range(16, 1025, 13)) + [721, 722, 1023, 1024]:
        split, one = [], []
        for ms in [m for m in SIZES if usable(nz, m)]:
            assert emul.colseg_shape(nz, ms, shape) == 0
            P, hw, E, nk = list(shape)
            assert nk == (2 * E + 1 if 2 * E + 1 < P else P)
            nzp, ly = P * ms, 2 * P + 4 * hw + 2
            img = 3 * nk * 2 * (4 * hw + 4) + kzs * 3 * ms + kzf * nzp + kcb
            split.append(8 * ((img + kpl * nzpml + nzp + 1) // 2 * 2 + 4 * ly + 3 * nzp))
            if ms <= 8:
                one.append(8 * ((img + 1) // 2 * 2 + 4 * ly + nzp))
        assert min(split) <= 160 * 1024, (nz, min(split))
        assert all(v <= 160 * 1024 for v in one), (nz, one)
