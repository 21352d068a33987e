"""CPU emulation of the index arithmetic of the column pass on row-pair fields
(sparc_flows_amd/csrc/sparc_colseg.hip: k_colsplit and k_colone), for every launch
shape that colsplit_fits admits: segment lengths of SPARC_COLSEG_SIZES with at most 64
segments and a last one of at least 3 real rows, block widths TC of 1, 2, 4, 8 and 16,
at most 3 x 128 lanes (k_colsplit) or 512 (k_colone, lengths up to 8), interface
half-widths 0, 3 and P and kinds of interface rows 1, 5 and P in turn.  Every global
access must stay inside its array and on 16 bytes where it moves a pair, every LDS
access inside the block's dynamic LDS, and the stores of a field must hit each of its
real rows once.

The expressions are the kernels' own, for every thread of a block and every unrolled
row; blocks are taken at the grid's extremes (first and last column group and source)."""
import re
from pathlib import Path

import numpy as np
import pytest

CSRC = Path(__file__).resolve().parent.parent / "sparc_flows_amd" / "csrc"
SIZES = [int(v) for v in re.findall(r"X\((\d+)\)", re.search(
    r"#define SPARC_COLSEG_SIZES\(X\)(.*)", (CSRC / "sparc_launch.h").read_text()).group(1))]
ONE_SIZES = [int(v) for v in re.findall(r"X\((\d+)\)", re.search(
    r"#define SPARC_COLONE_SIZES\(X\)(.*)", (CSRC / "sparc_colseg.hip").read_text()).group(1))]
KZS, KZF, KCB, KPL = 15, 6, 12, 7


def cases():
    """(nz, MS): nz 16..40 in full, then both ends of (MS, P) up to 1024 with P up to 9
    and around the segment counts where a block's lanes or waves change."""
    out = set()
    for ms in SIZES:
        for p in (*range(1, 10), 15, 16, 17, 31, 32, 33, 47, 63, 64):
            for nz in ((p - 1) * ms + 3, (p - 1) * ms + 4, p * ms - 1, p * ms):
                if 16 <= nz <= 1024 and -(-nz // ms) == p and nz - (p - 1) * ms >= 3:
                    out.add((nz, ms))
        for nz in range(16, 41):
            if nz - (-(-nz // ms) - 1) * ms >= 3:
                out.add((nz, ms))
    return sorted(out)


class Check:
    def __init__(self, what):
        self.what = what

    def idx(self, name, v, size, mask=None, low=0):
        v = np.asarray(v)
        if mask is not None:
            v = v[np.broadcast_to(mask, v.shape)]
        if v.size:
            assert v.min() >= low and v.max() < size, f"{self.what}: {name} in [{v.min()}, {v.max()}], [{low}, {size})"

    def pair(self, name, v, size, mask=None):
        """A 16-byte access at element v."""
        v = np.asarray(v)
        assert not (v & 1).any(), f"{self.what}: {name} not on 16 bytes"
        self.idx(name, v, size - 1, mask)


def kind(s, P, E):
    return np.where(s < E, s, np.where(s >= P - E, 2 * E + 1 - (P - s), E))


def emulate(one, nz, ms, tc, nx, S, nb, nt, hw, E):
    P = -(-nz // ms)
    nzp, nzq, npml = P * ms, (nz + 1) // 2 * 2, nb + nt
    nk = 2 * E + 1 if 2 * E + 1 < P else P
    if nk == P:
        E = P
    nrow, LY, hw2 = 2 * (4 * hw + 4), 2 * P + 4 * hw + 2, 2 * hw
    nband, n, lastp = nk * nrow, nzq * nx, nzq // 2 - 1
    zl = 3 * nband
    zf = zl + KZS * 3 * ms
    cbl = zf + KZF * nzp
    img = cbl + KCB
    if one:
        block = -(-tc * P // 64) * 64
        staged = (img + 1) // 2 * 2
        yb = staged
        rowbuf = yb + 4 * tc * LY                       # p
        lds = staged + 4 * tc * LY + tc * nzp
    else:
        G = -(-tc * P // 64) * 64
        block = 3 * G
        pml = img
        zpl = pml + KPL * npml * tc
        staged = (zpl + nzp + 1) // 2 * 2
        yb = staged
        rowbuf = yb + 4 * tc * LY                       # wl: group 1, group 0, p
        lds = staged + 4 * tc * LY + 3 * tc * nzp
    if 8 * lds > 160 * 1024:
        return 0                                        # colsplit_fits refuses it
    chk = Check(f"{'one' if one else 'split'} nz={nz} MS={ms} TC={tc} nx={nx} S={S} hw={hw} E={E}")
    assert nband % 2 == 0 and nrow % 2 == 0 and yb % 2 == 0 and LY % 2 == 0
    tid = np.arange(block)[:, None]
    if one:
        c, s0 = tid % tc, tid // tc
        act = s0 < P
        s = np.minimum(s0, P - 1)
        corr = np.ones_like(act)                        # every lane runs the correction
    else:
        f = tid // G
        l_ = tid - f * G
        c, s0 = l_ % tc, l_ // tc
        act = s0 < P
        s = np.where(act, s0, 0)
        corr = act
    a = s * ms
    h0 = a >> 1
    last = a + ms > nz - 2
    i = np.arange(ms)[None, :]
    i2 = np.arange(0, ms, 2)[None, :]
    j = a + i
    real = act & (j < nz)
    off = lambda h: np.clip(h, 0, lastp) * 2 * nx
    gx = nx // tc
    for bx in {0, gx - 1}:
        for b in {0, S - 1}:
            x = bx * tc + c
            col = b * n + 2 * x
            chk.idx("column", x, nx)
            # loads: the derivative's window, its end rows, the epilogue's rows, the filter's
            chk.pair("window", col + off(h0 - 2 + np.arange(0, ms + 8, 2)[None, :] // 2), S * n)
            r = nz - 5 + np.arange(5)[None, :]
            chk.idx("end rows", col + (r >> 1) * 2 * nx + (r & 1), S * n, last)
            chk.pair("epilogue rows", col + off(h0 + i2 // 2), S * n)
            chk.pair("coefficient rows", 2 * x + off(h0 + i2 // 2), n)
            chk.pair("filter window", col + off(h0 - 3 + np.arange(0, ms + 12, 2)[None, :] // 2), S * n)
            # the window's element k is row a - 4 + k wherever that row exists
            k = np.arange(ms + 8)[None, :]
            row = 2 * np.clip(h0 - 2 + (k >> 1), 0, lastp) + (k & 1)
            want = a - 4 + k
            assert np.all(row[np.broadcast_to((want >= 0) & (want < nzq), row.shape)] ==
                          want[(want >= 0) & (want < nzq)])
            # stores
            on = act & (a + i2 < nz)
            at = col + (h0 + i2 // 2) * 2 * nx
            chk.pair("stores", at, S * n, on)
            for g in range(1 if one else 3):
                m = on if one else on & (f == g)
                hit = at[np.broadcast_to(m, at.shape)]
                assert hit.size == tc * nzq // 2 and np.unique(hit).size == hit.size
            chk.idx("topbc", b * nx + x, S * nx)
            # z-PML rows
            if one:
                pj = np.where(j < nb, j, np.where((j >= nz - nt) & (j < nz), nb + j - (nz - nt), -1))
                pin = pj >= 0
                even, odd = pj[:, 0::2], pj[:, 1::2]
                for p in (np.where(even >= 0, even, odd), np.where(odd >= 0, odd, even)):
                    use = (even >= 0) | (odd >= 0)
                    chk.idx("PML load", p * nx + x, npml * nx, use)
                    chk.idx("PML field load", ((S + b) * npml + p) * nx + x, 2 * S * npml * nx, use)
                chk.idx("PML store", ((S + b) * npml + pj) * nx + x, 2 * S * npml * nx, pin & act)
                chk.idx("source profile", j, nz, j < nz)
            else:
                jc = np.minimum(j, nz - 1)
                pj = np.where(jc < nb, jc, np.minimum(npml - 1, nb + np.maximum(jc - (nz - nt), 0)))
                for kk in range(KPL):
                    chk.idx("staged PML", pml + (kk * npml + pj) * tc + c, zpl)
                for q in (b, S + b):
                    chk.idx("PML store", (q * npml + pj) * nx + x, 2 * S * npml * nx, act)
                chk.idx("staged source profile", zpl + j, staged)
            # outputs at their extreme slots
            for nsnap, nf in ((3, 6), (5, 4)):
                slot = (b * nsnap + nsnap - 1) * nf + nf - 1
                chk.idx("snapshot", (slot * nz + j) * nx + x, S * nsnap * nf * nz * nx, real)
            # LDS: tables, end values, row buffers
            zt = np.where(s == 0, 0, np.where(s == P - 1, 2, 1)) * ms
            chk.idx("segment tables", zl + zt + (KZS - 1) * 3 * ms + i, zf, low=zl)
            chk.idx("profiles", zf + (KZF - 1) * nzp + a + i, cbl)
            kd = kind(s, P, E)
            chk.idx("interface kind", kd, nk)
            chk.idx("interface rows", 2 * nband + kd * nrow + np.arange(nrow)[None, :], 3 * nband)
            for g in range(4):
                yc = yb + (g * tc + c) * LY
                chk.idx("end values", yc + hw2 + 2 * s + np.array([[0, 1]]), yc.max() + LY, act)
                win = yc + 2 * (s - 1) + np.arange(4 * hw + 8)[None, :]
                chk.idx("end-value windows", win, lds, corr)
                assert not ((yc + 2 * (s - 1)) & 1).any()
                # outside the lane's own column only where the sum is dropped
                own = (win >= yc) & (win < yc + LY)
                first, lastw = win - yc - 2 * (s - 1) < 4 * hw + 4, win - yc - 2 * (s - 1) >= 4
                assert np.all(own | (np.broadcast_to((s == 0), win.shape) & ~lastw)
                              | (np.broadcast_to(s == P - 1, win.shape) & ~first) | ~np.broadcast_to(corr, win.shape))
            nbuf = 1 if one else 3
            for g in range(nbuf):
                chk.idx("row buffers", rowbuf + (g * tc + c) * nzp + j, lds, act)
            pc = rowbuf + ((nbuf - 1) * tc + c) * nzp
            chk.idx("p window", pc + np.clip(a - 3 + np.arange(ms + 6)[None, :], 0, nz - 1), lds)
            chk.idx("p end rows", pc + nz - 5 + np.arange(5)[None, :], lds, last)
    # staging: the image in pairs (k_colone), or element by element with the z-PML data
    if one:
        chk.idx("image", np.arange(staged // 2) * 2 + 1, staged)
    else:
        npl, x0, b = npml * tc, (gx - 1) * tc, S - 1
        q = np.arange(npl)
        chk.idx("staging PML", (q // tc) * nx + x0 + q % tc, npml * nx)
        chk.idx("staging PML fields", ((S + b) * npml + q // tc) * nx + x0 + q % tc, 2 * S * npml * nx)
        # the pads of the end-value buffers, and nothing else of them
        padw = LY - 2 * P
        q = np.arange(4 * tc * padw)
        r, u = q // padw, q % padw
        pad = r * LY + np.where(u < hw2, u, 2 * P + u)
        vals = (np.arange(4 * tc)[:, None] * LY + hw2 + np.arange(2 * P)[None, :]).ravel()
        assert np.array_equal(np.sort(np.concatenate([pad, vals])), np.arange(4 * tc * LY))
    return 1


@pytest.mark.parametrize("one", [False, True])
def test_every_shape_stays_in_bounds(one):
    n = 0
    for count, (nz, ms) in enumerate(cases()):
        if one and ms not in ONE_SIZES:
            continue
        P = -(-nz // ms)
        for tc in (1, 2, 4, 8, 16):
            if tc * P > 512 if one else -(-tc * P // 64) > 2:
                continue
            for nx, S in ((16, 1), (1008, 2)):
                if nx % tc:
                    continue
                npml = min(12, (nz - 1) // 2 - 1)
                hw = (0, 3, min(P, 12))[(count + tc) % 3]
                E = (0, 2, P)[(count + S) % 3]
                n += emulate(one, nz, ms, tc, nx, S, npml, npml, hw, E)
    assert n > (300 if one else 1000), n


def test_offsets_fit_32_bits():
    """The largest batch that sparc_create admits (nsrc nz nx < 2^27): the padded rows of
    an odd nz keep every byte offset below 2^31."""
    for nz, nx in ((17, 16), (17, 1024), (1023, 16), (1023, 1023)):
        S = (2 ** 27 - 1) // (nz * nx)
        assert 8 * S * ((nz + 1) // 2 * 2) * nx < 2 ** 31
