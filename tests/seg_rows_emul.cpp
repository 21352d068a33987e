// CPU run of a z-derivative as the lanes of one column do it, through the
// kernels' own templates (sparc_seg.h) and tables (sparc_segtab.cpp):
//   * the column pass (k_colsplit, k_colone): interface rows by kind, seg_correct_rows;
//   * the z kernels (k_zder, the 3D z passes): the banded inverse, seg_correct.
// The column's end-value buffer lies between two others; all LDS but its own part is
// NaN, so that a read outside that reaches a result shows.  Built by
// tests/test_seg_rows.py with g++.
#include <cmath>
#include <cstring>
#include <vector>

#include "sparc_seg.h"

using namespace sparc;

namespace {

struct Buf {
    std::vector<double> v;
    double *yp;                 // the middle column's buffer, on 16 bytes
    Buf(int ly) : v((size_t)3 * ly + 1, std::nan(""))
    {
        double *p = v.data();
        if ((size_t)p & 8) p++;
        yp = p + ly;
        std::fill(yp, yp + ly, 0.0);
    }
};

// correct(Y, s, yp, tab): the interface correction of segment s.
template <int MS, typename Tables, typename Correct>
void column(int nz, int P, int hw, int ibc, const double *B, double preset0, double presetN, double *out,
            Tables tables, Correct correct)
{
    double c1, c2, cb[kCB];
    dbyd2_coefs(nz, c1, c2, cb);
    Buf b(yb_len(P, hw));
    std::vector<double> Ys((size_t)P * MS);
    for (int s = 0; s < P; s++) {
        const int a = s * MS;
        const bool last = a + MS > nz - 2;
        auto ld = [&](int k) {
            const int r = a - 3 + k;
            return B[r < 0 ? 0 : (r > nz - 1 ? nz - 1 : r)];
        };
        double e[5] = {0.0, 0.0, 0.0, 0.0, 0.0}, Y[MS];
        if (last)
            for (int k = 0; k < 5; k++) e[k] = B[nz - 5 + k];
        seg_rhs<MS>(ld, e, Y, a, nz, s == 0, last, ibc, preset0, presetN, c1, c2, cb);
        seg_solve<MS>(Y, tables(s));
        b.yp[2 * hw + 2 * s] = Y[0];
        b.yp[2 * hw + 2 * s + 1] = Y[MS - 1];
        std::memcpy(&Ys[(size_t)s * MS], Y, sizeof Y);
    }
    for (int s = 0; s < P; s++) {
        double Y[MS];
        std::memcpy(Y, &Ys[(size_t)s * MS], sizeof Y);
        correct(Y, s, b.yp, tables(s));
        for (int i = 0; i < MS && s * MS + i < nz; i++) out[s * MS + i] = Y[i];
    }
}

template <int MS, int U>
int rows(int nz, int ibc, const double *B, double preset0, double presetN, double *out)
{
    SegRows t;
    std::vector<double> kt;
    if (ibc < 1 || ibc > 3 || !build_seg_rows(nz, MS, t) || !seg_kind_tables(t, kt)) return -2;
    const int P = t.P, nw = 4 * t.hw + 4, nk = seg_band_kinds(P, t.E), slot = ibc - 1;
    if (t.rows.size() != (size_t)3 * nk * 2 * nw) return -3;
    std::vector<double> al(t.rows.size() + 1);
    double *r = al.data() + (((size_t)al.data() & 8) ? 1 : 0);
    std::copy(t.rows.begin(), t.rows.end(), r);
    auto tables = [&](int s) {
        return [&kt, s, slot, P](int k, int i) { return kt[((size_t)(slot * 5 + k) * 3 + seg_kind(s, P)) * MS + i]; };
    };
    column<MS>(nz, P, t.hw, ibc, B, preset0, presetN, out, tables, [&](double (&Y)[MS], int s, const double *yp, auto tab) {
        const int k = seg_band_kind(s, P, t.E);
        seg_correct_rows<MS, U>(Y, s, P, t.hw, yp, r + ((size_t)slot * nk + k) * 2 * nw, tab);
    });
    return 0;
}

template <int MS>
int band(int nz, int ibc, const double *B, double preset0, double presetN, double *out)
{
    const int sets[4] = {0, 1, 2, 3}, P = (nz + MS - 1) / MS;
    int hw = 0;
    std::vector<double> img;
    if (!build_zseg(nz, MS, 4, sets, hw, img)) return -2;
    const int nset = zseg_set_len(P, hw, MS);
    if (img.size() != (size_t)4 * nset) return -3;
    std::vector<double> al(img.size() + 1);
    double *const base = al.data() + (((size_t)al.data() & 8) ? 1 : 0);
    std::copy(img.begin(), img.end(), base);
    const double *const bd = base + (size_t)ibc * nset, *const zt = bd + 2 * P * (4 * hw + 4);
    auto tables = [&](int s) {
        return [zt, s, P](int k, int i) { return zt[(k * 3 + seg_kind(s, P)) * MS + i]; };
    };
    column<MS>(nz, P, hw, ibc, B, preset0, presetN, out, tables,
               [&](double (&Y)[MS], int s, const double *yp, auto tab) { seg_correct<MS>(Y, s, P, hw, yp, bd, tab); });
    return 0;
}

}  // namespace

// dbyd2 of one column by the column pass's tables (unroll 1: k_colone, 2: k_colsplit).
extern "C" int colseg_column(int nz, int ms, int unroll, int ibc, const double *B, double preset0, double presetN,
                             double *out)
{
#define X(M)                                                                       \
    if (ms == M) return unroll == 1 ? rows<M, 1>(nz, ibc, B, preset0, presetN, out) \
                                    : rows<M, 2>(nz, ibc, B, preset0, presetN, out);
    COLSEG_SIZES(X)
#undef X
    return -1;
}

// The same by the z kernels' tables of this nz; -1 where it has no cut.
extern "C" int zseg_column(int nz, int ibc, const double *B, double preset0, double presetN, double *out)
{
    const int ms = zseg_length(nz);
#define X(M) if (ms == M) return band<M>(nz, ibc, B, preset0, presetN, out);
    SPARC_ZDER_SIZES(X)
#undef X
    return -1;
}

extern "C" int zseg_length_of(int nz) { return zseg_length(nz); }

// Shape of the column pass's tables: P, hw, E, kinds.
extern "C" int colseg_shape(int nz, int ms, int shape[4])
{
    SegRows t;
    if (!build_seg_rows(nz, ms, t)) return -2;
    shape[0] = t.P;
    shape[1] = t.hw;
    shape[2] = t.E;
    shape[3] = seg_band_kinds(t.P, t.E);
    return 0;
}
