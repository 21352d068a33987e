// sparc_segtab.cpp -- host construction of the dbyd2 coefficients, matrix and
// segmented-solve tables (dbyd2.f:85-195, mtridag.f:95-112) shared by the
// library and the CPU check of the column pass's algorithm.  Plain C++.
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "sparc_seg.h"

namespace sparc {

void dbyd2_coefs(int N2, double &c1, double &c2, double cb[kCB])
{
    const float d2i = (float)(N2 - 1);
    c1 = (double)(d2i * 7.0f / 9.0f);
    c2 = (double)(d2i / 36.0f);
    cb[CB_B + 0] = (double)(-(43.f / 96.f * d2i));
    cb[CB_B + 1] = (double)(-(5.f / 6.f * d2i));
    cb[CB_B + 2] = (double)(9.f / 8.f * d2i);
    cb[CB_B + 3] = (double)(1.f / 6.f * d2i);
    cb[CB_B + 4] = (double)(-(1.f / 96.f * d2i));
    cb[CB_F + 0] = (double)(-(10.0f / 3.f * d2i));
    cb[CB_F + 1] = (double)(-(3.0f * d2i));
    cb[CB_F + 2] = (double)(6.f * d2i);
    cb[CB_F + 3] = (double)(1.f / 3.f * d2i);
    const float alpha2 = 3.f / 4.f, gamma2 = 1.f / 8.f, beta1 = 3.f;
    cb[CB_ALPHA2] = alpha2;
    cb[CB_BETA1] = beta1;
    cb[CB_CNST] = (double)(1.f / (alpha2 - beta1 * gamma2));
}

void dbyd2_matrix(int N2, int ibc, std::vector<double> &lowr, std::vector<double> &uppr)
{
    const float alpha = 1.f / 3.f, alpha2 = 3.f / 4.f, gamma2 = 1.f / 8.f;
    const float alpha1 = 6.0f, beta1 = 3.f;
    const float cnst = 1.f / (alpha2 - beta1 * gamma2);
    const float up1 = (alpha1 * alpha2 - beta1) * cnst;
    uppr.assign(N2, 0.0);
    lowr.assign(N2, 0.0);
    for (int j = 2; j <= N2 - 3; j++) uppr[j] = alpha;
    uppr[0] = (ibc % 2 == 0) ? 0.0 : (double)up1;
    uppr[1] = alpha2;
    uppr[N2 - 2] = gamma2;
    for (int j = 0; j < N2; j++) lowr[j] = uppr[N2 - 1 - j];
    lowr[N2 - 1] = (ibc != 1 && ibc != 2) ? 0.0 : (double)up1;
    lowr[0] = 0.0;
    uppr[N2 - 1] = 0.0;
}

namespace {

// Invert an n x n matrix with unit diagonal blocks and a band around them (Gauss-Jordan,
// partial pivoting).  Columns of A up to the pivot's are not read again, and what lies
// below kTiny is too small to reach an entry that the tables keep (above 1e-24 of its
// row's largest, which is of order 1): neither is touched, and the tables come out bit for
// bit as with every element.  ms for the z-derivative's seven sets and the column pass's
// three, every element -> here: nz = 150 0.29 -> 0.22, 300 1.5 -> 0.78, 1000 5.1 -> 0.88.
bool invert(std::vector<double> A, int n, std::vector<double> &inv)
{
    constexpr double kTiny = 1e-60;
    inv.assign((size_t)n * n, 0.0);
    for (int i = 0; i < n; i++) inv[(size_t)i * n + i] = 1.0;
    for (int c = 0; c < n; c++) {
        int pr = c;
        for (int r = c + 1; r < n; r++)
            if (std::fabs(A[(size_t)r * n + c]) > std::fabs(A[(size_t)pr * n + c])) pr = r;
        if (A[(size_t)pr * n + c] == 0.0) return false;
        if (pr != c)
            for (int k = 0; k < n; k++) {
                std::swap(A[(size_t)pr * n + k], A[(size_t)c * n + k]);
                std::swap(inv[(size_t)pr * n + k], inv[(size_t)c * n + k]);
            }
        double *const ac = A.data() + (size_t)c * n, *const ic = inv.data() + (size_t)c * n;
        const double d = 1.0 / ac[c];
        int a1 = n, i0 = 0, i1 = n;
        while (a1 > c + 1 && ac[a1 - 1] == 0.0) a1--;
        while (i0 < n && std::fabs(ic[i0]) < kTiny) i0++;
        while (i1 > i0 && std::fabs(ic[i1 - 1]) < kTiny) i1--;
        for (int k = c + 1; k < a1; k++) ac[k] *= d;
        for (int k = i0; k < i1; k++) ic[k] *= d;
        for (int r = 0; r < n; r++) {
            if (r == c) continue;
            const double f = A[(size_t)r * n + c];
            if (std::fabs(f) < kTiny) continue;
            double *const ar = A.data() + (size_t)r * n, *const ir = inv.data() + (size_t)r * n;
            for (int k = c + 1; k < a1; k++) ar[k] -= f * ac[k];
            for (int k = i0; k < i1; k++) ir[k] -= f * ic[k];
        }
    }
    return true;
}

}  // namespace

namespace {

// The five segment tables of one tridiagonal matrix (sub- and super-diagonals
// lo, up of N rows, diagonal 1), rows [5][nzp] at tabs, and the exact inverse
// of its 2P x 2P interface system; widens hw to the largest distance in
// segments to an entry of the inverse above cut of its row maximum.
bool seg_one(int N, int m, const std::vector<double> &lo, const std::vector<double> &up, double *tabs,
             std::vector<double> &Minv, int &hw, double cut = 1e-24)
{
    const int P = (N + m - 1) / m;
    const int nzp = P * m, n2 = 2 * P;
    std::vector<double> lowr(nzp, 0.0), uppr(nzp, 0.0);
    for (int j = 0; j < N; j++) { lowr[j] = lo[j]; uppr[j] = up[j]; }
    std::vector<double> rbl(nzp, 1.0), gl(nzp, 0.0), V(nzp, 0.0), W(nzp, 0.0), bet(nzp, 1.0);
    for (int s = 0; s < P; s++) {
        const int a0 = s * m;
        for (int j = a0 + 1; j < a0 + m; j++) {
            gl[j] = uppr[j - 1] / bet[j - 1];
            bet[j] = 1.0 - lowr[j] * gl[j];
            rbl[j] = 1.0 / bet[j];
        }
        auto lsolve = [&](std::vector<double> r, double *out) {
            r[0] = r[0] * rbl[a0];
            for (int i = 1; i < m; i++) r[i] = (r[i] - lowr[a0 + i] * r[i - 1]) * rbl[a0 + i];
            for (int i = m - 2; i >= 0; i--) r[i] = r[i] - gl[a0 + i + 1] * r[i + 1];
            for (int i = 0; i < m; i++) out[a0 + i] = r[i];
        };
        std::vector<double> r(m, 0.0);
        if (s > 0) { r[0] = lowr[a0]; lsolve(r, V.data()); }
        std::fill(r.begin(), r.end(), 0.0);
        if (s < P - 1) { r[m - 1] = uppr[a0 + m - 1]; lsolve(r, W.data()); }
    }
    std::vector<double> M((size_t)n2 * n2, 0.0);
    for (int s = 0; s < P; s++) {
        const int f = s * m, l = s * m + m - 1;
        M[(size_t)(2 * s) * n2 + 2 * s] = 1.0;
        M[(size_t)(2 * s + 1) * n2 + 2 * s + 1] = 1.0;
        if (s > 0) {
            M[(size_t)(2 * s) * n2 + 2 * s - 1] += V[f];
            M[(size_t)(2 * s + 1) * n2 + 2 * s - 1] += V[l];
        }
        if (s < P - 1) {
            M[(size_t)(2 * s) * n2 + 2 * s + 2] += W[f];
            M[(size_t)(2 * s + 1) * n2 + 2 * s + 2] += W[l];
        }
    }
    if (!invert(M, n2, Minv)) return false;
    for (int k = 0; k < n2; k++) {
        double rm = 0.0;
        for (int q = 0; q < n2; q++) rm = std::max(rm, std::fabs(Minv[(size_t)k * n2 + q]));
        for (int q = 0; q < n2; q++)
            if (std::fabs(Minv[(size_t)k * n2 + q]) > cut * rm) hw = std::max(hw, std::abs(q / 2 - k / 2));
    }
    const std::vector<double> *all[5] = {&lowr, &rbl, &gl, &V, &W};
    for (int k = 0; k < 5; k++) std::copy(all[k]->begin(), all[k]->end(), tabs + (size_t)k * nzp);
    return true;
}

// Band storage of an interface inverse: row k keeps the entries q =
// 2 (k/2 - hw) + w, w < 4 hw + 4 (the window around its own segment), zero
// outside 0..2P-1.
void band_rows(const std::vector<double> &Minv, int n2, int hw, double *band)
{
    const int W = 4 * hw + 4;
    for (int k = 0; k < n2; k++)
        for (int w = 0; w < W; w++) {
            const int q = 2 * (k / 2 - hw) + w;
            band[(size_t)k * W + w] = q >= 0 && q < n2 ? Minv[(size_t)k * n2 + q] : 0.0;
        }
}

// Rows [nrow][3][m] of the first, an interior and the last segment of rows
// [nrow][nzp]; false if some interior segment's tables differ from the first
// interior one's.
bool kind_rows(const double *rows, int nrow, int P, int m, std::vector<double> &out)
{
    const int nzp = P * m, sk[3] = {0, P > 1 ? 1 : 0, P - 1};
    for (int r = 0; r < nrow; r++) {
        const double *row = rows + (size_t)r * nzp;
        for (int s = 2; s < P - 1; s++)
            if (std::memcmp(row + (size_t)s * m, row + m, (size_t)m * sizeof(double))) return false;
        for (int k = 0; k < 3; k++) out.insert(out.end(), row + (size_t)sk[k] * m, row + (size_t)(sk[k] + 1) * m);
    }
    return true;
}

}  // namespace

bool build_seg_tables(int N, int m, SegTables &t)
{
    const int P = (N + m - 1) / m;
    const int nzp = P * m, n2 = 2 * P;
    t.P = P;
    t.m = m;
    t.nzp = nzp;
    t.slots.assign((size_t)3 * 5 * nzp, 0.0);
    std::vector<double> minv[3];
    int hw = 0;
    const int ibcs[3] = {1, 2, 3};
    for (int slot = 0; slot < 3; slot++) {
        std::vector<double> lo, up;
        dbyd2_matrix(N, ibcs[slot], lo, up);
        if (!seg_one(N, m, lo, up, t.slots.data() + (size_t)5 * slot * nzp, minv[slot], hw)) return false;
    }
    t.hw = hw;
    const int W = 4 * hw + 4;
    t.band.assign((size_t)3 * n2 * W, 0.0);
    for (int slot = 0; slot < 3; slot++) band_rows(minv[slot], n2, hw, t.band.data() + (size_t)slot * n2 * W);
    return true;
}

bool build_seg_rows(int N, int m, SegRows &t)
{
    const int P = (N + m - 1) / m;
    const int nzp = P * m, n2 = 2 * P;
    t.P = P;
    t.m = m;
    t.nzp = nzp;
    t.hw = 0;
    t.slots.assign((size_t)3 * 5 * nzp, 0.0);
    std::vector<double> minv[3];
    const int ibcs[3] = {1, 2, 3};
    for (int slot = 0; slot < 3; slot++) {
        std::vector<double> lo, up;
        dbyd2_matrix(N, ibcs[slot], lo, up);
        if (!seg_one(N, m, lo, up, t.slots.data() + (size_t)5 * slot * nzp, minv[slot], t.hw, 1e-19)) return false;
    }
    const int nw = 4 * t.hw + 4;
    // the two rows of segment s: row 2s-1 around segment s-1, row 2s+2 around s+1
    auto pair_rows = [&](int slot, int s) {
        std::vector<double> r((size_t)2 * nw, 0.0);
        for (int h = 0; h < 2; h++) {
            const int k = h ? 2 * s + 2 : 2 * s - 1, c = h ? s + 1 : s - 1;
            if (c < 0 || c >= P) continue;
            for (int w = 0; w < nw; w++) {
                const int q = 2 * (c - t.hw) + w;
                if (q >= 0 && q < n2) r[(size_t)h * nw + w] = minv[slot][(size_t)k * n2 + q];
            }
        }
        return r;
    };
    const int mid = P / 2;
    t.E = 0;
    for (int slot = 0; slot < 3; slot++) {
        const std::vector<double> ref = pair_rows(slot, mid);
        double big = 0.0;
        for (double v : ref) big = std::max(big, std::fabs(v));
        for (int s = 0; s < P; s++) {
            const std::vector<double> r = pair_rows(slot, s);
            double d = 0.0;
            for (size_t q = 0; q < r.size(); q++) d = std::max(d, std::fabs(r[q] - ref[q]));
            if (d > 1e-18 * big) t.E = std::max(t.E, std::min(s, P - 1 - s) + 1);
        }
    }
    const int nk = seg_band_kinds(P, t.E);
    if (nk == P) t.E = P;                                     // too short a column to repeat: every segment its own
    t.rows.clear();
    for (int slot = 0; slot < 3; slot++)
        for (int k = 0; k < nk; k++) {
            const int s = t.E == P || k < t.E ? k : (k == t.E ? mid : P - (2 * t.E + 1 - k));
            const std::vector<double> r = pair_rows(slot, s);
            t.rows.insert(t.rows.end(), r.begin(), r.end());
        }
    return true;
}

int zseg_length(int N)
{
    static const int sizes[] = {
#define X(v) v,
        SPARC_ZDER_SIZES(X)
#undef X
    };
    for (int m : sizes) {
        const int P = (N + m - 1) / m;
        if (P <= (N <= 160 ? kZSegP / 2 : kZSegP) && N - (P - 1) * m >= 3) return m;
    }
    return 0;
}

bool build_zseg(int N, int m, int nset, const int *sets, int &hw, std::vector<double> &img)
{
    const int P = (N + m - 1) / m;
    const int nzp = P * m, n2 = 2 * P;
    std::vector<std::vector<double>> minv(nset), tabs(nset);
    hw = 0;
    for (int k = 0; k < nset; k++) {
        std::vector<double> lo, up;
        dbyd2_matrix(N, sets[k] & 3, lo, up);
        if (sets[k] & kZSegT) {                               // the transposed matrix
            std::vector<double> lt(N, 0.0), ut(N, 0.0);
            for (int j = 1; j < N; j++) lt[j] = up[j - 1];
            for (int j = 0; j + 1 < N; j++) ut[j] = lo[j + 1];
            lo = lt;
            up = ut;
        }
        tabs[k].assign((size_t)5 * nzp, 0.0);
        if (!seg_one(N, m, lo, up, tabs[k].data(), minv[k], hw)) return false;
    }
    const int W = 4 * hw + 4;
    img.clear();
    for (int k = 0; k < nset; k++) {
        std::vector<double> band((size_t)n2 * W);
        band_rows(minv[k], n2, hw, band.data());
        img.insert(img.end(), band.begin(), band.end());
        if (!kind_rows(tabs[k].data(), 5, P, m, img)) return false;
        if (img.size() & 1) img.push_back(0.0);               // every set starts on 16 bytes
    }
    return true;
}

void dbyd2_edge_rows(int N2, int ibc, double eb[20])
{
    double c1, c2, cb[kCB];
    dbyd2_coefs(N2, c1, c2, cb);
    for (int k = 0; k < 5; k++) {
        const double f = k < 4 ? cb[CB_F + k] : 0.0, b = cb[CB_B + k];
        const double far = (cb[CB_ALPHA2] * f - cb[CB_BETA1] * b) * cb[CB_CNST];
        eb[k] = ibc & 1 ? far : 0.0;
        eb[5 + k] = b;
        eb[10 + 4 - k] = -b;
        eb[15 + 4 - k] = ibc == 1 || ibc == 2 ? -far : 0.0;
    }
}

bool seg_kind_tables(const SegRows &t, std::vector<double> &out)
{
    out.clear();
    out.reserve((size_t)15 * 3 * t.m);
    return kind_rows(t.slots.data(), 15, t.P, t.m, out);
}

bool seg_kind_tables(const SegTables &t, std::vector<double> &out)
{
    out.clear();
    out.reserve((size_t)15 * 3 * t.m);
    return kind_rows(t.slots.data(), 15, t.P, t.m, out);
}

}  // namespace sparc
