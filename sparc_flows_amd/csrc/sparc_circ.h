// sparc_circ.h -- the spectral derivative of a line whose length n is not a
// power of two (16 <= n <= 1024): the same linear map as the FFT form (bin k
// times i*dmul[k]; an odd n has no Nyquist bin to drop), as a circulant product
//     (D z)[x] = sum_m c[m] z[x - m],  indices mod n,
// with c the map's first column.  O(n^2): the work is in the products, so they are
// halved where n is even and fed from registers.
//
//   * Even n = 2 h.  z^n - 1 = (z^h - 1)(z^h + 1): the product splits into a
//     cyclic one of length h on u[j] = z[j] + z[j+h] and a negacyclic one on
//     w[j] = z[j] - z[j+h], with columns cp[m] = (c[m] + c[m+h])/2 and
//     cm[m] = (c[m] - c[m+h])/2; the halves of the result are p + q and p - q.
//     That is half the multiplications, and sums of half the length.  An odd n
//     runs the one product of length n.
//   * A lane makes kCircR = 5 neighbouring outputs of two real lines at once
//     (one double2): per m it loads one new element of its window (16 bytes) and the
//     one coefficient all outputs share, for 10 multiply-adds.  LDS then takes about
//     as long as the FP64 units; one output per lane and m (a coefficient from LDS
//     for every product) spent two LDS cycles per multiply-add.  An odd R keeps the
//     lanes' 16-byte windows on different banks.
//   * The lines are held twice over (negated below 0 for w), so that x - m needs no
//     wrap.  m runs in whole chunks of kCircK; the coefficients past the end are zero
//     and the line is led by zeros, so that a chunk past the end adds zeros.
//
// us per launch, a row on 64 lanes with every coefficient from LDS -> here.  Row pass
// (one source; 300 rows were 300 waves on 1024 SIMDs): nx = 300, nz = 300 43.5 ->
// 16.4; 96 x 100 13.6 -> 9.9; 1000 x 100 554 -> 41; 8 sources of 300 x 300 94 -> 49.
// 3D derivatives at 96 x 90 x 100 (mean of launches of one and three fields): x 24 ->
// 14.4, y 28 -> 13.3.
#pragma once
#include <hip/hip_runtime.h>

namespace sparc {

constexpr int kCircR = 5;     // outputs per lane
constexpr int kCircK = 10;    // m per chunk, a multiple of kCircR
constexpr int kCircUnits = 256;   // compute units

struct CircShape {
    int n, nk, len;           // line, products (2: cyclic and negacyclic halves), their length
    int L, lanes;             // lanes per product and per line
    int plen, ext;            // padded column length, elements of one product's doubled line
};
__host__ __device__ inline CircShape circ_shape(int n)
{
    CircShape s;
    s.n = n;
    s.nk = n & 1 ? 1 : 2;
    s.len = n / s.nk;
    s.L = (s.len + kCircR - 1) / kCircR;
    s.lanes = s.nk * s.L;
    s.plen = (s.len + kCircK - 1) / kCircK * kCircK;
    s.ext = kCircK + 2 * s.len + kCircR;
    return s;
}

// Element j of product kind k (0: u, or the line itself; 1: w) into both places of its
// doubled line e = ext[k], whose index 0 is element -len - kCircK.
__device__ __forceinline__ void circ_put(double2 *e, int len, int kind, int j, double2 v)
{
    e[kCircK + len + j] = v;
    e[kCircK + j] = kind ? make_double2(-v.x, -v.y) : v;
}

// acc[r] += sum over the chunks [m0, m1) of c[m] z[x0 + r - m], r < kCircR; src = the
// address of z[x0].  Reads z[x0 - m1 + 1 .. x0 + kCircR - 1], c[m0 .. m1).
__device__ __forceinline__ void circ_sum(double (&ar)[kCircR], double (&ai)[kCircR], const double2 *src,
                                         const double *c, int m0, int m1)
{
    constexpr int R = kCircR, K = kCircK;
    double2 w[K + R - 1];             // w[i] = z[x0 + R-1 - m - i]
#pragma unroll
    for (int i = 0; i < R - 1; i++) w[i] = src[R - 1 - m0 - i];
    for (int m = m0; m < m1; m += K) {
        double cv[K];
#pragma unroll
        for (int i = 0; i < K; i++) cv[i] = c[m + i];
#pragma unroll
        for (int i = 0; i < K; i++) w[R - 1 + i] = src[-m - i];
#pragma unroll
        for (int i = 0; i < K; i++) {
#pragma unroll
            for (int r = 0; r < R; r++) {
                ar[r] += cv[i] * w[R - 1 - r + i].x;
                ai[r] += cv[i] * w[R - 1 - r + i].y;
            }
        }
#pragma unroll
        for (int i = 0; i < R - 1; i++) w[i] = w[i + K];
    }
}

// One line per block of B lanes (the row pass): lane t holds z[t + B j2], j2 < N2,
// B N2 >= n; slots past n carry nothing and get garbage.  With one line per block
// the m range is split as well, over as many groups of lanes as fit (at most 4), and
// their sums are added through LDS.
template <int B, int N2> struct CircLds {
    static constexpr int raw = B * N2;
    // doubled lines (even: 2 (n + 15), odd: 2 n + 15), or the partial sums
    // (splits n, at most 5 B elements: splits <= B / ceil(n / 5))
    static constexpr int work = 2 * B * N2 + 30 > 5 * B ? 2 * B * N2 + 30 : 5 * B;
    static constexpr int n = raw + work;
    static constexpr int c = B * N2 + 20;        // the table
};

// z: CircLds<B, N2>::n elements; cc: the table.  Every lane of the block must call
// this (it contains block barriers).
template <int B, int N2>
__device__ __forceinline__ void circ_deriv_block(double (&re)[N2], double (&im)[N2], int t, double2 *z,
                                                 const double *cc, int n, double stretch)
{
    const CircShape s = circ_shape(n);
    double2 *const work = z + CircLds<B, N2>::raw;
#pragma unroll
    for (int j2 = 0; j2 < N2; j2++) {
        const int x = t + B * j2;
        if (x < n) z[x] = make_double2(re[j2], im[j2]);
    }
    __syncthreads();
    for (int q = t; q < kCircK * s.nk; q += B) work[q < kCircK ? q : s.ext + q - kCircK] = make_double2(0.0, 0.0);
    for (int j = t; j < s.len; j += B) {
        const double2 a = z[j];
        if (s.nk == 1) {
            circ_put(work, s.len, 0, j, a);
        } else {
            const double2 o = z[j + s.len];
            circ_put(work, s.len, 0, j, make_double2(a.x + o.x, a.y + o.y));
            circ_put(work + s.ext, s.len, 1, j, make_double2(a.x - o.x, a.y - o.y));
        }
    }
    __syncthreads();
    // group of lanes g = split, then product, then output block
    const int ns = min(4, B / s.lanes), chunks = s.plen / kCircK;
    const int g = t / s.lanes, l = t - g * s.lanes, kind = l >= s.L ? 1 : 0, x0 = kCircR * (l - kind * s.L);
    double ar[kCircR], ai[kCircR];
#pragma unroll
    for (int r = 0; r < kCircR; r++) ar[r] = ai[r] = 0.0;
    if (g < ns)
        circ_sum(ar, ai, work + kind * s.ext + kCircK + s.len + x0, cc + kind * s.plen, kCircK * (g * chunks / ns),
                 kCircK * ((g + 1) * chunks / ns));
    __syncthreads();       // the doubled lines make room for the partial sums
    if (g < ns) {
#pragma unroll
        for (int r = 0; r < kCircR; r++)
            if (x0 + r < s.len) work[g * n + kind * s.len + x0 + r] = make_double2(ar[r], ai[r]);
    }
    __syncthreads();
#pragma unroll
    for (int j2 = 0; j2 < N2; j2++) {
        const int x = t + B * j2;
        if (x < n) {
            const int hi = s.nk == 2 && x >= s.len, j = hi ? x - s.len : x;
            double pr = 0.0, pi = 0.0, qr = 0.0, qi = 0.0;
            for (int k = 0; k < ns; k++) {
                const double2 p = work[k * n + j];
                pr += p.x;
                pi += p.y;
                if (s.nk == 2) {
                    const double2 q = work[k * n + s.len + j];
                    qr += q.x;
                    qi += q.y;
                }
            }
            re[j2] = (hi ? pr - qr : pr + qr) * stretch;
            im[j2] = (hi ? pi - qi : pi + qi) * stretch;
        }
    }
}

// Many lines: blocks of 256 lanes take G pairs of lines, lanes of them a pair: as many
// pairs as fit a block, unless that would leave more than half of the compute units without one;
// then only as many as spread them over all units, and the lanes left over split the
// m range, ns groups a pair.  us a call of 100 rows (host and wait included: 20), full
// blocks / spread: n = 17 24.2 / 21.8, 75 26.0 / 22.1, 121 27.6 / 22.7, 300 26.9 / 23.4;
// 800 rows of 300 27.7 / 25.7, 1600 28.1 / 27.7.
struct CircBatch {
    CircShape s;
    int G, ns;
    size_t lds;               // bytes
};
inline CircBatch circ_batch(int n, int axis, long pairs)
{
    CircBatch b;
    b.s = circ_shape(n);
    const size_t table = sizeof(double) * b.s.nk * b.s.plen, line = sizeof(double2) * b.s.nk * b.s.ext;
    const int lds = (int)((65536 - table) / line);       // lines a block holds
    b.G = 256 / b.s.lanes < lds ? 256 / b.s.lanes : lds;
    // along y the G column pairs of a block are neighbours: whole 64-byte pieces of
    // each row
    if (axis == 1 && b.G > 4) b.G -= b.G % 4;
    b.ns = 1;
    const long spread = (pairs + kCircUnits - 1) / kCircUnits;
    if (2 * spread <= b.G) {
        b.G = (int)spread;
        while (b.ns < 4 && (b.ns + 1) * b.G * b.s.lanes <= 256 && (b.ns + 1) * b.G <= lds) b.ns++;
    }
    b.lds = table + line * b.G * b.ns;
    return b;
}

}  // namespace sparc
