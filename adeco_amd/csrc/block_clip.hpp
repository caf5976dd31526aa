// Exact shares of a tet in the cells of a small block, for FP64 deposits on grids of unit scaled
// cells (host and device).
//
// A block is cx * cy * cz unit cells; the tet is given in cells relative to the block's corner.  The
// share of cell (a, b, k) is a difference of cumulative shares
//     G(p, q, h) = |T ∩ {x < p, y < q, z < h}| / |T|
// over the block's face planes, so a plane between two cells is cut once for both, and a tet that
// lies inside the block is cut by its inner planes only:
//   * x: with the vertices sorted by x, the part of T below plane p is a corner tet (1 vertex below),
//     a wedge of 3 tets (2), T minus the corner beyond (3) or T itself (4);
//   * y: each of these pieces (and T itself, once for all planes it is whole in) is cut by the y planes
//     in the same way;
//   * z: the share of a piece below a plane is closed form in its 4 sorted heights.
// Only the coordinates still needed are carried: (y, z) after the x cut, z after the y cut.  A piece's
// volume is its parent's times a product of edge ratios, so no determinant is taken.  A share's absolute error is a
// few ulps of the whole tet, and of a tet (or piece of it) that is thin across y or z and cut along there, a few
// roundings of the coordinate over the thickness.  A cell whose share is small against that error (small_share) is
// recomputed alone by exact_cell_share, whose pieces do not overlap and whose terms are all positive.
#pragma once

#include "adeco_geom.hpp"

namespace adeco {

// Largest number of cells in a block.
constexpr int kBlockCells = 24;
// Shares of a cell below kNoShare (18 ulps of the tet, which large tets are first made smaller for: the differences'
// rounding) are empty; between that and small_share() they are recomputed by exact_cell_share.
constexpr double kNoShare = 4e-15;
constexpr double kSmallShare = 1e-8, kThinShare = 1e-9;
// A share this close to a whole cell's is one: a cell that lies wholly in the tet is exact.
constexpr double kNearFull = 2e-15;
// Tets of more than 30 cells' volume are replaced by smaller ones, block by block (shrink_tet).
constexpr double kLargeTet = 1.0 / 30.0;
// Where more than 20 000 cells' volume are left of one (two faces at a small angle across the block), or where the
// rounding of its planes' distance counts (tets about 1000 cells wide), the block's cells are recomputed alone.
constexpr double kHugeTet = 1.0 / 20000.0, kVastTet = 1e-8;

// 1 / b for a positive denominator, within an ulp or two
ADECO_HD double recip(double b) {
#if defined(__HIP_DEVICE_COMPILE__)
    double r = __builtin_amdgcn_rcp(b);
    r = fma(fma(-b, r, 1.0), r, r);
    return fma(fma(-b, r, 1.0), r, r);
#else
    return 1.0 / b;
#endif
}

// int(floor(v)) of a value clamped to [-1, top]
ADECO_HD int floor_clamped(double v, int top) { return int(floor(fmax(fmin(v, double(top)), -1.0))); }
// int(ceil(v)) of a value clamped to [-1, top + 1]
ADECO_HD int ceil_clamped(double v, int top) { return int(ceil(fmax(fmin(v, double(top + 1)), -1.0))); }

ADECO_HD int imin(int a, int b) { return a < b ? a : b; }

// Compare-and-swap network by key, payloads carried along.
ADECO_HD void order2(double& ka, double& kb, double& pa, double& pb) {
    const bool s = kb < ka;
    const double k0 = s ? kb : ka, k1 = s ? ka : kb, p0 = s ? pb : pa, p1 = s ? pa : pb;
    ka = k0; kb = k1; pa = p0; pb = p1;
}
ADECO_HD void order3(double& ka, double& kb, double& pa, double& pb, double& qa, double& qb) {
    const bool s = kb < ka;
    const double q0 = s ? qb : qa, q1 = s ? qa : qb;
    order2(ka, kb, pa, pb);
    qa = q0; qb = q1;
}

// Planes first..last (of 0..n) cut a tet whose key coordinates, sorted, are k0 <= k1 <= k2 <= k3; the
// whole tet counts from row `whole` (n: in none) on: the first whose upper plane has 3 of its vertices
// below it or all of it on the low side, unless plane 0 has as well.
struct PlaneRange {
    int first, last, whole;
    ADECO_HD void set(double k0, double k2, double k3, int n) {
        const int c3 = ceil_clamped(k3, n) - 1;
        first = floor_clamped(k0, n) + 1;
        last = imin(c3, n);
        last = last < first - 1 ? first - 1 : last;  // (a flat piece on a plane)
        whole = imin(floor_clamped(k2, n), c3);
        whole = k2 < 0.0 || whole < 0 ? n : whole;
    }
};

// The cut of a tet, sorted by its key coordinate (k0 <= k1 <= k2 <= k3), by a plane that n (1-3) of
// its vertices lie below: the four edge ratios in use.  Edges: A = (0, 3); B = (0, 2), or (1, 3) when
// n = 3; C = (0, 1), (1, 3), (2, 3) for n = 1, 2, 3; D = (1, 2), used when n = 2.  The part below is
//   n = 1  the corner (v0, A, B, C),                       share tA tB tC
//   n = 2  (v0, A, B, v1), (D, A, B, v1), (D, A, C, v1),   shares tA tB, tA uB tD, uA tD tC
//   n = 3  the tet minus (v3, A, B, C),                    share uA uB uC
// with t the ratio from the edge's lower end and u = 1 - t.
struct EdgeCut {
    double tA, tB, tC, tD;
    double w0, w1, w2;  // signed shares of the pieces
    bool one, three;    // n == 1, n == 3
    ADECO_HD void set(double k0, double k1, double k2, double k3, double plane) {
        one = !(k1 < plane);
        three = k2 < plane;
        const double lB = three ? k1 : k0, hB = three ? k3 : k2;
        const double lC = one ? k0 : (three ? k2 : k1), hC = one ? k1 : k3;
        const double rA = recip(k3 - k0), rB = recip(hB - lB), rC = recip(hC - lC), rD = recip(k2 - k1);
        tA = (plane - k0) * rA;
        tB = (plane - lB) * rB;
        tC = (plane - lC) * rC;
        tD = (plane - k1) * rD;
        const double uA = (k3 - plane) * rA, uB = (hB - plane) * rB;
        const double cA = three ? uA : tA, cB = three ? uB : tB, cC = three ? (hC - plane) * rC : tC;
        const double ab = cA * cB;
        const bool two = !one && !three;
        w0 = two ? ab : (three ? -ab * cC : ab * cC);
        w1 = tA * uB * tD;
        w2 = uA * tD * tC;
    }
    ADECO_HD int pieces() const { return one || three ? 1 : 3; }
    // values at the cut points of a coordinate that is v0..v3 at the vertices
    ADECO_HD double atA(double v0, double v3) const { return fma(tA, v3 - v0, v0); }
    ADECO_HD double atB(double v0, double v1, double v2, double v3) const {
        const double l = three ? v1 : v0, h = three ? v3 : v2;
        return fma(tB, h - l, l);
    }
    ADECO_HD double atC(double v0, double v1, double v2, double v3) const {
        const double l = one ? v0 : (three ? v2 : v1), h = one ? v1 : v3;
        return fma(tC, h - l, l);
    }
    ADECO_HD double atD(double v1, double v2) const { return fma(tD, v2 - v1, v1); }
};

// Keeps a value from being computed ahead of the loop it is used in: the plane loops mostly run once,
// and what would be hoisted out of them costs registers.
#if defined(__HIP_DEVICE_COMPILE__)
#define ADECO_KEEP_IN_LOOP(v) asm volatile("" : "+v"(v))
#else
#define ADECO_KEEP_IN_LOOP(v)
#endif

// Where a piece counts: + in row (or column) `at` and, as the difference of neighbouring cumulative
// shares, - in row `at` + 1 (`both`).
struct Rows {
    int at;
    bool both;
};

// The same for a row and a column of cells: the index of the first cell of column yr in row xr, and the steps
// to the next column and row (0: not counted there), in a block of cy columns of cz cells.
struct Target {
    int base, dy, dx, cz;
    ADECO_HD Target() {}
    ADECO_HD Target(Rows xr, Rows yr, int cy, int cz_)
        : base((xr.at * cy + yr.at) * cz_), dy(yr.both ? cz_ : 0), dx(xr.both ? cy * cz_ : 0), cz(cz_) {}
};

// Shares of a tet below this are recomputed: the rounding of a cut point counts against the extents of what it
// is cut from, so by far less in a flat tet across y or z (1e-4 cells thick and cut along, shares of 1e-8..1e-6: 1.5e-5
// off at most with kSmallShare alone, 4e-9 so, 5e-7 one tet per thread; 3 % more recomputes of ordinary tets).  Not
// across x, whose coordinates are the vertices' own.
ADECO_HD double small_share(const double y[4], const double z[4]) {
    const double ey = fmax(fmax(y[0], y[1]), fmax(y[2], y[3])) - fmin(fmin(y[0], y[1]), fmin(y[2], y[3]));
    const double ez = fmax(fmax(z[0], z[1]), fmax(z[2], z[3])) - fmin(fmin(z[0], z[1]), fmin(z[2], z[3]));
    return fma(kThinShare, recip(fmin(ey, ez)), kSmallShare);
}

// A share as an integer of 2^-62, and a sum of such.  Pieces reach a block's sums in an order that depends on what
// else the wave clips, and a sum of integers does not depend on its order (the unit is far below the rounding of a
// share, and what wraps on the way wraps back).  The lower part of a tiny negative share rounds up to 2^32, which has
// no conversion to unsigned.
ADECO_HD long long fixed_share(double share) {
    const double t = share * 0x1p30, hi = floor(t);
    return (long long)((unsigned long long)(unsigned)int(hi) << 32 | unsigned(fmin((t - hi) * 0x1p32, 4294967295.0)));
}
ADECO_HD double from_fixed(unsigned long long v) { return double((long long)v) * 0x1p-62; }

// Adds the shares of a piece with heights z0..z3 (any order) and signed share w between the z planes
// 0..cz, cell by cell, where t says.  Without branches but for the loop over the planes that cut it: an add
// that does not apply adds 0 to the same cell.  Acc: term(share) a value to sum (with its negative), add(cell,
// value).
template <class Acc>
ADECO_HD void block_leaf(double z0, double z1, double z2, double z3, double w, Target t, Acc& acc) {
#define ADECO_MINMAX(u, v)        \
    {                             \
        const double lo_ = fmin(u, v); \
        v = fmax(u, v);           \
        u = lo_;                  \
    }
    ADECO_MINMAX(z0, z1) ADECO_MINMAX(z2, z3) ADECO_MINMAX(z0, z2) ADECO_MINMAX(z1, z3) ADECO_MINMAX(z1, z2)
#undef ADECO_MINMAX
    // planes first..last cut the piece
    const int first = floor_clamped(z0, t.cz) + 1, last = ceil_clamped(z3, t.cz) - 1;
    const int base = t.base, by = base + t.dy, bx = base + t.dx, bxy = bx + t.dy;
    const double d20 = z2 - z0, d30 = z3 - z0, d31 = z3 - z1;
    const double D1 = (z1 - z0) * d20 * d30, D2 = d20 * d30 * (z2 - z1) * d31, D3 = d30 * d31 * (z3 - z2);
    double prev = 0.0;
    int h = first;
    const auto emit = [&](int k, double v) {
        const auto u = acc.term(v), zero = u - u, vx = t.dx ? -u : zero;
        acc.add(base + k, u);
        acc.add(by + k, t.dy ? -u : zero);
        acc.add(bx + k, vx);
        acc.add(bxy + k, t.dy ? -vx : zero);
    };
    for (; h <= last; ++h) {
        const double zh = double(h);
        const double a = zh - z0, b = zh - z1, c = z2 - zh, e = z3 - zh;
        const bool one = zh <= z1, three = zh > z2;
        const double ab = a * b, apb = a + b;
        double num2 = ab * ab + ab * apb * (c + e) + c * e * (apb * apb - ab);
        ADECO_KEEP_IN_LOOP(num2);
        const double k = one ? a : e;
        const double num = one || three ? k * k * k : num2;
        const double f = num * recip(one ? D1 : (three ? D3 : D2));
        const double below = three ? 1.0 - f : f;
        emit(h > 0 ? h - 1 : 0, h > 0 ? w * (below - prev) : 0.0);
        prev = below;
    }
    // the cell above the last plane, or the piece's only cell
    const bool top = last < t.cz && z3 > 0.0 && z0 < double(t.cz);
    emit(top ? h - 1 : 0, top ? w * (1.0 - prev) : 0.0);
}

// Takes the leaves (pieces of both cuts) of block_shares as they come.  On the device one that gathers them over
// the lanes of a wave takes its place, whose loops therefore go on while any lane has work: any(b) is true if b
// is for any of them.
template <class Acc>
struct LeafSums {
    Acc& acc;
    ADECO_HD bool any(bool b) const { return b; }
    ADECO_HD void leaf(bool on, double z0, double z1, double z2, double z3, double w, Target t) {
        if (on) block_leaf(z0, z1, z2, z3, w, t, acc);
    }
};

// One piece (y, z at its vertices, any order; signed share w) against the y planes 0..cy.
template <class Leaves>
ADECO_HD void block_piece(bool on, double y0, double y1, double y2, double y3, double z0, double z1, double z2, double z3, double w,
                          Rows xr, int cy, int cz, Leaves& leaves) {
    order2(y0, y1, z0, z1);
    order2(y2, y3, z2, z3);
    order2(y0, y2, z0, z2);
    order2(y1, y3, z1, z3);
    order2(y1, y2, z1, z2);
    PlaneRange r;
    r.set(y0, y2, y3, cy);
    for (int q = r.whole < cy ? r.first - 1 : r.first; leaves.any(on && q <= r.last); ++q) {
        // the piece itself, or what the cut by plane q leaves below it
        const bool t = q < r.first;
        ADECO_KEEP_IN_LOOP(y0);
        ADECO_KEEP_IN_LOOP(y1);
        ADECO_KEEP_IN_LOOP(y2);
        ADECO_KEEP_IN_LOOP(z1);
        ADECO_KEEP_IN_LOOP(z3);
        EdgeCut e;
        e.set(y0, y1, y2, y3, double(q));
        const double hC = e.atC(z0, z1, z2, z3), hD = e.atD(z1, z2);
        const double hA = t ? z3 : e.atA(z0, z3);
        double hB = t ? z2 : e.atB(z0, z1, z2, z3);
        double g0 = !t && e.three ? z3 : z0;
        const double g3 = t || (!e.one && !e.three) ? z1 : hC;
        double s = t ? w : (q > 0 ? w : -w) * e.w0;
        const int np = on && q <= r.last ? (t ? 1 : e.pieces()) : 0;
        const Rows yr{t ? r.whole : (q > 0 ? q - 1 : 0), !t && q > 0 && q < cy};
        const Target at(xr, yr, cy, cz);
        for (int k = 0;;) {
            leaves.leaf(k < np, g0, hA, hB, g3, s, at);
            if (!leaves.any(++k < np)) break;
            hB = k == 2 ? hC : hB;
            g0 = hD;
            s = (q > 0 ? w : -w) * (k == 1 ? e.w1 : e.w2);
        }
    }
}

// Gives `leaves` the pieces of the tet (vertices x, y, z in cells from the block's corner) that sum to its share
// in every cell of the block (index (a * cy + b) * cz + k).  cx * cy * cz <= kBlockCells.  on: there is a tet.
template <class Leaves>
ADECO_HD void block_shares(bool on, const double x[4], const double y[4], const double z[4], int cx, int cy, int cz,
                           Leaves& leaves) {
    double x0 = x[0], x1 = x[1], x2 = x[2], x3 = x[3];
    double y0 = y[0], y1 = y[1], y2 = y[2], y3 = y[3];
    double z0 = z[0], z1 = z[1], z2 = z[2], z3 = z[3];
    order3(x0, x1, y0, y1, z0, z1);
    order3(x2, x3, y2, y3, z2, z3);
    order3(x0, x2, y0, y2, z0, z2);
    order3(x1, x3, y1, y3, z1, z3);
    order3(x1, x2, y1, y2, z1, z2);
    PlaneRange r;
    r.set(x0, x2, x3, cx);
    for (int p = r.whole < cx ? r.first - 1 : r.first; leaves.any(on && p <= r.last); ++p) {
        // the tet itself, or the pieces of the part below plane p
        const bool t = p < r.first;
        ADECO_KEEP_IN_LOOP(x0);
        ADECO_KEEP_IN_LOOP(x1);
        ADECO_KEEP_IN_LOOP(x2);
        ADECO_KEEP_IN_LOOP(y1);
        ADECO_KEEP_IN_LOOP(y3);
        ADECO_KEEP_IN_LOOP(z1);
        ADECO_KEEP_IN_LOOP(z3);
        EdgeCut e;
        e.set(x0, x1, x2, x3, double(p));
        const double cy_ = e.atC(y0, y1, y2, y3), cz_ = e.atC(z0, z1, z2, z3);
        const double dy_ = e.atD(y1, y2), dz_ = e.atD(z1, z2);
        const bool two = !e.one && !e.three;
        double py0 = !t && e.three ? y3 : y0, pz0 = !t && e.three ? z3 : z0;
        const double py1 = t ? y3 : e.atA(y0, y3), pz1 = t ? z3 : e.atA(z0, z3);
        double py2 = t ? y2 : e.atB(y0, y1, y2, y3), pz2 = t ? z2 : e.atB(z0, z1, z2, z3);
        const double py3 = t || two ? y1 : cy_, pz3 = t || two ? z1 : cz_;
        double w = t ? 1.0 : (p > 0 ? e.w0 : -e.w0);
        const int np = on && p <= r.last ? (t ? 1 : e.pieces()) : 0;
        const Rows xr{t ? r.whole : (p > 0 ? p - 1 : 0), !t && p > 0 && p < cx};
        for (int k = 0;;) {
            block_piece(k < np, py0, py1, py2, py3, pz0, pz1, pz2, pz3, w, xr, cy, cz, leaves);
            if (!leaves.any(++k < np)) break;
            py2 = k == 2 ? cy_ : py2;
            pz2 = k == 2 ? cz_ : pz2;
            py0 = dy_;
            pz0 = dz_;
            w = k == 1 ? e.w1 : e.w2;
            w = p > 0 ? w : -w;
        }
    }
}

// The part of a tet with key >= 0 as non-overlapping pieces: windows i..i+3 (i < count) of a sequence
// of 6 points of M coordinates, with their shares.  k: the key at the vertices, v: the coordinates.
template <int M>
struct PositivePart {
    double s[M][6], w[3];
    int count;
    ADECO_HD void set(const double kin[4], const double vin[M][4]) {
        double k[4] = {kin[0], kin[1], kin[2], kin[3]}, v[M][4];
        for (int m = 0; m < M; ++m)
            for (int i = 0; i < 4; ++i) v[m][i] = vin[m][i];
#define ADECO_ORDER(a, b)                                                  \
    {                                                                      \
        const bool sw = k[b] < k[a];                                       \
        const double ka = sw ? k[b] : k[a], kb = sw ? k[a] : k[b];         \
        k[a] = ka; k[b] = kb;                                              \
        for (int m = 0; m < M; ++m) {                                      \
            const double va = sw ? v[m][b] : v[m][a], vb = sw ? v[m][a] : v[m][b]; \
            v[m][a] = va; v[m][b] = vb;                                    \
        }                                                                  \
    }
        ADECO_ORDER(0, 1) ADECO_ORDER(2, 3) ADECO_ORDER(0, 2) ADECO_ORDER(1, 3) ADECO_ORDER(1, 2)
#undef ADECO_ORDER
        const int n = int(k[0] < 0.0) + int(k[1] < 0.0) + int(k[2] < 0.0) + int(k[3] < 0.0);
        w[0] = 1.0;
        w[1] = w[2] = 0.0;
        if (n == 0 || n == 4) {
            for (int m = 0; m < M; ++m) {
                for (int i = 0; i < 4; ++i) s[m][i] = v[m][i];
                s[m][4] = s[m][5] = v[m][3];
            }
            count = n == 0 ? 1 : 0;
            return;
        }
        if (n == 1) {  // (v1, v2, v3) - (p1, p2, p3), p_i on the edge from v0
            double t[4], u[4];
            for (int i = 1; i < 4; ++i) {
                const double r = recip(k[i] - k[0]);
                t[i] = -k[0] * r;
                u[i] = k[i] * r;
            }
            for (int m = 0; m < M; ++m)
                for (int i = 1; i < 4; ++i) {
                    s[m][i - 1] = v[m][i];
                    s[m][i + 2] = fma(t[i], v[m][i] - v[m][0], v[m][0]);
                }
            w[0] = u[1];
            w[1] = t[1] * u[2];
            w[2] = t[1] * t[2] * u[3];
            count = 3;
        } else if (n == 2) {  // (v2, p20, p21) - (v3, p30, p31)
            const double r20 = recip(k[2] - k[0]), r21 = recip(k[2] - k[1]), r30 = recip(k[3] - k[0]), r31 = recip(k[3] - k[1]);
            const double t20 = k[2] * r20, t21 = k[2] * r21, t30 = k[3] * r30, t31 = k[3] * r31;
            for (int m = 0; m < M; ++m) {
                s[m][0] = v[m][2];
                s[m][1] = fma(t20, v[m][0] - v[m][2], v[m][2]);
                s[m][2] = fma(t21, v[m][1] - v[m][2], v[m][2]);
                s[m][3] = v[m][3];
                s[m][4] = fma(t30, v[m][0] - v[m][3], v[m][3]);
                s[m][5] = fma(t31, v[m][1] - v[m][3], v[m][3]);
            }
            w[0] = t20 * t21;
            w[1] = t30 * (-k[0] * r20) * t21;
            w[2] = (-k[1] * r21) * t30 * t31;
            count = 3;
        } else {  // the corner at v3
            double u[3];
            for (int i = 0; i < 3; ++i) u[i] = k[3] * recip(k[3] - k[i]);
            for (int m = 0; m < M; ++m) {
                s[m][0] = v[m][3];
                for (int i = 0; i < 3; ++i) s[m][i + 1] = fma(u[i], v[m][i] - v[m][3], v[m][3]);
                s[m][4] = s[m][5] = s[m][3];
            }
            w[0] = u[0] * u[1] * u[2];
            count = 1;
        }
    }
    // moves the next piece into points 0..3
    ADECO_HD void advance() {
        for (int m = 0; m < M; ++m)
            for (int i = 0; i < 5; ++i) s[m][i] = s[m][i + 1];
        w[0] = w[1];
        w[1] = w[2];
    }
};

// Share of a piece with heights z[4] in the slab 0 <= z <= 1: 1 minus the parts beyond either plane,
// each computed from the side with fewer vertices.
ADECO_HD double slab_share(const double z[4]) {
    double f = 1.0;
    const double lo = fmin(fmin(z[0], z[1]), fmin(z[2], z[3])), hi = fmax(fmax(z[0], z[1]), fmax(z[2], z[3]));
    if (lo < 0.0) f -= beyond_fraction(-z[0], -z[1], -z[2], -z[3]);
    if (hi > 1.0) f -= beyond_fraction(z[0] - 1.0, z[1] - 1.0, z[2] - 1.0, z[3] - 1.0);
    return f > 0.0 ? f : 0.0;
}

// Share of the tet in the unit cell [0, 1]^3 from non-overlapping pieces: x >= 0, x <= 1, y >= 0,
// y <= 1 in turn, then the z slab; all terms are positive.  keep(i), i < 15, is storage for the points of
// the first cut, so that only the inner cuts' stay in registers.  The work can be shared out: of the 27
// paths (one piece of each of the first three cuts) this call sums those with index `first`,
// `first` + `stride`, ... (stride a power of 2).
template <class Keep>
ADECO_HD double exact_cell_share(const double x[4], const double y[4], const double z[4], Keep keep, int first = 0,
                                 int stride = 1) {
    // whether any of the paths at..at + n - 1 is this call's
    const auto mine = [&](int at, int n) { return ((first - at) & (stride - 1)) < n; };
    int count;
    double p0[3], w0, w1, w2;
    {
        double v[3][4];
        for (int i = 0; i < 4; ++i) {
            v[0][i] = 1.0 - x[i];
            v[1][i] = y[i];
            v[2][i] = z[i];
        }
        PositivePart<3> a;
        a.set(x, v);
        for (int m = 0; m < 3; ++m) {
            p0[m] = a.s[m][0];
            for (int i = 0; i < 5; ++i) keep(3 * i + m) = a.s[m][i + 1];
        }
        count = a.count;
        w0 = a.w[0];
        w1 = a.w[1];
        w2 = a.w[2];
    }
    double sum = 0.0;
    for (int ka = 0;; ++ka) {
        while (ka < count && !mine(9 * ka, 9)) ++ka;
        if (ka >= count) break;
        double k2[4], v2[2][4];
        for (int i = 0; i < 4; ++i) {
            const int at = 3 * (ka + i - 1);
            const bool held = ka == 0 && i == 0;
            k2[i] = held ? p0[0] : keep(held ? 0 : at);
            v2[0][i] = held ? p0[1] : keep(held ? 0 : at + 1);
            v2[1][i] = held ? p0[2] : keep(held ? 0 : at + 2);
        }
        const double wa = ka == 0 ? w0 : (ka == 1 ? w1 : w2);
        PositivePart<2> b;
        b.set(k2, v2);
        for (int kb = 0;; ++kb) {
            for (; kb < b.count && !mine(9 * ka + 3 * kb, 3); ++kb) b.advance();
            if (kb >= b.count) break;
            double v3[2][4];
            for (int i = 0; i < 4; ++i) {
                v3[0][i] = 1.0 - b.s[0][i];
                v3[1][i] = b.s[1][i];
            }
            const double k3[4] = {b.s[0][0], b.s[0][1], b.s[0][2], b.s[0][3]};
            PositivePart<2> c;
            c.set(k3, v3);
            const double wb = wa * b.w[0];
            for (int kc = 0;; ++kc) {
                for (; kc < c.count && !mine(9 * ka + 3 * kb + kc, 1); ++kc) c.advance();
                if (kc >= c.count) break;
                const double v4[1][4] = {{c.s[1][0], c.s[1][1], c.s[1][2], c.s[1][3]}};
                const double k4[4] = {c.s[0][0], c.s[0][1], c.s[0][2], c.s[0][3]};
                PositivePart<1> d;
                d.set(k4, v4);
                const double wc = wb * c.w[0];
                for (int kd = 0; kd < d.count; ++kd) {
                    const double h[4] = {d.s[0][0], d.s[0][1], d.s[0][2], d.s[0][3]};
                    sum += wc * d.w[0] * slab_share(h);
                    d.advance();
                }
                c.advance();
            }
            b.advance();
        }
    }
    return sum;
}

}  // namespace adeco
