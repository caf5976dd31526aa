// How a tet's covered cells are cut into blocks, and what is to be done with each (host and device).
#pragma once

#include "batched_impl.hpp"
#include "block_clip.hpp"

namespace adeco {

// How covered cells are cut into blocks: blocks of b cells, n of them, per axis (x, y, z in the pair's
// order, extents ex <= ey <= ez).  A cover of at most kBlockCells cells is one block; else x keeps up to 2 cells,
// z up to 6 (more where x and y have few) and y what is left, the cells spread evenly over an axis' blocks.
// Large blocks cut fewer faces between blocks, and planes across z cost least.  24 cells are what the LDS of a
// wave holds; against 16 (2 x 2 x 4): 15.3 M pairs on 16^3-cell leaves 4.02 -> 3.71 ms, 6.7 M pairs on
// 32^3-cell leaves 10.9 -> 9.75, a 64^3 request on a 128^3 lattice 515 -> 409 us.
struct BlockShape {
    int b[3], n[3];
};
// Blocks of the largest cover, 1023^3 cells in blocks of 2 x 2 x 6.
constexpr unsigned kMostBlocks = 512u * 512u * 171u;

ADECO_HD BlockShape block_shape(int ex, int ey, int ez) {
    static_assert(kBlockCells == 24, "block sizes");
    const int e[3] = {ex, ey, ez};
    BlockShape s;
    for (int a = 0; a < 3; ++a) {
        s.b[a] = e[a];
        s.n[a] = 1;
    }
    if (ex * ey * ez <= kBlockCells) return s;
    const auto cut = [&](int a, int most) {
        if (e[a] <= most) return;
        const int n = int(udiv_small(unsigned(e[a] + most - 1), unsigned(most)));
        s.b[a] = int(udiv_small(unsigned(e[a] + n - 1), unsigned(n)));
        s.n[a] = int(udiv_small(unsigned(e[a] + s.b[a] - 1), unsigned(s.b[a])));
    };
    cut(0, 2);
    const int xy = s.b[0] * imin(ey, 4);
    cut(2, xy == 1 ? 24 : (xy == 2 ? 12 : (xy == 3 ? 8 : 6)));
    // 24 / (x * z): the quotient is at least 0.02 from the next whole number
    cut(1, int(24.5f * rcp_approx(float(s.b[0] * s.b[2]))));
    return s;
}

// Axis order of a cover, packed in 3 bits: the axis of z and whether x and y are the next two axes in
// cyclic order or the reverse.
ADECO_HD int role_axis(int code, int role) {
    const int za = code & 3, u = za == 2 ? 0 : za + 1, v = u == 2 ? 0 : u + 1;
    const bool swap = code & 4;
    return role == 2 ? za : ((role == 0) != swap ? u : v);
}

template <class T>
ADECO_HD T pick(int a, T v0, T v1, T v2) {
    return a == 0 ? v0 : (a == 1 ? v1 : v2);
}

// The order of the axes for extents e: z the longest (ties: z, then y), x the shorter of the others.
ADECO_HD int role_code(const int e[3]) {
    const int za = e[2] >= e[1] && e[2] >= e[0] ? 2 : (e[1] >= e[0] ? 1 : 0);
    const int u = za == 2 ? 0 : za + 1, w = u == 2 ? 0 : u + 1;
    return za | (pick(w, e[0], e[1], e[2]) < pick(u, e[0], e[1], e[2]) ? 4 : 0);
}

// Covered cells l..h of one axis for a tet between mn and mx (in cells from the grid's face): the cells
// whose box it can strictly overlap, widened by 1e-9 of a cell and kept inside the grid.
ADECO_HD void covered(double mn, double mx, int dims, int& l, int& h) {
    const double top = double(dims - 1);
    l = int(fmax(fmin(floor(mn - 1e-9), top), 0.0));
    h = int(fmax(fmin(floor(mx + 1e-9), top), 0.0));
}

// A tet in the cells of a grid: its cover and its vertices, from the cover's corner and in its axis order.
struct TetCover {
    int lo[3], e[3], code;
    double s[4][3];
};

// The vertices are scaled from the corner, rounded once at their distance from it: a coordinate of 50 cells from the
// grid's face would be off by up to 7e-15 cells, and by the scale's rounding as much again.  Grids against extended
// precision, rms (from the face; from the corner; one tet per thread): 32^3 lattice on 64^3 cells 2.2e-15, 3.8e-16,
// 2.4e-16; 12^3 on 28^3 2.2e-15, 3.6e-16, 1.0e-15; 24^3 on 60^3 1.9e-15, 3.6e-16, 6e-15.
ADECO_HD TetCover cover_of(const V3<double> v[4], const GridDesc& g) {
    double c[4][3];
    int lo[3], e[3];
    for (int a = 0; a < 3; ++a) {
        for (int q = 0; q < 4; ++q) c[q][a] = comp(v[q], a) - g.gmin[a];
        int h;
        covered(g.scale[a] * fmin(fmin(c[0][a], c[1][a]), fmin(c[2][a], c[3][a])),
                g.scale[a] * fmax(fmax(c[0][a], c[1][a]), fmax(c[2][a], c[3][a])), g.dims, lo[a], h);
        e[a] = h - lo[a] + 1;
        for (int q = 0; q < 4; ++q) c[q][a] = fma(c[q][a], g.scale_lo[a], fma(c[q][a], g.scale[a], -double(lo[a])));
    }
    TetCover t;
    t.code = role_code(e);
    for (int r = 0; r < 3; ++r) {
        const int a = role_axis(t.code, r);
        t.lo[r] = pick(a, lo[0], lo[1], lo[2]);
        t.e[r] = pick(a, e[0], e[1], e[2]);
        for (int q = 0; q < 4; ++q) t.s[q][r] = pick(a, c[q][0], c[q][1], c[q][2]);
    }
    return t;
}

// Orients a cover's tet positively in the cover's axis order (the face tests need it); vol: its signed volume, or
// a multiple.
ADECO_HD void orient(TetCover& t, double vol) {
    if ((vol < 0.0) == bool(t.code & 4)) return;
    for (int a = 0; a < 3; ++a) {
        const double s0 = t.s[0][a];
        t.s[0][a] = t.s[3][a];
        t.s[3][a] = s0;
    }
}

// A block of a cover: its corner cell (in the cover's axis order), its sizes, the tet's vertices from the corner,
// the share of the tet in a cell that lies wholly in it (cell volume / tet volume), and what its shares are to
// be multiplied with (shrink_tet).
struct Block {
    int lo[3], c[3];
    double x[4], y[4], z[4];
    double full, scale;
};

// lo, e: the cover's first cell and extents in its axis order; s: the vertices from its corner, in that order.
ADECO_HD Block make_block(const int lo[3], const int e[3], const double s[4][3], double full, unsigned unit) {
    Block b;
    b.full = full;
    b.scale = 1.0;
    const BlockShape sh = block_shape(e[0], e[1], e[2]);
    int i[3] = {0, 0, 0};
    if (unit) {
        const unsigned rest = sh.n[2] == 1 ? unit : udiv_small(unit, unsigned(sh.n[2]));
        i[2] = int(unit - rest * unsigned(sh.n[2]));
        i[0] = sh.n[1] == 1 ? int(rest) : int(udiv_small(rest, unsigned(sh.n[1])));
        i[1] = int(rest) - i[0] * sh.n[1];
    }
    for (int a = 0; a < 3; ++a) {
        b.lo[a] = lo[a] + i[a] * sh.b[a];
        b.c[a] = imin(sh.b[a], e[a] - i[a] * sh.b[a]);
    }
    for (int q = 0; q < 4; ++q) {
        b.x[q] = s[q][0] - double(b.lo[0] - lo[0]);
        b.y[q] = s[q][1] - double(b.lo[1] - lo[1]);
        b.z[q] = s[q][2] - double(b.lo[2] - lo[2]);
    }
    return b;
}

// Cell i of a block as a block of its own.
ADECO_HD Block cell_of(Block b, int i) {
    const int q = int(udiv_small(unsigned(i), unsigned(b.c[2]))), k = i - q * b.c[2];
    const int a = int(udiv_small(unsigned(q), unsigned(b.c[1]))), j = q - a * b.c[1];
    for (int v = 0; v < 4; ++v) {
        b.x[v] -= double(a);
        b.y[v] -= double(j);
        b.z[v] -= double(k);
    }
    b.lo[0] += a;
    b.lo[1] += j;
    b.lo[2] += k;
    b.c[0] = b.c[1] = b.c[2] = 1;
    return b;
}

// Where a block's cells lie: the offset of its first cell and the strides of its axes.
struct Place {
    int64_t corner, sx, sy, sz;
};

ADECO_HD Place place_of(const int lo[3], int code, int dims) {
    const int64_t s1 = dims, s2 = int64_t(dims) * dims;
    Place p;
    p.sx = pick(role_axis(code, 0), int64_t(1), s1, s2);
    p.sy = pick(role_axis(code, 1), int64_t(1), s1, s2);
    p.sz = pick(role_axis(code, 2), int64_t(1), s1, s2);
    p.corner = lo[0] * p.sx + lo[1] * p.sy + lo[2] * p.sz;
    return p;
}

// Visits the cells of a block in the order of its shares: f(index, offset in the grid).
template <class F>
ADECO_HD void for_cells(const int c[3], const Place& p, F f) {
    const int n = c[0] * c[1] * c[2];
    int b = 0, k = 0;
    int64_t at = p.corner;
    const int64_t next_y = p.sy - c[2] * p.sz, next_x = p.sx - c[1] * p.sy;
    for (int i = 0; i < n; ++i) {
        f(i, at);
        at += p.sz;
        if (++k == c[2]) {
            k = 0;
            at += next_y;
            if (++b == c[1]) {
                b = 0;
                at += next_x;
            }
        }
    }
}

// Work class of a block to clip: by the pieces that the x planes leave of the tet (1 for each plane with 1 or 3
// vertices below, else 3), and where they are few by the planes that cut it across y.  The class only groups
// blocks of similar loops (8 classes against 6 by the planes alone: 9.75 -> 9.2 ms for the large tets above,
// 3.71 -> 3.68 for the small ones).  mn, mx: the tet's extents from the block's corner.
ADECO_HD int work_class(const Block& b, const double mn[3], const double mx[3]) {
    const int fx = floor_clamped(mn[0], b.c[0]) + 1, lx = imin(ceil_clamped(mx[0], b.c[0]) - 1, b.c[0]);
    const int fy = floor_clamped(mn[1], b.c[1]) + 1, ly = imin(ceil_clamped(mx[1], b.c[1]) - 1, b.c[1]);
    const int py = ly - fy + 1;
    int pieces = 0;
    for (int p = 0; p <= 2; ++p) {  // (a block has at most 2 cells across x)
        const int n = int(b.x[0] < double(p)) + int(b.x[1] < double(p)) + int(b.x[2] < double(p)) + int(b.x[3] < double(p));
        pieces += p >= fx && p <= lx ? (n == 2 ? 3 : 1) : 0;
    }
    if (pieces <= 1) return 2 * pieces + int(py > pieces);
    if (pieces == 3) return 5 + int(py > 1);
    return pieces == 2 ? 4 : 7;
}

enum BlockClass : int { kBlockEmpty = -1, kBlockTet = -2, kBlockFull = -3 };

// What to do with a block: nothing, deposit the whole tet in its only cell, fill it, or clip it (the work
// class >= 0).  The tet is positively oriented in the block's axis order.
ADECO_HD int classify_block(const Block& b) {
    const double mn[3] = {fmin(fmin(b.x[0], b.x[1]), fmin(b.x[2], b.x[3])), fmin(fmin(b.y[0], b.y[1]), fmin(b.y[2], b.y[3])),
                          fmin(fmin(b.z[0], b.z[1]), fmin(b.z[2], b.z[3]))};
    const double mx[3] = {fmax(fmax(b.x[0], b.x[1]), fmax(b.x[2], b.x[3])), fmax(fmax(b.y[0], b.y[1]), fmax(b.y[2], b.y[3])),
                          fmax(fmax(b.z[0], b.z[1]), fmax(b.z[2], b.z[3]))};
    const double box[3] = {double(b.c[0]), double(b.c[1]), double(b.c[2])};
    bool hit = true, inside = true;
    for (int a = 0; a < 3; ++a) {
        hit = hit && mn[a] < box[a] && 0.0 < mx[a];
        inside = inside && mn[a] >= 0.0 && mx[a] <= box[a];
    }
    if (!hit) return kBlockEmpty;
    if (inside) {
        if (b.c[0] * b.c[1] * b.c[2] == 1) return kBlockTet;
    } else {
        V3<double> s[4];
        for (int q = 0; q < 4; ++q) s[q] = mk(b.x[q], b.y[q], b.z[q]);
        const int cls = classify_margin(s, box);
        if (cls == CLS_NONE) return kBlockEmpty;
        if (cls == CLS_CELL_IN_TET) return kBlockFull;
    }
    return work_class(b, mn, mx);
}

// Replaces a block's tet, where it is large, by a smaller one with the same part in the block: its copy about a
// point that lies on every face plane which cuts the block, shrunk as far as the other planes stay off the block.
// A share is a difference of shares of the whole tet, with their rounding: of a tet of V cells a cell's share
// carries about 3e-16 V of its own size, and cells of less than kNoShare of the tet are lost.  Grids of Kuhn tets
// against extended precision, rms: 27 cells wide 9e-15 (1.1e-13 without the copy, 3.4e-14 one tet per thread), 120
// wide 1.2e-13 (6.6e-12, 4.7e-13), 1000 wide 6e-15 (5e-9, 1.3e-13).  It costs little, as only blocks of large tets
// run it: 97^3 lattice in 32^3-cell leaves 9.3 -> 9.6 ms, 9^3 cubes on 90^3 cells 1.12 -> 1.20.
// The tet is positively oriented in the block's axis order.
ADECO_HD void shrink_tet(Block& b) {
    if (!(b.full < kLargeTet) || b.full < kVastTet) return;
    V3<double> s[4];
    for (int q = 0; q < 4; ++q) s[q] = mk(b.x[q], b.y[q], b.z[q]);
    const V3<double> e01 = sub(s[1], s[0]), e02 = sub(s[2], s[0]), e03 = sub(s[3], s[0]);
    const V3<double> n[4] = {cross(sub(s[3], s[1]), sub(s[2], s[1])), cross(e02, e03), cross(e03, e01), cross(e01, e02)};  // by opposite vertex
    const V3<double> r = mk(double(b.c[0]), double(b.c[1]), double(b.c[2])), mid = mk(0.5 * r.x, 0.5 * r.y, 0.5 * r.z);
    // a plane's value at p is v - n.p, positive inside; least: its least in the block
    double v[4], least[4];
    int keep = 0;  // planes that the point has to lie on
    for (int f = 0; f < 4; ++f) {
        const V3<double>& o = s[f == 0 ? 1 : 0];
        v[f] = n[f].x * o.x + n[f].y * o.y + n[f].z * o.z;
        least[f] = v[f] - (fmax(n[f].x * r.x, 0.0) + fmax(n[f].y * r.y, 0.0) + fmax(n[f].z * r.z, 0.0));
        const double sum = fabs(n[f].x) + fabs(n[f].y) + fabs(n[f].z);
        if (!(least[f] > 1e-3 * sum)) keep |= 1 << f;
    }
    double best = 1.0;
    V3<double> about = mid;
    for (int tries = 0; tries < 4 && keep != 15; ++tries) {
        V3<double> p = mid;
        const bool k0 = keep & 1, k1 = keep & 2, k2 = keep & 4, k3 = keep & 8;
        const int kept = int(k0) + int(k1) + int(k2) + int(k3);
        if (kept == 1) {
            // the centre's foot on the plane
            const V3<double> m = k0 ? n[0] : (k1 ? n[1] : (k2 ? n[2] : n[3]));
            const double at = k0 ? v[0] : (k1 ? v[1] : (k2 ? v[2] : v[3]));
            const double t = (at - (m.x * p.x + m.y * p.y + m.z * p.z)) * recip(m.x * m.x + m.y * m.y + m.z * m.z);
            p = mk(fma(t, m.x, p.x), fma(t, m.y, p.y), fma(t, m.z, p.z));
        } else if (kept >= 2) {
            // the edge of two planes (its point closest to the centre), the vertex of three
            const V3<double> u = !k0 ? s[0] : (!k1 ? s[1] : (!k2 ? s[2] : s[3]));
            const V3<double> w = !k3 ? s[3] : (!k2 ? s[2] : s[1]);
            const V3<double> d = sub(w, u), to = sub(p, u);
            const double dd = d.x * d.x + d.y * d.y + d.z * d.z;
            const double t = kept == 2 ? fmax(fmin((to.x * d.x + to.y * d.y + to.z * d.z) * recip(dd), 1.0), 0.0) : 0.0;
            p = mk(fma(t, d.x, u.x), fma(t, d.y, u.y), fma(t, d.z, u.z));
        }
        double ratio = 1.0 / 1024.0;
        int by = 0;
        for (int f = 0; f < 4; ++f) {
            const double at = v[f] - (n[f].x * p.x + n[f].y * p.y + n[f].z * p.z);
            const double q = (keep >> f) & 1 || !(at > 0.0) ? 0.0 : fma(-0.9375 * least[f], recip(at), 1.0);
            by = q > ratio ? 1 << f : by;
            ratio = fmax(ratio, q);
        }
        if (ratio < best) {
            best = ratio;
            about = p;
        }
        // still large, near another plane: on that one, too
        if (ratio * ratio * ratio < 128.0 * b.full || kept == 3) break;
        keep |= by;
    }
    if (best > 0.875) return;
    for (int q = 0; q < 4; ++q) {
        b.x[q] = fma(best, b.x[q] - about.x, about.x);
        b.y[q] = fma(best, b.y[q] - about.y, about.y);
        b.z[q] = fma(best, b.z[q] - about.z, about.z);
    }
    b.scale = best * best * best;
    b.full *= recip(b.scale);
}

}  // namespace adeco
