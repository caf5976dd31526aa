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

// A tet in the cells of a grid: its cover and its vertices, in the cover's axis order.
struct TetCover {
    int lo[3], e[3], code;
    double s[4][3];
};

ADECO_HD TetCover cover_of(const V3<double> v[4], const GridDesc& g) {
    double c[4][3];
    int lo[3], e[3];
    for (int a = 0; a < 3; ++a) {
        for (int q = 0; q < 4; ++q) c[q][a] = g.scale[a] * (comp(v[q], a) - g.gmin[a]);
        int h;
        covered(fmin(fmin(c[0][a], c[1][a]), fmin(c[2][a], c[3][a])), fmax(fmax(c[0][a], c[1][a]), fmax(c[2][a], c[3][a])), g.dims,
                lo[a], h);
        e[a] = h - lo[a] + 1;
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

// A block of a cover: its corner cell (in the cover's axis order), its sizes and the tet's vertices from
// the corner.
struct Block {
    int lo[3], c[3];
    double x[4], y[4], z[4];
};

// lo, e: the cover's first cell and extents in its axis order; s: the vertices in cells, in that order.
ADECO_HD Block make_block(const int lo[3], const int e[3], const double s[4][3], unsigned unit) {
    Block b;
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
        b.x[q] = s[q][0] - double(b.lo[0]);
        b.y[q] = s[q][1] - double(b.lo[1]);
        b.z[q] = s[q][2] - double(b.lo[2]);
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

}  // namespace adeco
