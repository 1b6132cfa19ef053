// Structured material sampling on the device: the cell-averaged values of
// z-stacked primitives at one Yee offset (StructuredMaterial3D, the C++
// class of src/Grid.cpp:736-874 behind emopt/grid.py:874-961), computed with
// exactly the arithmetic of the host sampler in emopt_amd/grid.py -- same
// points, same operation order, no fused multiply-adds -- so the two give
// identical doubles.
//
//   value(i, j, k) = sum over z segments s of fz(i, s) * v(s, j, k)
//                    + (1 - sum fz) * background
//   v(s, j, k)     = the in-plane average of the primitives active in
//                    segment s, by one of two rules:
//
// ss == 0, the reference's rule (src/Grid.cpp:460-525), spelled out above
// mat_within: corner-gated primitives each taking the exact area of what is
// left of the cell.
//
// ss > 0, supersampled: each primitive in priority order takes
// min(coverage, remaining), the rest is background.  Rectangle coverage is the
// exact overlap of the cell with the rectangle; ellipse and polygon coverage
// is the fraction of ss x ss sample points inside (cells outside the
// primitive's bounding box: 0).
#pragma once
#include "kernels.hpp"

namespace emf {

struct MatPrim {
    int kind;                 // 0 rectangle, 1 ellipse, 2 polygon
    int clip;                 // ellipse clipped to q[6..9]
    int v0, nv;               // polygon vertices
    double re, im;
    double z1, z2;
    double bbox[4];           // xmin, xmax, ymin, ymax
    double q[10];             // ellipse: x0, y0, a, b, cos, sin, clip box
};

__device__ inline bool mat_inside(const MatPrim &p, const double *__restrict__ vx,
                                  const double *__restrict__ vy, double x, double y)
{
#pragma clang fp contract(off)
    if (p.kind == 1) {
        const double c = p.q[4], s = p.q[5];
        const double u = (x - p.q[0]) * c + (y - p.q[1]) * s;
        const double v = -(x - p.q[0]) * s + (y - p.q[1]) * c;
        const double ua = u / p.q[2], vb = v / p.q[3];
        bool in = ua * ua + vb * vb <= 1.0;
        if (p.clip) in = in && x >= p.q[6] && x < p.q[7] && y >= p.q[8] && y < p.q[9];
        return in;
    }
    bool res = false;   // polygon, even-odd rule
    for (int a = 0; a < p.nv; ++a) {
        const int b = a + 1 < p.nv ? a + 1 : 0;
        const double xa = vx[p.v0 + a], ya = vy[p.v0 + a];
        const double xb = vx[p.v0 + b], yb = vy[p.v0 + b];
        if (ya == yb) continue;
        const bool cond = (ya > y) != (yb > y);
        const double xint = xa + (y - ya) * (xb - xa) / (yb - ya);
        res = res != (cond && x < xint);
    }
    return res;
}

__device__ inline double mat_coverage(const MatPrim &p, const double *__restrict__ vx,
                                      const double *__restrict__ vy, double xc, double yc,
                                      double dx, double dy, int ss)
{
#pragma clang fp contract(off)
    const double hx = dx / 2, hy = dy / 2;
    if (p.kind == 0) {
        const double fx = fmax(fmin(xc + hx, p.bbox[1]) - fmax(xc - hx, p.bbox[0]), 0.0) / dx;
        const double fy = fmax(fmin(yc + hy, p.bbox[3]) - fmax(yc - hy, p.bbox[2]), 0.0) / dy;
        return fy * fx;
    }
    if (!(xc + hx > p.bbox[0] && xc - hx < p.bbox[1] && yc + hy > p.bbox[2] && yc - hy < p.bbox[3]))
        return 0.0;
    int count = 0;
    for (int a = 0; a < ss; ++a) {
        const double y = yc + (((double)a + 0.5) / ss - 0.5) * dy;
        for (int b = 0; b < ss; ++b) {
            const double x = xc + (((double)b + 0.5) / ss - 0.5) * dx;
            count += mat_inside(p, vx, vy, x, y) ? 1 : 0;
        }
    }
    return (double)count / (double)(ss * ss);
}

// ---------------------------------------------------------------------------
// The reference's overlap rule (src/Grid.cpp:460-525 with GridCell::intersect,
// src/Grid.cpp:74-108).  Per cell, primitives in priority order:
//   * a primitive counts only when one of the four cell corners lies strictly
//     inside it (Rectangle::contains_point, src/Grid.cpp:219-225; Polygon via
//     boost::geometry::within, src/Grid.cpp:362-374: boundary points are out);
//   * all four corners inside and nothing of the cell taken yet: the cell is
//     the primitive's value;
//   * otherwise the primitive takes the part of the cell not yet taken that
//     it covers, exactly (boost::geometry::difference there);
//   * the cell stops when nothing is left; what is left is background.
// The taken part is the cell intersected with the union of the primitives
// that counted so far, so each overlap is the growth of that union's area.
// Rectangles are the polygon ring of src/Grid.cpp:204-213.  The reference
// clips in __float128 (src/Grid.hpp:22); this is double precision.
// ---------------------------------------------------------------------------
constexpr int MAT_MAXU = 8;     // primitives counted in one cell
constexpr int MAT_MAXE = 48;    // polygon edges through one cell
constexpr int MAT_MAXB = 256;   // x breakpoints in one cell

struct MatEdge {
    double x1, y1, x2, y2;
    int q;                      // which counted primitive
};

__device__ inline int mat_nvert(const MatPrim &p) { return p.kind == 0 ? 4 : p.nv; }

__device__ inline void mat_vertex(const MatPrim &p, const double *__restrict__ vx,
                                  const double *__restrict__ vy, int a, double &x, double &y)
{
    if (p.kind == 0) {
        x = a < 2 ? p.bbox[0] : p.bbox[1];
        y = (a == 0 || a == 3) ? p.bbox[2] : p.bbox[3];
    } else {
        x = vx[p.v0 + a];
        y = vy[p.v0 + a];
    }
}

// Strictly inside (a point on the boundary is not).  The wave's lanes take the
// edges; the answer is the whole wave's.
__device__ inline bool mat_within(const MatPrim &p, const double *__restrict__ vx,
                                  const double *__restrict__ vy, double x, double y, int lane)
{
#pragma clang fp contract(off)
    if (!(x > p.bbox[0] && x < p.bbox[1] && y > p.bbox[2] && y < p.bbox[3])) return false;
    if (p.kind == 0) return true;
    bool on = false;
    int odd = 0;
    for (int a0 = 0; a0 < p.nv; a0 += 64) {
        const int a = a0 + lane, b = a + 1 < p.nv ? a + 1 : 0;
        bool edge = false, cross = false;
        if (a < p.nv) {
            const double xa = vx[p.v0 + a], ya = vy[p.v0 + a];
            const double xb = vx[p.v0 + b], yb = vy[p.v0 + b];
            edge = (xb - xa) * (y - ya) - (yb - ya) * (x - xa) == 0.0 && x >= fmin(xa, xb) &&
                   x <= fmax(xa, xb) && y >= fmin(ya, yb) && y <= fmax(ya, yb);
            if ((ya > y) != (yb > y)) cross = x < xa + (y - ya) * (xb - xa) / (yb - ya);
        }
        on = on || __ballot(edge) != 0;
        odd ^= __popcll(__ballot(cross)) & 1;
    }
    return !on && odd;
}

// One cell's lists, in LDS.
struct MatCell {
    MatEdge e[MAT_MAXE];
    double bx[MAT_MAXB], sx[MAT_MAXB];   // breakpoints as found (then slab areas), sorted
    unsigned in[MAT_MAXB];               // per slab: primitives its midpoint is inside at y = ya
};

// Area of [xa, xb] x [ya, yb] inside the union of the primitives u[0..nu).
// Between consecutive x breakpoints (ends of the edges through the cell,
// their crossings of y = ya and y = yb, crossings of edges of different
// primitives inside the cell) the covered length of a vertical line is linear
// in x, so each slab contributes its width times the covered length at its
// midpoint.  Only edges through the cell are kept; whether the midpoint line
// enters the cell inside a primitive is the parity of that primitive's edges
// crossing it at or below ya, counted over all its edges (it can only change
// where a kept edge crosses y = ya, a breakpoint).  err is set when a cell
// exceeds the fixed limits above.
//
// The lanes of one wave take the edges, then the pairs of edges, then the
// slabs; the slabs' areas are added in order, so the sum is the host's.
__device__ inline double mat_union_area(const MatPrim *__restrict__ prims,
                                        const double *__restrict__ vx,
                                        const double *__restrict__ vy, MatCell &L, const int *u,
                                        int nu, double xa, double xb, double ya, double yb,
                                        int lane, bool &err)
{
#pragma clang fp contract(off)
    const unsigned long long below = (1ULL << lane) - 1;
    __syncthreads();                    // the lists of the last call are done with
    int ne = 0;
    for (int s = 0; s < nu; ++s) {
        const MatPrim &p = prims[u[s]];
        const int nv = mat_nvert(p);
        for (int a0 = 0; a0 < nv; a0 += 64) {
            const int a = a0 + lane;
            double x1 = 0, y1 = 0, x2 = 0, y2 = 0;
            bool keep = a < nv;
            if (keep) {
                mat_vertex(p, vx, vy, a, x1, y1);
                mat_vertex(p, vx, vy, a + 1 < nv ? a + 1 : 0, x2, y2);
                keep = !(fmax(x1, x2) <= xa || fmin(x1, x2) >= xb || fmax(y1, y2) <= ya ||
                         fmin(y1, y2) >= yb);
            }
            const unsigned long long m = __ballot(keep);
            const int at = ne + __popcll(m & below);
            if (keep && at < MAT_MAXE) L.e[at] = MatEdge{ x1, y1, x2, y2, s };
            ne += __popcll(m);
        }
    }
    if (ne > MAT_MAXE) { err = true; return 0.0; }
    static_assert(MAT_MAXE <= 64, "a lane per edge");
    int nb = 2;
    if (lane < 2) L.bx[lane] = lane ? xb : xa;
    auto push = [&](bool want, double x) {
        want = want && x > xa && x < xb;
        const unsigned long long m = __ballot(want);
        const int at = nb + __popcll(m & below);
        if (want && at < MAT_MAXB) L.bx[at] = x;
        nb += __popcll(m);
    };
    __syncthreads();
    const MatEdge h = L.e[lane < ne ? lane : 0];
    push(lane < ne, h.x1);
    push(lane < ne, h.x2);
    push(lane < ne && (h.y1 > ya) != (h.y2 > ya), h.x1 + (ya - h.y1) * (h.x2 - h.x1) / (h.y2 - h.y1));
    push(lane < ne && (h.y1 > yb) != (h.y2 > yb), h.x1 + (yb - h.y1) * (h.x2 - h.x1) / (h.y2 - h.y1));
    if (nu > 1)
        for (int i = 0; i + 1 < ne; ++i) {
            const MatEdge f = L.e[i];
            double x = 0;
            bool want = lane > i && lane < ne && f.q != h.q;
            if (want) {
                const double d = (f.x2 - f.x1) * (h.y2 - h.y1) - (f.y2 - f.y1) * (h.x2 - h.x1);
                want = d != 0.0;
                const double t = ((h.x1 - f.x1) * (h.y2 - h.y1) - (h.y1 - f.y1) * (h.x2 - h.x1)) / d;
                const double r = ((h.x1 - f.x1) * (f.y2 - f.y1) - (h.y1 - f.y1) * (f.x2 - f.x1)) / d;
                want = want && t > 0.0 && t < 1.0 && r > 0.0 && r < 1.0;
                const double y = f.y1 + t * (f.y2 - f.y1);
                want = want && y > ya && y < yb;
                x = f.x1 + t * (f.x2 - f.x1);
            }
            push(want, x);
        }
    if (nb > MAT_MAXB) { err = true; return 0.0; }
    __syncthreads();
    for (int b = lane; b < nb; b += 64) {       // each breakpoint counts those before it
        const double v = L.bx[b];
        int r = 0;
        for (int c = 0; c < nb; ++c) r += L.bx[c] < v || (L.bx[c] == v && c < b);
        L.sx[r] = v;
        L.in[b] = 0;
    }
    __syncthreads();
    for (int s = 0; s < nu; ++s) {
        const MatPrim &p = prims[u[s]];
        const int nv = mat_nvert(p);
        for (int a0 = 0; a0 < nv; a0 += 64) {
            const int a = a0 + lane;
            double x1 = 0, y1 = 0, x2 = 0, y2 = 0;
            if (a < nv) {
                mat_vertex(p, vx, vy, a, x1, y1);
                mat_vertex(p, vx, vy, a + 1 < nv ? a + 1 : 0, x2, y2);
            }
            const double lo = fmin(x1, x2), hi = fmax(x1, x2);
            if (!__ballot(a < nv && lo < xb && hi > xa)) continue;
            for (int b = 0; b + 1 < nb; ++b) {
                const double xm = 0.5 * (L.sx[b] + L.sx[b + 1]);
                const bool under = a < nv && lo < xm && hi > xm &&
                                   y1 + (xm - x1) * (y2 - y1) / (x2 - x1) <= ya;
                if ((__popcll(__ballot(under)) & 1) && lane == 0) L.in[b] ^= 1u << s;
            }
        }
    }
    __syncthreads();
    for (int b = lane; b + 1 < nb; b += 64) {
        const double w = L.sx[b + 1] - L.sx[b];
        double part = 0.0;
        if (w > 0.0) {
            const double xm = 0.5 * (L.sx[b] + L.sx[b + 1]);
            unsigned in = L.in[b];
            double len = 0.0, yp = ya;
            for (int last = -1;;) {             // the edges the line crosses, from below
                double yn = 0.0;
                int next = -1;
                for (int i = 0; i < ne; ++i) {
                    const MatEdge &f = L.e[i];
                    if (!(fmin(f.x1, f.x2) < xm && fmax(f.x1, f.x2) > xm)) continue;
                    const double y = f.y1 + (xm - f.x1) * (f.y2 - f.y1) / (f.x2 - f.x1);
                    if (!(y > ya && y < yb)) continue;
                    if (last >= 0 && !(y > yp || (y == yp && i > last))) continue;
                    if (next < 0 || y < yn) { yn = y; next = i; }
                }
                if (next < 0) break;
                if (in) len += yn - yp;
                yp = yn;
                in ^= 1u << L.e[next].q;
                last = next;
            }
            if (in) len += yb - yp;
            part = w * len;
        }
        L.bx[b] = part;
    }
    __syncthreads();
    double area = 0.0;
    for (int b = 0; b + 1 < nb; ++b) area += L.bx[b];
    return area;
}

// v(s, j, k) for the used segments by the reference's rule above (rectangles
// and polygons only): v2[(s * nj + jj) * nk + kk].  One wave per cell; its
// lanes first take the primitives (64 bounding boxes at a time), then the edges
// of those whose box holds a corner.  Bound by the serial chain of the cells on
// the boundaries, a few thousand of them: a thread per cell took 8.5 ms for
// 240x120 cells of 40 polygons, the slowest cell's time, with its lists in
// scratch memory.
__global__ __launch_bounds__(64) void k_mat_exact(
    const MatPrim *__restrict__ prims, const double *__restrict__ vx, const double *__restrict__ vy,
    const int *__restrict__ seg_off, const int *__restrict__ seg_prim, int nseg, int k1, int nk,
    int j1, int nj, double sx, double sy, double dx, double dy, double bg_re, double bg_im,
    double2 *__restrict__ v2, int *__restrict__ err)
{
#pragma clang fp contract(off)
    __shared__ MatCell L;
    __shared__ int u[MAT_MAXU];
    const int lane = (int)threadIdx.x;
    const long long total = (long long)nseg * nj * nk;
    for (long long g = blockIdx.x; g < total; g += gridDim.x) {
        const int kk = (int)(g % nk), jj = (int)((g / nk) % nj), s = (int)(g / ((long long)nk * nj));
        const double xc = ((double)(k1 + kk) + sx) * dx;
        const double yc = ((double)(j1 + jj) + sy) * dy;
        const double xa = xc - dx / 2, xb = xc + dx / 2, ya = yc - dy / 2, yb = yc + dy / 2;
        const double A = (xb - xa) * (yb - ya);
        double vr = 0.0, vi = 0.0, rem = A;
        int nu = 0;
        bool full = false, bad = false, done = false;
        for (int q0 = seg_off[s]; q0 < seg_off[s + 1] && !done; q0 += 64) {
            const int q = q0 + lane;
            int mine = 0;
            bool near = q < seg_off[s + 1];
            if (near) {
                mine = seg_prim[q];
                const double *b = prims[mine].bbox;
                near = ((xa > b[0] && xa < b[1]) || (xb > b[0] && xb < b[1])) &&
                       ((ya > b[2] && ya < b[3]) || (yb > b[2] && yb < b[3]));
            }
            for (unsigned long long m = __ballot(near); m && !done; m &= m - 1) {
                const int pi = __builtin_amdgcn_readlane(mine, __ffsll((long long)m) - 1);
                const MatPrim &p = prims[pi];
                const bool c1 = mat_within(p, vx, vy, xa, ya, lane);
                const bool c2 = mat_within(p, vx, vy, xb, ya, lane);
                const bool c3 = mat_within(p, vx, vy, xb, yb, lane);
                const bool c4 = mat_within(p, vx, vy, xa, yb, lane);
                if (c1 && c2 && c3 && c4 && rem == A) {
                    vr = p.re;
                    vi = p.im;
                    full = done = true;
                    continue;
                }
                if (c1 || c2 || c3 || c4) {
                    if (nu == MAT_MAXU) { bad = done = true; continue; }
                    if (lane == 0) u[nu] = pi;
                    ++nu;
                    double rn = A - mat_union_area(prims, vx, vy, L, u, nu, xa, xb, ya, yb, lane, bad);
                    if (rn <= A * 1e-13) rn = 0.0;   // fully taken (an empty difference there)
                    const double ov = (rem - rn) / A;
                    vr += ov * p.re;
                    vi += ov * p.im;
                    rem = rn;
                    done = bad || rem == 0.0;
                }
            }
        }
        if (bad && lane == 0) *err = 1;
        if (!full && rem > 0.0) {
            const double r = rem / A;
            vr += r * bg_re;
            vi += r * bg_im;
        }
        if (lane == 0) v2[g] = make_double2(vr, vi);
        __syncthreads();
    }
}

// v(s, j, k) by supersampled coverage, a thread per cell: each primitive takes
// at most what is left of the cell.
__global__ void k_mat_inplane(const MatPrim *__restrict__ prims, const double *__restrict__ vx,
                              const double *__restrict__ vy, const int *__restrict__ seg_off,
                              const int *__restrict__ seg_prim, int nseg, int k1, int nk, int j1,
                              int nj, double sx, double sy, double dx, double dy, int ss,
                              double bg_re, double bg_im, double2 *__restrict__ v2)
{
#pragma clang fp contract(off)
    const long long total = (long long)nseg * nj * nk;
    for (long long g = blockIdx.x * (long long)blockDim.x + threadIdx.x; g < total;
         g += (long long)gridDim.x * blockDim.x) {
        const int kk = (int)(g % nk), jj = (int)((g / nk) % nj), s = (int)(g / ((long long)nk * nj));
        const double xc = ((double)(k1 + kk) + sx) * dx;
        const double yc = ((double)(j1 + jj) + sy) * dy;
        double vr = 0.0, vi = 0.0, rem = 1.0;
        for (int q = seg_off[s]; q < seg_off[s + 1]; ++q) {
            const MatPrim &p = prims[seg_prim[q]];
            const double cov = fmin(mat_coverage(p, vx, vy, xc, yc, dx, dy, ss), rem);
            vr += cov * p.re;
            vi += cov * p.im;
            rem -= cov;
        }
        vr += rem * bg_re;
        vi += rem * bg_im;
        v2[g] = make_double2(vr, vi);
    }
}

// out[(ii * nj + jj) * nk + kk] = sum_s fz * v(s) + (1 - sum fz) * background
__global__ void k_mat_combine(const double2 *__restrict__ v2, const double *__restrict__ zab,
                              int nseg, int i1, int ni, int nj, int nk, double sz, double dz,
                              double bg_re, double bg_im, double2 *__restrict__ out)
{
#pragma clang fp contract(off)
    const long long total = (long long)ni * nj * nk;
    const long long plane = (long long)nj * nk;
    for (long long g = blockIdx.x * (long long)blockDim.x + threadIdx.x; g < total;
         g += (long long)gridDim.x * blockDim.x) {
        const int ii = (int)(g / plane);
        const long long jk = g % plane;
        const double zc = ((double)(i1 + ii) + sz) * dz;
        const double zlo = zc - dz / 2, zhi = zc + dz / 2;
        double orr = 0.0, oi = 0.0, covered = 0.0;
        for (int s = 0; s < nseg; ++s) {
            const double fz = fmax(fmin(zhi, zab[2 * s + 1]) - fmax(zlo, zab[2 * s]), 0.0) / dz;
            if (fz > 0) {
                const double2 v = v2[s * plane + jk];
                orr += fz * v.x;
                oi += fz * v.y;
            }
            covered += fz;
        }
        orr += (1.0 - covered) * bg_re;
        oi += (1.0 - covered) * bg_im;
        out[g] = make_double2(orr, oi);
    }
}

// ------------------------------------------- index of distinct eps triples
//
// The E pass reads a 2- or 4-byte index per cell into a table of the distinct
// real (eps_x, eps_y, eps_z).  The index is built on the device, where the
// arrays are: an open-addressing table whose slots hold the number of the
// first cell seen with a triple, so a slot is one compare-and-swap and the
// triples themselves are compared in the eps arrays.  Runs of equal cells are
// the common case: only the first cell of a run within a wave probes, the
// others take its slot.
//
// Memory-bound: 48 B read and 4 B written per cell, then 4 B read and 2 B
// written.  240x120x80 with 40 ellipses: 64 us to find, 54 us to number (4 M
// slots), 6 us to write, where the host's hash map took 20 ms and more.
constexpr unsigned IDX_EMPTY = 0xFFFFFFFFu;
constexpr int IDX_LIMIT = 1 << 20;    // distinct triples; more: no index

struct EpsBits {
    unsigned long long a, b, c;
};

__device__ __forceinline__ EpsBits eps_bits(const double2 *ex, const double2 *ey, const double2 *ez,
                                            long long g)
{
    EpsBits k;
    k.a = (unsigned long long)__double_as_longlong(ex[g].x);
    k.b = (unsigned long long)__double_as_longlong(ey[g].x);
    k.c = (unsigned long long)__double_as_longlong(ez[g].x);
    return k;
}

__device__ __forceinline__ bool same_bits(const EpsBits &x, const EpsBits &y)
{
    return x.a == y.a && x.b == y.b && x.c == y.c;
}

// head[0]: distinct triples found.  table: mask + 1 slots, IDX_EMPTY at first.
__global__ void k_idx_find(const double2 *__restrict__ ex, const double2 *__restrict__ ey,
                           const double2 *__restrict__ ez, long long n, unsigned *table,
                           unsigned mask, unsigned *head, unsigned *__restrict__ slot)
{
    const long long step = (long long)gridDim.x * blockDim.x;
    const int lane = (int)(threadIdx.x & 63);
    // whole waves take part in the shuffles: the bound is rounded up to a wave
    for (long long g = blockIdx.x * (long long)blockDim.x + threadIdx.x; g < ((n + 63) & ~63LL); g += step) {
        const bool in = g < n;
        EpsBits k{ 0, 0, 0 };
        if (in) k = eps_bits(ex, ey, ez, g);
        EpsBits l;
        l.a = __shfl_up(k.a, 1); l.b = __shfl_up(k.b, 1); l.c = __shfl_up(k.c, 1);
        const bool first = in && (lane == 0 || !same_bits(k, l));
        unsigned at = 0;
        if (first) {
            unsigned long long h = k.a * 0x9E3779B97F4A7C15ULL;
            h ^= k.b + 0x9E3779B97F4A7C15ULL + (h << 6) + (h >> 2);
            h ^= k.c + 0x9E3779B97F4A7C15ULL + (h << 6) + (h >> 2);
            h ^= h >> 32;
            at = (unsigned)h & mask;
            for (unsigned tries = 0; tries <= mask; ++tries, at = (at + 1) & mask) {
                unsigned rep = __hip_atomic_load(table + at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (rep == IDX_EMPTY) {
                    rep = atomicCAS(table + at, IDX_EMPTY, (unsigned)g);
                    if (rep == IDX_EMPTY) {
                        atomicAdd(head, 1u);
                        break;
                    }
                }
                if (same_bits(k, eps_bits(ex, ey, ez, rep))) break;
                // too many triples: the result is not used
                if (__hip_atomic_load(head, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) > (unsigned)IDX_LIMIT)
                    break;
            }
        }
        const unsigned long long heads = __ballot(first);
        const unsigned long long upto = heads & (~0ULL >> (63 - lane));
        const unsigned got = __shfl(at, upto ? 63 - __clzll((long long)upto) : 0);
        if (in) slot[g] = got;
    }
}

// Numbers the occupied slots (in no particular order) in place and writes their triples.
__global__ void k_idx_number(const double2 *__restrict__ ex, const double2 *__restrict__ ey,
                             const double2 *__restrict__ ez, unsigned *table, unsigned slots,
                             unsigned *next, double *__restrict__ tab)
{
    for (unsigned q = blockIdx.x * blockDim.x + threadIdx.x; q < slots; q += gridDim.x * blockDim.x) {
        const unsigned rep = table[q];
        if (rep == IDX_EMPTY) continue;
        const unsigned id = atomicAdd(next, 1u);
        tab[3 * id] = ex[rep].x;
        tab[3 * id + 1] = ey[rep].x;
        tab[3 * id + 2] = ez[rep].x;
        table[q] = id;
    }
}

template <typename T>
__global__ void k_idx_write(const unsigned *__restrict__ slot, const unsigned *__restrict__ table,
                            long long n, T *__restrict__ idx)
{
    for (long long g = blockIdx.x * (long long)blockDim.x + threadIdx.x; g < n;
         g += (long long)gridDim.x * blockDim.x)
        idx[g] = (T)table[slot[g]];
}

__global__ void k_fill_u32(unsigned *a, long long n, unsigned v)
{
    for (long long g = blockIdx.x * (long long)blockDim.x + threadIdx.x; g < n;
         g += (long long)gridDim.x * blockDim.x)
        a[g] = v;
}

}  // namespace emf
