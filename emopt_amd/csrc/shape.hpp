// Analytic derivatives of structured-material cells on the device: the host
// rule of emopt_amd/shape.py operation for operation (no fused multiply-adds),
// so the two give the same doubles.
#pragma once
#include "material.hpp"

namespace emf {

// A moving edge: P0, P1, its length and the normal velocity at either end.
struct ShapeEdge {
    double x0, y0, x1, y1, len, w0, w1;
};

// Cells of one component: [k1, k1 + nk) x [j1, j1 + nj) in every segment,
// results from `off`, in-cell offset (sx, sy).
struct ShapeBox {
    long long off;
    int k1, nk, j1, nj;
    double sx, sy;
};

struct ShapeArgs {
    const MatPrim *prims;
    const double *vx, *vy;
    const int *seg_off, *seg_prim, *seg_p;    // rings of a segment in priority order; the moving one's place
    const ShapeEdge *edges;
    int nseg, nedges;
    ShapeBox box[3];
    double dx, dy, bg_re, bg_im;
};

// d(in-plane value)/dp, a wave per cell: its lanes take the primitives, then the
// edges of those near, as in k_mat_exact.  A few thousand cells at most, so
// the time is one cell's chain; err is set when a cell counts more than
// MAT_MAXU primitives.  16 parameters of a 180x60x80 grating, about 1600 cells
// each: 8 us a launch, 75 us a call with its copies, where the host loop took
// 4 ms.
__global__ __launch_bounds__(64) void k_shape_deps(ShapeArgs A, long long total,
                                                   double2 *__restrict__ out, int *__restrict__ err)
{
#pragma clang fp contract(off)
    __shared__ int u[MAT_MAXU];          // counted primitives, by their place in the segment
    const int lane = (int)threadIdx.x;
    for (long long g = blockIdx.x; g < total; g += gridDim.x) {
        const int c = g >= A.box[2].off ? 2 : (g >= A.box[1].off ? 1 : 0);
        const ShapeBox B = c == 2 ? A.box[2] : (c == 1 ? A.box[1] : A.box[0]);
        const long long r = g - B.off;
        const int kk = (int)(r % B.nk), jj = (int)((r / B.nk) % B.nj), s = (int)(r / ((long long)B.nk * B.nj));
        const double xc = ((double)(B.k1 + kk) + B.sx) * A.dx, yc = ((double)(B.j1 + jj) + B.sy) * A.dy;
        const double xa = xc - A.dx / 2, xb = xc + A.dx / 2, ya = yc - A.dy / 2, yb = yc + A.dy / 2;
        const int p0 = A.seg_off[s], np = A.seg_off[s + 1] - p0, mine = A.seg_p[s];
        int nu = 0;
        bool counted = false, none = false;
        __syncthreads();
        for (int q0 = 0; q0 < np && !none; q0 += 64) {
            bool near = q0 + lane < np;
            if (near) {
                const double *b = A.prims[A.seg_prim[p0 + q0 + lane]].bbox;
                near = ((xa > b[0] && xa < b[1]) || (xb > b[0] && xb < b[1])) &&
                       ((ya > b[2] && ya < b[3]) || (yb > b[2] && yb < b[3]));
            }
            for (unsigned long long m = __ballot(near); m && !none; m &= m - 1) {
                const int q = q0 + __ffsll((long long)m) - 1;
                const MatPrim &p = A.prims[A.seg_prim[p0 + q]];
                const bool c1 = mat_within(p, A.vx, A.vy, xa, ya, lane);
                const bool c2 = mat_within(p, A.vx, A.vy, xb, ya, lane);
                const bool c3 = mat_within(p, A.vx, A.vy, xb, yb, lane);
                const bool c4 = mat_within(p, A.vx, A.vy, xa, yb, lane);
                if (!(c1 || c2 || c3 || c4)) continue;
                if (nu == 0 && c1 && c2 && c3 && c4) { none = true; continue; }   // its value outright
                if (nu == MAT_MAXU) {
                    if (lane == 0) *err = 1;
                    none = true;
                    continue;
                }
                if (lane == 0) u[nu] = q;
                ++nu;
                counted = counted || q == mine;
            }
        }
        __syncthreads();
        double tr = 0.0, ti = 0.0;
        const MatPrim &P = A.prims[A.seg_prim[p0 + mine]];
        for (int n = 0; n < A.nedges && counted && !none; ++n) {
            const ShapeEdge e = A.edges[n];
            const double dx = e.x1 - e.x0, dy = e.y1 - e.y0;
            double t0 = 0.0, t1 = 1.0;
            bool out_ = false;
            auto clip = [&](double dv, double lo, double hi, double pv) {
                if (dv == 0.0) {
                    out_ = out_ || pv < lo || pv > hi;
                    return;
                }
                double a = (lo - pv) / dv, b = (hi - pv) / dv;
                if (a > b) { const double w = a; a = b; b = w; }
                t0 = fmax(t0, a);
                t1 = fmin(t1, b);
                out_ = out_ || t0 >= t1;
            };
            clip(dx, xa, xb, e.x0);
            if (!out_) clip(dy, ya, yb, e.y0);
            if (out_) continue;
            // the parts between the crossings with the other counted primitives, in turn
            for (double ta = t0; ta < t1;) {
                double tb = t1;
                for (int a = 0; a < nu; ++a) {
                    if (u[a] == mine) continue;
                    const MatPrim &p = A.prims[A.seg_prim[p0 + u[a]]];
                    const int nv = mat_nvert(p);
                    for (int v = lane; v < nv; v += 64) {
                        double x1, y1, x2, y2;
                        mat_vertex(p, A.vx, A.vy, v, x1, y1);
                        mat_vertex(p, A.vx, A.vy, v + 1 < nv ? v + 1 : 0, x2, y2);
                        const double ex = x2 - x1, ey = y2 - y1, den = dx * ey - dy * ex;
                        if (den == 0.0) continue;
                        const double t = ((x1 - e.x0) * ey - (y1 - e.y0) * ex) / den;
                        const double w = ((x1 - e.x0) * dy - (y1 - e.y0) * dx) / den;
                        if (t0 < t && t < t1 && 0.0 <= w && w <= 1.0 && t > ta && t < tb) tb = t;
                    }
                }
#pragma unroll
                for (int w = 32; w > 0; w >>= 1) tb = fmin(tb, __shfl_xor(tb, w));
                const double tm = 0.5 * (ta + tb);
                const double xm = e.x0 + tm * (e.x1 - e.x0), ym = e.y0 + tm * (e.y1 - e.y0);
                bool hidden = false, found = false;
                double nr = A.bg_re, ni = A.bg_im;
                for (int a = 0; a < nu && !hidden && !found; ++a) {
                    if (u[a] == mine) continue;
                    const MatPrim &p = A.prims[A.seg_prim[p0 + u[a]]];
                    if (!mat_within(p, A.vx, A.vy, xm, ym, lane)) continue;
                    if (u[a] < mine) hidden = true;
                    else { found = true; nr = p.re; ni = p.im; }
                }
                if (!hidden) {
                    const double integ = e.len * (e.w0 * (tb - ta) + (e.w1 - e.w0) * 0.5 * (tb * tb - ta * ta));
                    tr += (P.re - nr) * integ;
                    ti += (P.im - ni) * integ;
                }
                ta = tb;
            }
        }
        const double area = (xb - xa) * (yb - ya);
        if (lane == 0) out[g] = make_double2(tr / area, ti / area);
    }
}

}  // namespace emf
