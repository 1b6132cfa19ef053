// Resident solve steps: many time steps per launch with the whole state of the
// grid held in registers.
//
// A grid of up to 655 thousand cells fits the vector registers of the chip
// (512 KB per CU) with its CPML psi and coefficients, one of up to 1.3 million
// without them.  Each work-group owns one box of cells, one (x, y) column of
// up to NZ planes per thread, loads E, H and the coefficients once, and takes
// `nsteps` steps; only the box faces travel between work-groups, through halo
// slots in device memory, and only neighbours wait for each other.  x and y
// neighbours inside a box go through LDS, z neighbours are the thread's own
// registers.  The CPML psi of a thread's cells are registers too (zero, with
// zero coefficients, outside the slabs).
//
// Slots carry their own validity: a slot is EMPTY (a signalling NaN, which no
// arithmetic result is) until the producer stores a value, and the consumer stores
// EMPTY back once it has read it.  A value and its arrival are then one
// transfer, where data followed by a flag would be two.  Slots are accessed
// with relaxed agent-scope atomics, which are coherent across the XCDs' L2s.
// Every slot exists twice (step parity): the EMPTY that a consumer stores at
// step s is complete when it has polled its slots of step s + 1 (the poll waits
// for all of the thread's memory operations), which happens before it sends
// the faces the producer needs to reach step s + 2 and reuse the slot.
//
// All work-groups have to run at the same time: the grid has at most one per
// CU, and the host admits launches together only where each XCD has a CU for all of
// their work-groups on it (ResGate).  Where they still do not run (another process
// holding CUs with a launch of the same kind), a poll gives up after RES_SPIN
// tries, sets conv->stalled and every work-group runs through without waiting; the
// host then repeats the solve with the two passes, and tries resident steps again
// some solves later.
#pragma once
#include "twopass.hpp"

namespace emf {

constexpr int RES_T = 512;            // threads of the largest box
constexpr int RES_STEPS = 64;         // steps per launch (their factors travel as arguments)
constexpr int RES_SPIN = 1 << 21;     // polls before a launch counts as stalled (seconds; ResArgs::spin)
constexpr int RES_PL = 592;           // doubles of one LDS plane: (BX + 1) (BY + 1) at most
constexpr int RES_W = 64;             // largest box width in x and in y
constexpr unsigned long long RES_EMPTY = 0x7FF4A5C3D2E1F00DULL;

struct ResArgs {
    int GX, GY, GZ;                   // boxes per axis
    int BX, BY;                       // largest box width in x and in y
    int nsteps;
    int spin;                         // polls before the launch counts as stalled
    unsigned long long *halo;         // [parity][E, H][box][res_slots]
    ConvState *conv;
    const SrcBlk *blk;
    int nsrc;
    int ub[6];                        // union box of the sources (PassSrc::ub)
    int src_cap;                      // deep boxes: double2 of LDS for source values
    double fac[RES_STEPS][6];         // per step: sin t, cos t, env(t) of the H and E halves
};

// Planes per thread with the whole state in registers; boxes with more planes
// are deep: only the fields stay in registers, psi and the E coefficients
// (which a step reads once) are read from memory, where each box's part
// stays in the L2 of its XCD or in the Infinity Cache, one plane ahead of
// their use.  us a step, two passes -> deep: 118x78x66 26.2 -> 16.3, 180x60x80
// 31.9 -> 20.3, 152x100x68 37.3 -> 25.3, 173x101x67 with complex eps 42.8 ->
// 30.2; of these about 6 us are psi's loads and stores and 1 to 6 the
// coefficients.  8 planes and more spill some registers (20 to 60).
constexpr int res_planes(bool ceps, bool mu) { return ceps || mu ? 3 : 5; }
// Deepest boxes.  Complex eps reads 24 B a cell more; non-uniform mu has no deep kernel.
constexpr int res_planes_deep(bool mu) { return mu ? 3 : 10; }
// x and y halo slots polled per thread
constexpr int res_items(bool deep) { return deep ? 2 : 1; }

// E and H share one LDS buffer (two more barriers per step) where the planes
// of both do not fit, and the E coefficients live in LDS, where the registers are full
constexpr bool res_share(int nz, bool deep) { return deep || nz > 4; }
constexpr bool res_tight(int nz, bool deep) { return !deep && nz > 4; }

// Whether the kernel keeps source values in LDS: the deep one of real eps.
// From memory, the box that holds a source waited for every plane of the column
// in turn, twice a step, and all other boxes for it (180x60x80, us a step:
// one source plane 25 -> 20, the six faces of an adjoint source 38 -> 26).
// With few planes the waits are few, and the longer code costs 2 to 6 %
// (126x51x64 39.1 -> 41.8 ms a solve); with complex eps it costs registers that
// the deep kernel spills (173x101x67 29.2 -> 29.9 ms).
constexpr bool res_src_in_lds(bool deep, bool ceps) { return deep && !ceps; }

constexpr size_t res_lds(int nz, bool deep, int bx, int by)
{
    return 8 * ((size_t)(res_share(nz, deep) ? 3 : 6) * nz * RES_PL +
                (res_tight(nz, deep) ? 3 * nz * RES_T : 0) + 6 * (size_t)(bx + by + nz) + 6 * RES_STEPS);
}

// halo slots of one box, field and parity: x face [component][plane][RES_W],
// y face the same, z face [component][column]
constexpr unsigned res_slots(int nz) { return 4u * nz * RES_W + 2u * RES_T; }

typedef __attribute__((address_space(1))) unsigned long long gslot;

__device__ __forceinline__ unsigned long long slot_load(const unsigned long long *base, unsigned off)
{
    return __hip_atomic_load((const gslot *)(reinterpret_cast<const char *>(base) + off),
                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ void slot_store(unsigned long long *base, unsigned off,
                                           unsigned long long v)
{
    __hip_atomic_store((gslot *)(reinterpret_cast<char *>(base) + off), v, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ void slot_put(unsigned long long *base, unsigned off, double v)
{
    slot_store(base, off, (unsigned long long)__double_as_longlong(v));
}

// Hides where a value comes from, so that what is computed from it inside the
// step loop is computed there: hoisted out of the loop, the addresses of every
// plane would take the registers that hold the state.
__device__ __forceinline__ void fresh(unsigned &v) { asm volatile("" : "+v"(v)); }
__device__ __forceinline__ void fresh_uniform(unsigned &v) { asm volatile("" : "+s"(v)); }

// CPML of one derivative: d becomes ki d + psi with psi <- c d + b psi
__device__ __forceinline__ void res_stretch(double &d, double &psi, double c, double b, double ki)
{
    psi = c * d + b * psi;
    d = ki * d + psi;
}

// the same with psi as it is in memory: c carries the spacing factor r of the axis, ri = 1 / r
__device__ __forceinline__ void res_stretch(double &d, double &psi, double c, double b, double ki,
                                            double ri)
{
    psi = c * d + b * psi;
    d = fma(ri, psi, ki * d);
}

template <int NZ, bool CEPS, bool MU>
__global__ __launch_bounds__(RES_T, 2) void k_resident(ResArgs R, FusedArgs A, Geo g,
                                                       const int *__restrict__ done)
{
    extern __shared__ double lds[];
    if (done && *done) return;
    constexpr bool DEEP = NZ > res_planes(CEPS, MU);
    constexpr bool TIGHT = res_tight(NZ, DEEP), SHARE = res_share(NZ, DEEP);
    constexpr int ITEMS = res_items(DEEP);
    constexpr int NP = DEEP ? 1 : NZ;     // planes of the arrays that deep boxes keep in memory
    static_assert(!(DEEP && MU), "no deep kernel with a mu array");
    constexpr int comp = NZ * RES_PL;
    const int Nx = g.Nx, Ny = g.Ny, Nz = g.Nz;
    const int GX = R.GX, GY = R.GY, GZ = R.GZ, nb = GX * GY * GZ;
    const int bl = (int)xcd_remap(blockIdx.x, (unsigned)nb);
    const int bx = bl % GX, by = (bl / GX) % GY, bz = bl / (GX * GY);
    const int x0 = bx * Nx / GX, xw = (bx + 1) * Nx / GX - x0;
    const int y0 = by * Ny / GY, yw = (by + 1) * Ny / GY - y0;
    const int z0 = bz * Nz / GZ, zw = (bz + 1) * Nz / GZ - z0;
    // planes: NZ, or NZ - 1 with a spare one on top.  Its E stays zero (no coefficients);
    // its H does not, but only the spare plane's own E and the neighbours' spare
    // planes read it.
    const bool full = zw == NZ;
    const int p = (int)threadIdx.x, nt = (int)blockDim.x;
    const bool on = p < xw * yw;
    const int y = on ? p / xw : 0, x = on ? p - y * xw : 0;
    const int k = x0 + x, j = y0 + y;
    const unsigned cs = A.cs, oz = (unsigned)g.nxy * 8u;
    const unsigned o = (((unsigned)z0 * (unsigned)Ny + (unsigned)j) * (unsigned)Nx + (unsigned)k) * 8u;
    const int CS = R.BX + 1;          // LDS row stride

    // LDS: E (halo column at x = xw, row at y = yw), H (halo column and row at
    // -1, stored shifted by one), E coefficients, CPML coefficients (H c, b,
    // 1/kappa, E c, b, 1/kappa) by x, y and plane, step factors
    double *const eb = lds, *const hb = SHARE ? eb : eb + 3 * comp;
    double *const bb = hb + 3 * comp;
    double *const xc = bb + (TIGHT ? 3 * NZ * RES_T : 0);
    double *const yc = xc + 6 * R.BX, *const zc = yc + 6 * R.BY, *const fac = zc + 6 * NZ;

    // CPML: which axes this box meets (uniform)
    const bool hasx = x0 < g.w[0] || x0 + xw > Nx - g.w[1];
    const bool hasy = y0 < g.w[2] || y0 + yw > Ny - g.w[3];
    const bool hasz = z0 < g.w[4] || z0 + zw - 1 > Nz - g.w[5];
    const Layout L = make_layout(g);
    {
        for (int q = p; q < xw + yw + NZ; q += nt) {
            const int a = q < xw ? 0 : (q < xw + yw ? 1 : 2);
            const int u = q - (a == 0 ? 0 : (a == 1 ? xw : xw + yw));
            Slab s = a == 0 ? slab_x(g, 0, 0, x0 + u)
                                  : (a == 1 ? slab_y(g, 0, y0 + u, 0) : slab_z(g, z0 + u, 0, 0));
            if (a == 2 && u >= zw) s.in = false;
            double *const c = (a == 0 ? xc : (a == 1 ? yc : zc)) + 6 * u;
            const unsigned t = L.tbo[a] + (s.in ? (unsigned)s.par * 8u : 0u), n = L.tbl[a];
            const double ra = !DEEP ? 1.0 : (a == 0 ? g.rx : (a == 1 ? g.ry : g.rz));
            c[0] = s.in ? ra * ldc(A.tab, t + 2 * n) : 0.0;
            c[1] = s.in ? ldc(A.tab, t + n) : 0.0;
            c[2] = s.in ? 1.0 / ldc(A.tab, t) : 1.0;
            c[3] = s.in ? ra * ldc(A.tab, t + 5 * n) : 0.0;
            c[4] = s.in ? ldc(A.tab, t + 4 * n) : 0.0;
            c[5] = s.in ? 1.0 / ldc(A.tab, t + 3 * n) : 1.0;
        }
        const double *f = &R.fac[0][0];
        for (int q = p; q < R.nsteps * 6; q += nt) fac[q] = f[q];
    }

    const double rx = g.rx, ry = g.ry, rz = g.rz;
    // state.  The E coefficients carry one of the curl's two spacing factors
    // (the other enters as a ratio, 1 on a cubic grid), the H ones both.
    double ex[NZ], ey[NZ], ez[NZ], hx[NZ], hy[NZ], hz[NZ];
    double b0[TIGHT ? 1 : NP], b1[TIGHT ? 1 : NP], b2[TIGHT ? 1 : NP];
    double a0[CEPS ? NP : 1], a1[CEPS ? NP : 1], a2[CEPS ? NP : 1];
    double m0[MU ? NZ : 1], m1[MU ? NZ : 1], m2[MU ? NZ : 1];
    // psi of d/dx of the y and z components, d/dy of x and z, d/dz of x and y,
    // in units of the undivided differences
    double px0[NP], px1[NP], py0[NP], py1[NP], pz0[NP], pz1[NP];
    double qx0[NP], qx1[NP], qy0[NP], qy1[NP], qz0[NP], qz1[NP];
    // f(offset, H psi, E psi, axis) of every psi of the column
    auto each_psi = [&](auto &&f) {
#pragma unroll
        for (int q = 0; q < NP; ++q) {
            if (q >= zw) break;
            __builtin_amdgcn_sched_barrier(0);
            const Slab sx = slab_x(g, z0 + q, j, k), sy = slab_y(g, z0 + q, j, k),
                       sz = slab_z(g, z0 + q, j, k);
            if (hasx && on && sx.in) {
                f(psof(L, 0, sx.lo, 0) + sx.io, px0[q], qx0[q], 0);
                f(psof(L, 0, sx.lo, 1) + sx.io, px1[q], qx1[q], 0);
            }
            if (hasy && on && sy.in) {
                f(psof(L, 1, sy.lo, 0) + sy.io, py0[q], qy0[q], 1);
                f(psof(L, 1, sy.lo, 1) + sy.io, py1[q], qy1[q], 1);
            }
            if (hasz && on && sz.in) {
                f(psof(L, 2, sz.lo, 0) + sz.io, pz0[q], qz0[q], 2);
                f(psof(L, 2, sz.lo, 1) + sz.io, pz1[q], qz1[q], 2);
            }
        }
    };
#pragma unroll
    for (int q = 0; q < NZ; ++q) {
        __builtin_amdgcn_sched_barrier(0);
        const unsigned c = o + (unsigned)q * oz;
        const bool v = on && q < zw;
        ex[q] = ey[q] = ez[q] = hx[q] = hy[q] = hz[q] = 0;
        if (DEEP) {
            if (v) {
                ex[q] = ldo(A.Eo, c); ey[q] = ldo(A.Eo, c + cs); ez[q] = ldo(A.Eo, c + 2 * cs);
                hx[q] = ldo(A.Ho, c); hy[q] = ldo(A.Ho, c + cs); hz[q] = ldo(A.Ho, c + 2 * cs);
            }
            continue;
        }
        const int u = DEEP ? 0 : q;
        px0[u] = px1[u] = py0[u] = py1[u] = pz0[u] = pz1[u] = 0;
        qx0[u] = qx1[u] = qy0[u] = qy1[u] = qz0[u] = qz1[u] = 0;
        double u0 = 0, u1 = 0, u2 = 0;
        if (v) {
            ex[q] = ldo(A.Eo, c); ey[q] = ldo(A.Eo, c + cs); ez[q] = ldo(A.Eo, c + 2 * cs);
            hx[q] = ldo(A.Ho, c); hy[q] = ldo(A.Ho, c + cs); hz[q] = ldo(A.Ho, c + 2 * cs);
            u0 = ldo(A.bE, c) * rz; u1 = ldo(A.bE, c + cs) * rx; u2 = ldo(A.bE, c + 2 * cs) * ry;
        }
        if (TIGHT) {
            bb[(3 * q) * RES_T + p] = u0;
            bb[(3 * q + 1) * RES_T + p] = u1;
            bb[(3 * q + 2) * RES_T + p] = u2;
        } else {
            b0[TIGHT ? 0 : u] = u0; b1[TIGHT ? 0 : u] = u1; b2[TIGHT ? 0 : u] = u2;
        }
        if (CEPS) {
            a0[u] = v ? ldo(A.aE, c) : 0; a1[u] = v ? ldo(A.aE, c + cs) : 0;
            a2[u] = v ? ldo(A.aE, c + 2 * cs) : 0;
        }
        if (MU) {
            m0[q] = v ? ldo(A.mH, c) : 0; m1[q] = v ? ldo(A.mH, c + cs) : 0;
            m2[q] = v ? ldo(A.mH, c + 2 * cs) : 0;
        }
    }
    if (!DEEP && (hasx || hasy || hasz))
        each_psi([&](unsigned off, double &ph, double &pe, int a) {
            const double ri = a == 0 ? 1.0 / rx : (a == 1 ? 1.0 / ry : 1.0 / rz);
            ph = ldo(A.pho, off) * ri;
            pe = ldo(A.pe, off) * ri;
        });

    // the halo slot this thread polls: of the box's x face (2 NZ yw: the two
    // tangential components of each plane and row) and y face (2 NZ xw)
    constexpr unsigned SB = 8u * res_slots(NZ);   // bytes of a box's slots
    constexpr unsigned YF = 16u * NZ * RES_W, ZF = 2 * YF;   // y and z faces in them
    constexpr unsigned QB = 8u * RES_W;           // bytes to the next plane of a face
    const unsigned fb = (unsigned)nb * SB;        // to the next field
    const unsigned own = (unsigned)bl * SB;
    unsigned slot[ITEMS], pos[ITEMS];   // byte offset of the slot; LDS byte of the E halo
    int dpos[ITEMS];                        // from the E to the H place
    bool oke[ITEMS], okh[ITEMS];        // there is a neighbour on that side
#pragma unroll
    for (int it = 0; it < ITEMS; ++it) {
        const int t = p + it * nt, nxi = 2 * NZ * yw;
        slot[it] = own;
        pos[it] = 0;
        dpos[it] = 0;
        oke[it] = okh[it] = false;
        if (t < nxi) {
            const int c = t / (NZ * yw), r = t - c * NZ * yw, q = r / yw, u = r - q * yw;
            slot[it] = own + 8u * (unsigned)((c * NZ + q) * RES_W + u);
            pos[it] = 8u * (unsigned)((1 + c) * comp + q * RES_PL + u * CS + xw);
            dpos[it] = 8 * (CS - xw);
            oke[it] = bx + 1 < GX;
            okh[it] = bx > 0;
        } else if (t < nxi + 2 * NZ * xw) {
            const int s = t - nxi, c = s / (NZ * xw), r = s - c * NZ * xw, q = r / xw, u = r - q * xw;
            slot[it] = own + YF + 8u * (unsigned)((c * NZ + q) * RES_W + u);
            pos[it] = 8u * (unsigned)(2 * c * comp + q * RES_PL + yw * CS + u);
            dpos[it] = 8 * (1 - yw * CS);
            oke[it] = by + 1 < GY;
            okh[it] = by > 0;
        }
    }
    constexpr unsigned ZB = 8u * RES_T;           // bytes to the second component of the z face
    unsigned zslot = own + ZF + 8u * (unsigned)p;
    bool dead = false;

    // wait for the halo of the field and parity at byte offset f: the x and y
    // slots xy, returned in v, and the two z neighbours of the column (zon)
    auto recv = [&](unsigned f, const bool (&xy)[ITEMS], bool zon, double (&vd)[ITEMS],
                    double &z0v, double &z1v) {
        unsigned long long v[ITEMS] = {}, a = 0, b = 0;
        const unsigned sz = f + zslot;
        for (int spin = 1;; ++spin) {
#pragma unroll
            for (int it = 0; it < ITEMS; ++it)
                if (xy[it]) v[it] = slot_load(R.halo, f + slot[it]);
            if (zon) { a = slot_load(R.halo, sz); b = slot_load(R.halo, sz + ZB); }
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            bool miss = a == RES_EMPTY || b == RES_EMPTY;
#pragma unroll
            for (int it = 0; it < ITEMS; ++it) miss |= v[it] == RES_EMPTY;
            if (!miss || dead) break;
            if (spin >= R.spin) {
                __hip_atomic_store(&R.conv->stalled, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                dead = true;
            } else if ((spin & 1023) == 0) {
                dead = __hip_atomic_load(&R.conv->stalled, __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_AGENT) != 0;
            }
        }
#pragma unroll
        for (int it = 0; it < ITEMS; ++it) {
            if (xy[it]) slot_store(R.halo, f + slot[it], RES_EMPTY);
            vd[it] = __longlong_as_double(v[it]);
        }
        if (zon) { slot_store(R.halo, sz, RES_EMPTY); slot_store(R.halo, sz + ZB, RES_EMPTY); }
        z0v = __longlong_as_double(a);
        z1v = __longlong_as_double(b);
    };

    // this thread's cells in the LDS planes (bytes), and its places in the box faces
    unsigned le = 8u * (unsigned)(y * CS + x), lh = 8u * (unsigned)((y + 1) * CS + x + 1);
    const unsigned rs = 8u * (unsigned)CS;        // LDS row
    unsigned yx = own + YF + 8u * (unsigned)x, yy = own + 8u * (unsigned)y;
    const bool elx = on && x == 0, ely = on && y == 0, ehx = on && x == xw - 1, ehy = on && y == yw - 1;
    const unsigned dz = (unsigned)(GX * GY) * SB, dy = (unsigned)GX * SB;
    auto E = [&](int c, int q, unsigned at) -> double & {
        return *reinterpret_cast<double *>(reinterpret_cast<char *>(eb) + at +
                                           8u * (unsigned)(c * comp + q * RES_PL));
    };
    auto H = [&](int c, int q, unsigned at) -> double & {
        return *reinterpret_cast<double *>(reinterpret_cast<char *>(hb) + at +
                                           8u * (unsigned)(c * comp + q * RES_PL));
    };
    // E of the box to LDS; its min faces to the neighbours; 0 past the grid's max faces
    auto put_e = [&](unsigned f) {
        if (bz > 0 && on) {
            const unsigned d = f + zslot - dz;
            slot_put(R.halo, d, ex[0]); slot_put(R.halo, d + ZB, ey[0]);
        }
        if (by > 0 && ely) {
            const unsigned d = f + yx - dy;
#pragma unroll
            for (int q = 0; q < NZ; ++q) {
                slot_put(R.halo, d + q * QB, ex[q]);
                slot_put(R.halo, d + (NZ + q) * QB, ez[q]);
            }
        }
        if (bx > 0 && elx) {
            const unsigned d = f + yy - SB;
#pragma unroll
            for (int q = 0; q < NZ; ++q) {
                slot_put(R.halo, d + q * QB, ey[q]);
                slot_put(R.halo, d + (NZ + q) * QB, ez[q]);
            }
        }
        if (on) {
#pragma unroll
            for (int q = 0; q < NZ; ++q) { E(0, q, le) = ex[q]; E(1, q, le) = ey[q]; E(2, q, le) = ez[q]; }
        }
        if (bx == GX - 1 && ehx) {
#pragma unroll
            for (int q = 0; q < NZ; ++q) E(1, q, le + 8u) = E(2, q, le + 8u) = 0;
        }
        if (by == GY - 1 && ehy) {
#pragma unroll
            for (int q = 0; q < NZ; ++q) E(0, q, le + rs) = E(2, q, le + rs) = 0;
        }
    };
    // min-face ghost rule of H: '0' -> 0, 'E' -> -H(first), 'H' -> +H(first)
    auto sign = [](int b) { return b == 'E' ? -1.0 : (b == 'H' ? 1.0 : 0.0); };
    // H of the box to LDS; its max faces to the neighbours; ghosts past the grid's min faces
    auto put_h = [&](unsigned f) {
        if (bz + 1 < GZ && on) {
            const unsigned d = f + zslot + dz;
            slot_put(R.halo, d, full ? hx[NZ - 1] : hx[NZ > 1 ? NZ - 2 : 0]);
            slot_put(R.halo, d + ZB, full ? hy[NZ - 1] : hy[NZ > 1 ? NZ - 2 : 0]);
        }
        if (by + 1 < GY && ehy) {
            const unsigned d = f + yx + dy;
#pragma unroll
            for (int q = 0; q < NZ; ++q) {
                slot_put(R.halo, d + q * QB, hx[q]);
                slot_put(R.halo, d + (NZ + q) * QB, hz[q]);
            }
        }
        if (bx + 1 < GX && ehx) {
            const unsigned d = f + yy + SB;
#pragma unroll
            for (int q = 0; q < NZ; ++q) {
                slot_put(R.halo, d + q * QB, hy[q]);
                slot_put(R.halo, d + (NZ + q) * QB, hz[q]);
            }
        }
        if (on) {
#pragma unroll
            for (int q = 0; q < NZ; ++q) { H(0, q, lh) = hx[q]; H(1, q, lh) = hy[q]; H(2, q, lh) = hz[q]; }
        }
        if (bx == 0 && elx) {
            const double sg = sign(g.bc[0]);
#pragma unroll
            for (int q = 0; q < NZ; ++q) { H(1, q, lh - 8u) = sg * hy[q]; H(2, q, lh - 8u) = sg * hz[q]; }
        }
        if (by == 0 && ely) {
            const double sg = sign(g.bc[1]);
#pragma unroll
            for (int q = 0; q < NZ; ++q) { H(0, q, lh - rs) = sg * hx[q]; H(2, q, lh - rs) = sg * hz[q]; }
        }
    };

    const bool anysrc = R.nsrc > 0 && x0 < R.ub[5] && x0 + xw > R.ub[4] && y0 < R.ub[3] &&
                        y0 + yw > R.ub[2] && z0 < R.ub[1] && z0 + zw > R.ub[0];
    // The box's part of a block: its corner, extent and place in the LDS list, where
    // the values wait times the factor of the update they enter (6 n double2,
    // component by component; as many blocks as src_cap holds).
    constexpr bool LSRC = res_src_in_lds(DEEP, CEPS);
    double2 *const sl = reinterpret_cast<double2 *>(fac + 6 * RES_STEPS);
    struct Part { int k, j, i, K, J, I, n; };
    auto part = [&](const SrcBlk &b, Part &t) {
        t.k = max(b.k0, x0); t.j = max(b.j0, y0); t.i = max(b.i0, z0);
        t.K = min(b.k0 + b.K, x0 + xw) - t.k;
        t.J = min(b.j0 + b.J, y0 + yw) - t.j;
        t.I = min(b.i0 + b.I, z0 + zw) - t.i;
        t.n = t.K > 0 && t.J > 0 && t.I > 0 ? t.K * t.J * t.I : 0;
        return t.n > 0;
    };
    if (LSRC && anysrc) {
        int base = 0;
        for (int s = 0; s < R.nsrc; ++s) {
            const SrcBlk sb = src_blk(R.blk, s);
            Part t;
            if (!part(sb, t) || base + 6 * t.n > R.src_cap) continue;
            for (int e = p; e < t.n; e += nt) {
                const int i = t.i + e / (t.J * t.K), jj = t.j + e / t.K % t.J, kk = t.k + e % t.K;
                long long m;
                in_box(sb, i, jj, kk, m);
                const unsigned c = (((unsigned)i * (unsigned)Ny + (unsigned)jj) * (unsigned)Nx + (unsigned)kk) * 8u;
#pragma unroll
                for (int f = 0; f < 6; ++f) {
                    const double w = f < 3 ? ldo(A.bE, c + (unsigned)f * cs)
                                           : (MU ? ldo(A.mH, c + (unsigned)(f - 3) * cs) : A.m_s);
                    double2 v = ld2(sb.f[f] + m);
                    v.x *= w; v.y *= w;
                    sl[base + f * t.n + e] = v;
                }
            }
            base += 6 * t.n;
        }
    }
    // for every source cell of the column: put(q, value times factor) of those in
    // LDS, add(q, value) of the others, of the block's components c0 .. c0 + 2
    auto sources = [&](int c0, double st, double ct, double env, auto &&put, auto &&add) {
        int base = 0;
        for (int s = 0; s < R.nsrc; ++s) {
            const SrcBlk sb = src_blk(R.blk, s);
            if (sb.k0 >= x0 + xw || sb.k0 + sb.K <= x0 || sb.j0 >= y0 + yw ||
                sb.j0 + sb.J <= y0 || sb.i0 >= z0 + zw || sb.i0 + sb.I <= z0)
                continue;
            Part t;
            if (LSRC) part(sb, t);
            if (LSRC && base + 6 * t.n <= R.src_cap) {
                const int a = k - t.k, b = j - t.j, zs = t.i - z0, ze = zs + t.I;
                if (on && (unsigned)a < (unsigned)t.K && (unsigned)b < (unsigned)t.J) {
                    const double2 *v = sl + base + c0 * t.n + b * t.K + a;
#pragma unroll
                    for (int q = 0; q < NZ; ++q)
                        if (q >= zs && q < ze) {
                            const double2 *w = v + (q - zs) * t.J * t.K;
                            const double2 vx = w[0], vy = w[t.n], vz = w[2 * t.n];
                            put(q, env * (st * vx.x + ct * vx.y), env * (st * vy.x + ct * vy.y),
                                env * (st * vz.x + ct * vz.y));
                        }
                }
                base += 6 * t.n;
                continue;
            }
#pragma unroll
            for (int q = 0; q < NZ; ++q) {
                long long m;
                if (q < zw && on && in_box(sb, z0 + q, j, k, m)) {
                    const double2 vx = ld2(sb.f[c0] + m), vy = ld2(sb.f[c0 + 1] + m),
                                  vz = ld2(sb.f[c0 + 2] + m);
                    add(q, env * (st * vx.x + ct * vx.y), env * (st * vy.x + ct * vy.y),
                        env * (st * vz.x + ct * vz.y));
                }
            }
        }
    };

    // curl factors: H coefficients times the spacing factors, and the ratios of the E update
    const double sx = MU ? rx : A.m_s * rx, sy = MU ? ry : A.m_s * ry, sz = MU ? rz : A.m_s * rz;
    const double ryz = ry / rz, rzx = rz / rx, rxy = rx / ry;
    auto coef = [&](const double (&f)[TIGHT ? 1 : NP], int c, int q) {
        if (DEEP) return ldo(A.bE, o + (unsigned)q * oz + (unsigned)c * cs) * (c == 0 ? rz : (c == 1 ? rx : ry));
        return TIGHT ? bb[(3 * q + c) * RES_T + p] : f[TIGHT || DEEP ? 0 : q];
    };
    // plane q + 1 of an E component: the column's own, past its top the neighbour's
    auto above = [&](const double (&f)[NZ], int q, double top) {
        if (q + 1 >= NZ) return top;
        const double v = f[q + 1 < NZ ? q + 1 : q];
        return q + 2 < NZ || full ? v : top;
    };
    // Deep boxes: psi and coefficients of this thread's cells in memory, through
    // buffer accesses, whose range check makes the code straight: a cell that
    // has no such value has the offset NONE, which loads 0 and stores nothing.
    // A box that meets both faces of an axis has slabs of one width there.
    constexpr unsigned NONE = 0x80000000u;   // past every array, also with what is added to it
    unsigned ox_ = NONE, oy_ = NONE, oz_ = NONE;
    unsigned dxs = 0, dxc = 0, dys = 0, dyc = 0;       // to the next plane and the second array
    unsigned zin = 0, zlo = 0, za0 = 0, za1 = 0, zb0 = 0, zb1 = 0;   // planes in a z slab, in the min one; plane z0 in each
    if (DEEP) {
        const Slab a = slab_x(g, z0, j, k), b = slab_y(g, z0, j, k);
        if (on && a.in) ox_ = psof(L, 0, a.lo, 0) + a.io;
        if (on && b.in) oy_ = psof(L, 1, b.lo, 0) + b.io;
        if (on) oz_ = ((unsigned)j * (unsigned)Nx + (unsigned)k) * 8u;
        const unsigned wx = (unsigned)(x0 < g.w[0] ? g.w[0] : g.w[1]), wy = (unsigned)(y0 < g.w[2] ? g.w[2] : g.w[3]);
        dxs = (unsigned)Ny * wx * 8u; dxc = (unsigned)Nz * dxs;
        dys = (unsigned)Nx * wy * 8u; dyc = (unsigned)Nz * dys;
        for (int q = 0; q < zw; ++q) {
            const Slab z = slab_z(g, z0 + q, 0, 0);
            zin |= z.in ? 1u << q : 0u;
            zlo |= z.lo ? 1u << q : 0u;
        }
        za0 = psof(L, 2, true, 0) + (unsigned)z0 * oz; za1 = psof(L, 2, true, 1) + (unsigned)z0 * oz;
        zb0 = psof(L, 2, false, 0) + (unsigned)(z0 - Nz + g.w[5]) * oz;
        zb1 = psof(L, 2, false, 1) + (unsigned)(z0 - Nz + g.w[5]) * oz;
    }
    const unsigned pbytes = 2u * 8u * (unsigned)((g.w[0] + g.w[1]) * Nz * Ny + (g.w[2] + g.w[3]) * Nz * Nx +
                                                 (g.w[4] + g.w[5]) * Ny * Nx);
    typedef __attribute__((__vector_size__(2 * sizeof(unsigned)))) unsigned u2;
    auto buf_get = [](__amdgpu_buffer_rsrc_t r, unsigned v, unsigned so) {
        return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, (int)v, (int)so, 0));
    };
    auto buf_put = [](__amdgpu_buffer_rsrc_t r, unsigned v, unsigned so, double d) {
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u2, d), r, (int)v, (int)so, 0);
    };
    auto rsrc = [](const double *p, unsigned bytes) {
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<double *>(p), 0, (int)bytes, 0x00020000);
    };
    unsigned ozs = oz, css = cs;
    auto fresh_deep = [&] {
        fresh(ox_); fresh(oy_); fresh(oz_);
        fresh_uniform(dxs); fresh_uniform(dxc); fresh_uniform(dys); fresh_uniform(dyc);
        fresh_uniform(zin); fresh_uniform(zlo);
        fresh_uniform(za0); fresh_uniform(za1); fresh_uniform(zb0); fresh_uniform(zb1);
        fresh_uniform(ozs); fresh_uniform(css);
    };
    // plane q's psi from, or to, the arrays of one field
    auto psi_off = [&](int q, unsigned &vx, unsigned &vy, unsigned &vz, unsigned &z0o, unsigned &z1o) {
        const unsigned spare = q < zw ? 0u : NONE;
        vx = ox_ | spare;
        vy = oy_ | spare;
        vz = oz_ | ((zin >> q) & 1u ? 0u : NONE);
        const bool lo = (zlo >> q) & 1u;
        z0o = (lo ? za0 : zb0) + (unsigned)q * ozs;
        z1o = (lo ? za1 : zb1) + (unsigned)q * ozs;
    };
    auto psi_get = [&](const double *f, int q, double (&v)[6]) {
        unsigned vx, vy, vz, za, zb;
        psi_off(q, vx, vy, vz, za, zb);
        const auto r = rsrc(f, pbytes);
        v[0] = buf_get(r, vx, (unsigned)q * dxs); v[1] = buf_get(r, vx, (unsigned)q * dxs + dxc);
        v[2] = buf_get(r, vy, (unsigned)q * dys); v[3] = buf_get(r, vy, (unsigned)q * dys + dyc);
        v[4] = buf_get(r, vz, za); v[5] = buf_get(r, vz, zb);
    };
    auto psi_put = [&](double *f, int q, const double (&v)[6]) {
        unsigned vx, vy, vz, za, zb;
        psi_off(q, vx, vy, vz, za, zb);
        const auto r = rsrc(f, pbytes);
        buf_put(r, vx, (unsigned)q * dxs, v[0]); buf_put(r, vx, (unsigned)q * dxs + dxc, v[1]);
        buf_put(r, vy, (unsigned)q * dys, v[2]); buf_put(r, vy, (unsigned)q * dys + dyc, v[3]);
        buf_put(r, vz, za, v[4]); buf_put(r, vz, zb, v[5]);
    };
    // plane q's E coefficients: b and, with complex eps, a (0 where there is no cell)
    unsigned ob = on ? o : NONE;
    auto coef_get = [&](int q, double (&v)[CEPS ? 6 : 3]) {
        const unsigned c = ob | (q < zw ? 0u : NONE), so = (unsigned)q * ozs;
        const auto r = rsrc(A.bE, 3u * css);
        v[0] = buf_get(r, c, so); v[1] = buf_get(r, c, so + css); v[2] = buf_get(r, c, so + 2 * css);
        if (CEPS) {
            const auto ra = rsrc(A.aE, 3u * css);
            v[CEPS ? 3 : 0] = buf_get(ra, c, so); v[CEPS ? 4 : 0] = buf_get(ra, c, so + css);
            v[CEPS ? 5 : 0] = buf_get(ra, c, so + 2 * css);
        }
    };
    const double rix = 1.0 / rx, riy = 1.0 / ry, riz = 1.0 / rz;
    // Every box runs the CPML arithmetic (with psi = 0 and c = b = 0 outside
    // the slabs): a box waits for its neighbours each half step, so the boxes in
    // the corners, which need it on all axes, set the pace, and a straight line
    // of code runs faster than one with a branch per axis.
    {
        unsigned fe = 0;              // field offset of E at this step's parity; H follows
        put_e(fe);
        for (int s = 0; s < R.nsteps; ++s) {
            double zx, zy;
            double pn[6] = {};        // deep: the next plane's psi
            double cn[CEPS ? 6 : 3] = {};
            // ------------------------------------------------------ H half
            if (DEEP) fresh_deep();
            fresh(zslot); fresh(le); fresh(lh); fresh(yx); fresh(yy);
            {
                double v[ITEMS];
                if (DEEP) psi_get(A.pho, 0, pn);
                recv(fe, oke, on && bz + 1 < GZ, v, zx, zy);
#pragma unroll
                for (int it = 0; it < ITEMS; ++it)
                    if (oke[it]) E(0, 0, pos[it]) = v[it];
            }
            __syncthreads();
            {
                const double cx = xc[6 * x], bx_ = xc[6 * x + 1], kx = xc[6 * x + 2];
                const double cy = yc[6 * y], by_ = yc[6 * y + 1], ky = yc[6 * y + 2];
                const unsigned lr = le + rs;
#pragma unroll
                for (int q = 0; q < NZ; ++q) {
                    __builtin_amdgcn_sched_barrier(0);
                    const double cz = zc[6 * q], bz_ = zc[6 * q + 1], kz = zc[6 * q + 2];
                    double dzy_ = above(ey, q, zy) - ey[q], dyz_ = E(2, q, lr) - ez[q];
                    double dxz_ = E(2, q, le + 8u) - ez[q], dzx_ = above(ex, q, zx) - ex[q];
                    double dyx_ = E(0, q, lr) - ex[q], dxy_ = E(1, q, le + 8u) - ey[q];
                    if (DEEP) {
                        double pc[6];
#pragma unroll
                        for (int n = 0; n < 6; ++n) pc[n] = pn[n];
                        if (q + 1 < NZ) psi_get(A.pho, q + 1, pn);
                        res_stretch(dzy_, pc[5], cz, bz_, kz, riz);
                        res_stretch(dzx_, pc[4], cz, bz_, kz, riz);
                        res_stretch(dyz_, pc[3], cy, by_, ky, riy);
                        res_stretch(dyx_, pc[2], cy, by_, ky, riy);
                        res_stretch(dxz_, pc[1], cx, bx_, kx, rix);
                        res_stretch(dxy_, pc[0], cx, bx_, kx, rix);
                        psi_put(A.phn, q, pc);
                    } else {
                        const int u = DEEP ? 0 : q;
                        res_stretch(dzy_, pz1[u], cz, bz_, kz);
                        res_stretch(dzx_, pz0[u], cz, bz_, kz);
                        res_stretch(dyz_, py1[u], cy, by_, ky);
                        res_stretch(dyx_, py0[u], cy, by_, ky);
                        res_stretch(dxz_, px1[u], cx, bx_, kx);
                        res_stretch(dxy_, px0[u], cx, bx_, kx);
                    }
                    if (MU) {
                        hx[q] = fma(m0[MU ? q : 0], sz * dzy_ - sy * dyz_, hx[q]);
                        hy[q] = fma(m1[MU ? q : 0], sx * dxz_ - sz * dzx_, hy[q]);
                        hz[q] = fma(m2[MU ? q : 0], sy * dyx_ - sx * dxy_, hz[q]);
                    } else {
                        hx[q] = fma(sz, dzy_, fma(-sy, dyz_, hx[q]));
                        hy[q] = fma(sx, dxz_, fma(-sz, dzx_, hy[q]));
                        hz[q] = fma(sy, dyx_, fma(-sx, dxy_, hz[q]));
                    }
                }
            }
            if (anysrc)
                sources(3, fac[6 * s], fac[6 * s + 1], fac[6 * s + 2],
                        [&](int q, double vx, double vy, double vz) { hx[q] += vx; hy[q] += vy; hz[q] += vz; },
                        [&](int q, double vx, double vy, double vz) {
                            hx[q] += vx * (MU ? m0[MU ? q : 0] : A.m_s);
                            hy[q] += vy * (MU ? m1[MU ? q : 0] : A.m_s);
                            hz[q] += vz * (MU ? m2[MU ? q : 0] : A.m_s);
                        });
            if (SHARE) __syncthreads();
            put_h(fe + fb);
            // ------------------------------------------------------ E half
            if (DEEP) { fresh_deep(); fresh(ob); }
            fresh(zslot); fresh(le); fresh(lh); fresh(yx); fresh(yy);
            {
                double v[ITEMS];
                if (DEEP) { psi_get(A.pe, 0, pn); coef_get(0, cn); }
                recv(fe + fb, okh, on && bz > 0, v, zx, zy);
#pragma unroll
                for (int it = 0; it < ITEMS; ++it)
                    if (okh[it]) H(0, 0, pos[it] + (unsigned)dpos[it]) = v[it];
            }
            if (bz == 0) { const double sg = sign(g.bc[2]); zx = sg * hx[0]; zy = sg * hy[0]; }
            __syncthreads();
            {
                const double cx = xc[6 * x + 3], bx_ = xc[6 * x + 4], kx = xc[6 * x + 5];
                const double cy = yc[6 * y + 3], by_ = yc[6 * y + 4], ky = yc[6 * y + 5];
                const unsigned lr = lh - rs, lx = lh - 8u;
#pragma unroll
                for (int q = 0; q < NZ; ++q) {
                    __builtin_amdgcn_sched_barrier(0);
                    const double cz = zc[6 * q + 3], bz_ = zc[6 * q + 4], kz = zc[6 * q + 5];
                    const int n = q > 0 ? q - 1 : 0;
                    double dyz_ = hz[q] - H(2, q, lr), dzy_ = hy[q] - (q > 0 ? hy[n] : zy);
                    double dzx_ = hx[q] - (q > 0 ? hx[n] : zx), dxz_ = hz[q] - H(2, q, lx);
                    double dxy_ = hy[q] - H(1, q, lx), dyx_ = hx[q] - H(0, q, lr);
                    if (DEEP) {
                        double pc[6], cc[CEPS ? 6 : 3];
#pragma unroll
                        for (int n = 0; n < 6; ++n) pc[n] = pn[n];
#pragma unroll
                        for (int n = 0; n < (CEPS ? 6 : 3); ++n) cc[n] = cn[n];
                        if (q + 1 < NZ) { psi_get(A.pe, q + 1, pn); coef_get(q + 1, cn); }
                        res_stretch(dyz_, pc[3], cy, by_, ky, riy);
                        res_stretch(dyx_, pc[2], cy, by_, ky, riy);
                        res_stretch(dzy_, pc[5], cz, bz_, kz, riz);
                        res_stretch(dzx_, pc[4], cz, bz_, kz, riz);
                        res_stretch(dxz_, pc[1], cx, bx_, kx, rix);
                        res_stretch(dxy_, pc[0], cx, bx_, kx, rix);
                        psi_put(A.pe, q, pc);
                        ex[q] = fma(fma(ry, dyz_, -(rz * dzy_)), cc[0],
                                    CEPS ? cc[CEPS ? 3 : 0] * ex[q] : ex[q]);
                        ey[q] = fma(fma(rz, dzx_, -(rx * dxz_)), cc[1],
                                    CEPS ? cc[CEPS ? 4 : 0] * ey[q] : ey[q]);
                        ez[q] = fma(fma(rx, dxy_, -(ry * dyx_)), cc[2],
                                    CEPS ? cc[CEPS ? 5 : 0] * ez[q] : ez[q]);
                    } else {
                        const int u = DEEP ? 0 : q, w = CEPS ? u : 0;
                        res_stretch(dyz_, qy1[u], cy, by_, ky);
                        res_stretch(dyx_, qy0[u], cy, by_, ky);
                        res_stretch(dzy_, qz1[u], cz, bz_, kz);
                        res_stretch(dzx_, qz0[u], cz, bz_, kz);
                        res_stretch(dxz_, qx1[u], cx, bx_, kx);
                        res_stretch(dxy_, qx0[u], cx, bx_, kx);
                        ex[q] = fma(fma(ryz, dyz_, -dzy_), coef(b0, 0, q), CEPS ? a0[w] * ex[q] : ex[q]);
                        ey[q] = fma(fma(rzx, dzx_, -dxz_), coef(b1, 1, q), CEPS ? a1[w] * ey[q] : ey[q]);
                        ez[q] = fma(fma(rxy, dxy_, -dyx_), coef(b2, 2, q), CEPS ? a2[w] * ez[q] : ez[q]);
                    }
                }
            }
            if (anysrc) {
                const double ix = 1.0 / rx, iy = 1.0 / ry, iz = 1.0 / rz;
                sources(0, fac[6 * s + 3], fac[6 * s + 4], fac[6 * s + 5],
                        [&](int q, double vx, double vy, double vz) { ex[q] -= vx; ey[q] -= vy; ez[q] -= vz; },
                        [&](int q, double vx, double vy, double vz) {
                            ex[q] -= vx * (coef(b0, 0, q) * iz);
                            ey[q] -= vy * (coef(b1, 1, q) * ix);
                            ez[q] -= vz * (coef(b2, 2, q) * iy);
                        });
            }
            if (SHARE) __syncthreads();
            fe = 2u * fb - fe;        // the other parity
            if (s + 1 < R.nsteps) put_e(fe);
        }
    }
#pragma unroll
    for (int q = 0; q < NZ; ++q) {
        if (on && q < zw) {
            const unsigned c = o + (unsigned)q * oz;
            sto(A.En, c, ex[q]); sto(A.En, c + cs, ey[q]); sto(A.En, c + 2 * cs, ez[q]);
            sto(A.Hn, c, hx[q]); sto(A.Hn, c + cs, hy[q]); sto(A.Hn, c + 2 * cs, hz[q]);
        }
    }
    if (!DEEP && (hasx || hasy || hasz))
        each_psi([&](unsigned off, double &ph, double &pe, int a) {
            const double r = a == 0 ? rx : (a == 1 ? ry : rz);
            sto(A.phn, off, ph * r);
            sto(A.pe, off, pe * r);
        });
}

__global__ void k_fill_slots(unsigned long long *s, long long n)
{
    for (long long q = blockIdx.x * (long long)blockDim.x + threadIdx.x; q < n;
         q += (long long)gridDim.x * blockDim.x)
        s[q] = RES_EMPTY;
}

}  // namespace emf
