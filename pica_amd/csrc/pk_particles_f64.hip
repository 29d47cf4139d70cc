// pk_particles_f64.hip -- fused interpolation + Boris push + current deposition, FP64,
// absolute positions, one workgroup per supercell (gfx950).
//
// Per workgroup (supercell s, XCD-aware numbering):
//   1. gather the E/B stencil of the supercell into LDS (FieldInterpolatorCICSupercell ctor,
//      FieldInterpolatorYeeGrid.h:197-223) and zero an LDS J tile
//      (CurrentDepositorCICSupercell ctor, CurrentDepositorYeeGrid.h:178-199);
//   2. stream the supercell's SoA particles, each wavefront its own 64-particle groups with no
//      workgroup barrier, coalesced: interpolate (:225-242, 257-281), push
//      (BorisPusher.h:32-47), deposit into the LDS tile with LDS atomics
//      (CurrentDepositorYeeGrid.h:215-262, or Esirkepov), write x, u back in place;
//   3. particles that leave are copied to the outbox in slot order (with their direction
//      class), and the stayers found past the final count fill the holes movers left below it
//      (ascending order on both sides);
//   4. flush the J tile x 1/V with one pass of global FP64 atomics (the destructor, :201-213).
// This file is compiled with -ffp-contract=off: interpolation, push and direct deposition are pica's
// arithmetic in pica's order, so positions and momenta agree with pica to the last bit given the same
// fields, and a particle's direct currents do; the order in which they are summed into J (atomics) is
// free.  Esirkepov's currents, which pica does not have, are rounded as esk_stay, esk_change and
// esk_window below evaluate them (nearer to the exact ones than the sum over old and new shape: of a
// staying TSC particle 1.3e-16 of its currents against 2.8e-15, of a CIC one 8e-17 against 1.2e-16).
#include "pk_internal.h"

namespace {

constexpr int WAVES = PK_BLOCK / 64;

// y- and x-strides (doubles) of the field and J tiles of a 4^3 supercell.  A row stride of 12 puts the 16 cells
// of an x plane on the 16 double-wide bank pairs (rows at 0, 12, 24 = 8, 36 = 4 of them), where the natural 7 and 8
// overlap; 80 and 96 are the next x-strides that keep every x plane on the same pattern.  128^3 x 16 ppc, TSC,
// Esirkepov kernel: 2.68 ms, with natural rows padded by 4 per plane 2.94 ms.
constexpr int ISY4 = 12, ISX4 = 80, DSY4 = 12, DSX4 = 96;

struct ScGeom {
    double inv[3], no[3], nos[3], nom[3];
    int ibase[3], its[3], dbase[3], dts[3];
    int isx, isy, itn, dsx, dsy, dtn;      // strides and size of one component's field and J tile
};

// NC == 4: 4^3 supercells (constant strides); NC == 0: any shape, with the strides of `flat`'s levels
template <int SHAPE, int DEP, int NC>
__device__ __forceinline__ void sc_geom(const GridView<double>& g, const EnsGeom& eg, FlatLevels flat, const int sidx[3], ScGeom& q)
{
#pragma unroll
    for (int d = 0; d < 3; d++) {
        const double step = g.step[d];
        const double scMin = (double)(sidx[d] * eg.ncps[d]) * step;
        q.inv[d] = 1.0 / step;
        q.no[d] = (scMin - step) / step;                 // FieldInterpolatorYeeGrid.h:201
        q.nos[d] = q.no[d] + 0.5;                        // :202
        q.nom[d] = (scMin - 2.0 * step) / step;
        const int base = (int)(scMin / step) + 1;       // :205
        q.ibase[d] = base;
        const int n = NC ? NC : eg.ncps[d];
        q.its[d] = n + (SHAPE == PK_CIC ? 2 : 3);
        if (SHAPE == PK_CIC && DEP == PK_DIRECT) {
            q.dbase[d] = base;                           // CurrentDepositorYeeGrid.h:185-186
            q.dts[d] = n + 3;
        } else {
            q.dbase[d] = base - 1;
            q.dts[d] = n + 4;
        }
    }
    q.isy = NC == 4 ? ISY4 : pk_flat_row(flat.field, q.its[2]);
    q.isx = NC == 4 ? ISX4 : pk_flat_plane(flat.field, q.its[1], q.isy, eg.ncps[1], 16, 0);
    q.itn = q.its[0] * q.isx;
    q.dsy = NC == 4 ? DSY4 : pk_flat_row(flat.j, q.dts[2]);
    q.dsx = NC == 4 ? DSX4 : pk_flat_plane(flat.j, q.dts[1], q.dsy, eg.ncps[1], 16, 0);
    q.dtn = q.dts[0] * q.dsx;
}

// E/J_x collocated in x; E/J_y in y; E/J_z in z; B_x staggered only in x, etc.
// (FieldInterpolatorYeeGrid.h:155-166)
__device__ __forceinline__ bool colloc(int comp, int d)
{
    // bit d of the mask of component comp
    const unsigned m[6] = {1u, 2u, 4u, 6u, 5u, 3u};
    return (m[comp] >> d) & 1u;
}

// pica's 8-point CIC sum, term order of FieldInterpolatorYeeGrid.h:273-280; t is the first node
__device__ __forceinline__ double cic8(const double* t, int sx, int sy, const double c[3])
{
    return t[0] * (1.0 - c[0]) * (1.0 - c[1]) * (1.0 - c[2]) +
           t[1] * (1.0 - c[0]) * (1.0 - c[1]) * c[2] +
           t[sy] * (1.0 - c[0]) * c[1] * (1.0 - c[2]) +
           t[sy + 1] * (1.0 - c[0]) * c[1] * c[2] +
           t[sx] * c[0] * (1.0 - c[1]) * (1.0 - c[2]) +
           t[sx + 1] * c[0] * (1.0 - c[1]) * c[2] +
           t[sx + sy] * c[0] * c[1] * (1.0 - c[2]) +
           t[sx + sy + 1] * c[0] * c[1] * c[2];
}

// pica's 8-point CIC scatter, CurrentDepositorYeeGrid.h:254-261, into LDS with atomics
__device__ __forceinline__ void cic8_add(double* t, int sx, int sy, const double c[3], double v)
{
    atomicAdd(&t[0], (1.0 - c[0]) * (1.0 - c[1]) * (1.0 - c[2]) * v);
    atomicAdd(&t[1], (1.0 - c[0]) * (1.0 - c[1]) * c[2] * v);
    atomicAdd(&t[sy], (1.0 - c[0]) * c[1] * (1.0 - c[2]) * v);
    atomicAdd(&t[sy + 1], (1.0 - c[0]) * c[1] * c[2] * v);
    atomicAdd(&t[sx], c[0] * (1.0 - c[1]) * (1.0 - c[2]) * v);
    atomicAdd(&t[sx + 1], c[0] * (1.0 - c[1]) * c[2] * v);
    atomicAdd(&t[sx + sy], c[0] * c[1] * (1.0 - c[2]) * v);
    atomicAdd(&t[sx + sy + 1], c[0] * c[1] * c[2] * v);
}

__device__ __forceinline__ void tsc_w(double d, double w[3])
{
    const double a = 0.5 - d, b = 0.5 + d;
    w[0] = 0.5 * a * a;
    w[1] = 0.75 - d * d;
    w[2] = 0.5 * b * b;
}

// nearest node i0 of xi; weights on i0-1..i0+1; returns i0-1
__device__ __forceinline__ int tsc_node(double xi, double w[3])
{
    const int i0 = (int)floor(xi + 0.5);
    tsc_w(xi - (double)i0, w);
    return i0 - 1;
}

__device__ __forceinline__ double tsc27(const double* t, int sx, int sy, const double w[3][3])
{
    double sa = 0.0;
#pragma unroll
    for (int a = 0; a < 3; a++) {
        double sb = 0.0;
#pragma unroll
        for (int bb = 0; bb < 3; bb++) {
            double sc = 0.0;
#pragma unroll
            for (int c = 0; c < 3; c++) sc += w[2][c] * t[a * sx + bb * sy + c];
            sb += w[1][bb] * sc;
        }
        sa += w[0][a] * sb;
    }
    return sa;
}

__device__ __forceinline__ void tsc27_add(double* t, int sx, int sy, const double w[3][3], double v)
{
#pragma unroll
    for (int a = 0; a < 3; a++)
#pragma unroll
        for (int bb = 0; bb < 3; bb++)
#pragma unroll
            for (int c = 0; c < 3; c++)
                atomicAdd(&t[a * sx + bb * sy + c], w[0][a] * w[1][bb] * w[2][c] * v);
}

__device__ __forceinline__ bool in_tile(const int b[3], int span, const int ts[3])
{
    return b[0] >= 0 && b[0] + span <= ts[0] && b[1] >= 0 && b[1] + span <= ts[1] && b[2] >= 0 &&
           b[2] + span <= ts[2];
}

template <int SHAPE>
__device__ __forceinline__ bool interp(const ScGeom& q, const double* tile, const double x[3], double e[3], double b[3])
{
    const int tn = q.itn;
    if (SHAPE == PK_CIC) {
        int ic[3], is[3];
        double cc[3], cs[3];
#pragma unroll
        for (int d = 0; d < 3; d++) {               // getIndexCoeff, :257-267
            const double np = x[d] * q.inv[d];
            double internal = np - q.no[d];
            ic[d] = (int)internal;
            cc[d] = internal - (double)ic[d];
            internal = np - q.nos[d];
            is[d] = (int)internal;
            cs[d] = internal - (double)is[d];
        }
        bool ok = true;
#pragma unroll
        for (int comp = 0; comp < 6; comp++) {
            int bi[3];
            double c[3];
#pragma unroll
            for (int d = 0; d < 3; d++) {
                bi[d] = colloc(comp, d) ? ic[d] : is[d];
                c[d] = colloc(comp, d) ? cc[d] : cs[d];
            }
            ok = ok && in_tile(bi, 2, q.its);
            const double v = ok ? cic8(tile + comp * tn + bi[0] * q.isx + bi[1] * q.isy + bi[2], q.isx, q.isy, c) : 0.0;
            if (comp < 3) e[comp] = v; else b[comp - 3] = v;
        }
        return ok;
    } else {
        int nc[3], ns[3];
        double wc[3][3], ws[3][3];
#pragma unroll
        for (int d = 0; d < 3; d++) {
            const double np = x[d] * q.inv[d];
            nc[d] = tsc_node(np - q.no[d], wc[d]);
            ns[d] = tsc_node(np - q.nos[d], ws[d]);
        }
        bool ok = true;
#pragma unroll
        for (int comp = 0; comp < 6; comp++) {
            int bi[3];
            double w[3][3];
#pragma unroll
            for (int d = 0; d < 3; d++) {
                const bool col = colloc(comp, d);
                bi[d] = col ? nc[d] : ns[d];
#pragma unroll
                for (int k = 0; k < 3; k++) w[d][k] = col ? wc[d][k] : ws[d][k];
            }
            ok = ok && in_tile(bi, 3, q.its);
            const double v = ok ? tsc27(tile + comp * tn + bi[0] * q.isx + bi[1] * q.isy + bi[2], q.isx, q.isy, w) : 0.0;
            if (comp < 3) e[comp] = v; else b[comp - 3] = v;
        }
        return ok;
    }
}

// BorisPusher::push (BorisPusher.h:32-47) with ParticleRef::setP / getVelocity
// (ParticleArray.h:209,257-263); returns v
__device__ __forceinline__ void boris(double coeff, double dt, const double e[3], const double b[3], double u[3],
                                      double x[3], double v[3])
{
    double eM[3], um[3], t[3], up[3], s[3], cr[3];
#pragma unroll
    for (int d = 0; d < 3; d++) eM[d] = e[d] * coeff;
#pragma unroll
    for (int d = 0; d < 3; d++) um[d] = u[d] + eM[d];
    const double um2 = um[0] * um[0] + um[1] * um[1] + um[2] * um[2];
    const double tk = coeff / sqrt(1.0 + um2);
#pragma unroll
    for (int d = 0; d < 3; d++) t[d] = b[d] * tk;
    cr[0] = um[1] * t[2] - um[2] * t[1];
    cr[1] = um[2] * t[0] - um[0] * t[2];
    cr[2] = um[0] * t[1] - um[1] * t[0];
#pragma unroll
    for (int d = 0; d < 3; d++) up[d] = um[d] + cr[d];
    const double t2 = t[0] * t[0] + t[1] * t[1] + t[2] * t[2];
    const double sk = 2.0 / (1.0 + t2);
#pragma unroll
    for (int d = 0; d < 3; d++) s[d] = t[d] * sk;
    cr[0] = up[1] * s[2] - up[2] * s[1];
    cr[1] = up[2] * s[0] - up[0] * s[2];
    cr[2] = up[0] * s[1] - up[1] * s[0];
#pragma unroll
    for (int d = 0; d < 3; d++) u[d] = um[d] + cr[d] + eM[d];
    const double u2 = u[0] * u[0] + u[1] * u[1] + u[2] * u[2];
    const double invGamma = 1.0 / sqrt(1.0 + u2);
#pragma unroll
    for (int d = 0; d < 3; d++) v[d] = u[d] * PK_C * invGamma;
#pragma unroll
    for (int d = 0; d < 3; d++) x[d] = x[d] + v[d] * dt;
}

template <int SHAPE>
__device__ __forceinline__ bool deposit_direct(const ScGeom& q, double* jt, const double x[3], const double cur[3])
{
    const int tn = q.dtn;
    if (SHAPE == PK_CIC) {
        int ic[3], is[3];
        double cc[3], cs[3];
#pragma unroll
        for (int d = 0; d < 3; d++) {               // CurrentDepositorYeeGrid.h:239-249
            const double np = x[d] * q.inv[d];
            double internal = np - q.no[d];
            ic[d] = (int)internal;
            cc[d] = internal - (double)ic[d];
            internal = np - q.nos[d];
            is[d] = (int)internal;
            cs[d] = internal - (double)is[d];
        }
        bool ok = true;
#pragma unroll
        for (int comp = 0; comp < 3; comp++) {
            int bi[3];
            double c[3];
#pragma unroll
            for (int d = 0; d < 3; d++) {
                bi[d] = colloc(comp, d) ? ic[d] : is[d];
                c[d] = colloc(comp, d) ? cc[d] : cs[d];
            }
            ok = ok && in_tile(bi, 2, q.dts);
        }
        if (!ok) return false;
#pragma unroll
        for (int comp = 0; comp < 3; comp++) {
            int bi[3];
            double c[3];
#pragma unroll
            for (int d = 0; d < 3; d++) {
                bi[d] = colloc(comp, d) ? ic[d] : is[d];
                c[d] = colloc(comp, d) ? cc[d] : cs[d];
            }
            cic8_add(jt + comp * tn + bi[0] * q.dsx + bi[1] * q.dsy + bi[2], q.dsx, q.dsy, c, cur[comp]);
        }
        return true;
    } else {
        int nc[3], ns[3];
        double wc[3][3], ws[3][3];
#pragma unroll
        for (int d = 0; d < 3; d++) {
            const double np = x[d] * q.inv[d];
            nc[d] = tsc_node(np - q.nom[d], wc[d]);
            ns[d] = tsc_node(np - (q.nom[d] + 0.5), ws[d]);
        }
        bool ok = true;
#pragma unroll
        for (int comp = 0; comp < 3; comp++) {
            int bi[3];
#pragma unroll
            for (int d = 0; d < 3; d++) bi[d] = colloc(comp, d) ? nc[d] : ns[d];
            ok = ok && in_tile(bi, 3, q.dts);
        }
        if (!ok) return false;
#pragma unroll
        for (int comp = 0; comp < 3; comp++) {
            int bi[3];
            double w[3][3];
#pragma unroll
            for (int d = 0; d < 3; d++) {
                const bool col = colloc(comp, d);
                bi[d] = col ? nc[d] : ns[d];
#pragma unroll
                for (int k = 0; k < 3; k++) w[d][k] = col ? wc[d][k] : ws[d][k];
            }
            tsc27_add(jt + comp * tn + bi[0] * q.dsx + bi[1] * q.dsy + bi[2], q.dsx, q.dsy, w, cur[comp]);
        }
        return true;
    }
}

// ---- Esirkepov (CPC 135 (2001) 144) deposition of a particle moving x0 -> x1 with charge qw.
// With M = (S0 + S1) / 2 and DS = S1 - S0 the decomposition's weight of a transverse node pair is
//   S0_1 S0_2 + DS_1 S0_2 / 2 + S0_1 DS_2 / 2 + DS_1 DS_2 / 3 = M_1 M_2 + DS_1 DS_2 / 12,
// and a particle whose lowest node stays has closed forms in the middle m of its move and its length:
// TSC, around the nearest node: M = (1/2 - m)^2 / 2 + d^2 / 8, 3/4 - m^2 - d^2 / 4, (1/2 + m)^2 / 2 + d^2 / 8,
// DS = d (m - 1/2), -2 m d, d (m + 1/2), currents through its two faces ~ d (1/2 - m), d (1/2 + m);
// CIC: M = 1 - m, m, DS = -d, d, one face ~ d.
// So a staying particle takes 54 (TSC) or 12 (CIC) LDS atomics on its own window.  One that changes node
// takes the 4- or 3-node window of old and new shape.  Where few of a wavefront's 64 change, each waits in its
// lane's registers until four do (or its lane meets another), and is then deposited by 16 lanes, one per
// transverse node pair.  Four of them cost 44 LDS shuffles, so from ESK_MANY changers of the 64 on each is
// deposited by its own lane at once.
// 128^3 x 16 ppc two-stream plasma, whole kernel: TSC 3.82 -> 2.68 ms, CIC 2.06 -> 1.65 ms against adding every
// particle's 4- (3-) node window, of which 3% of the particles need more than 3 (2) nodes a side; with the
// changers in a workgroup queue instead of registers 2.84 ms (its pass after the push waits at a barrier).
// Hot plasmas, 64^3 x 16 ppc, thermal u = 0.1, 0.3 and 2: TSC 444, 513, 593 us (16 lanes each always: 440, 580, 801;
// every particle's window by its lane: 598, 638, 691), CIC 231, 248, 266 us (238, 330, 476; 282, 287, 303).
// ESK_MANY 50% higher: TSC 447, 573, 596, CIC 239, 247, 270 us.
template <int SHAPE>
constexpr int ESK_MANY = SHAPE == PK_CIC ? 8 : 16;

// lowest node of the shape at cell-centre coordinate xi, and the offset its closed form takes: from the
// nearest node (TSC) or from the lower one (CIC)
template <int SHAPE>
__device__ __forceinline__ int esk_node(double xi, double& d)
{
    const double c = SHAPE == PK_CIC ? floor(xi) : floor(xi + 0.5);
    d = xi - c;
    return (int)c - (SHAPE == PK_CIC ? 0 : 1);
}

// the shape at distance r
template <int SHAPE>
__device__ __forceinline__ double esk_shape(double r)
{
    if (SHAPE == PK_CIC) return r < 1.0 ? 1.0 - r : 0.0;
    const double t = 1.5 - r;
    return r < 0.5 ? 0.75 - r * r : r < 1.5 ? 0.5 * t * t : 0.0;
}

// deposits a staying particle; -1: its window leaves the tile (nothing deposited), 1: it changes node in
// some dimension and is left to esk_change, 0: done
template <int SHAPE>
__device__ __forceinline__ int esk_stay(const ScGeom& q, double* jt, const double x0[3], const double x1[3], double qw,
                                        const double hdt[3])
{
    constexpr int KW = SHAPE == PK_CIC ? 3 : 4, K = SHAPE == PK_CIC ? 2 : 3;
    double m[3], dl[3];
    int w[3], change = 0;
#pragma unroll
    for (int d = 0; d < 3; d++) {
        const double off = q.nom[d] + 0.5;
        double d0, d1;
        const int a0 = esk_node<SHAPE>(x0[d] * q.inv[d] - off, d0), a1 = esk_node<SHAPE>(x1[d] * q.inv[d] - off, d1);
        w[d] = a0 < a1 ? a0 : a1;
        if (a0 - w[d] > 1 || a1 - w[d] > 1 || w[d] < 0 || w[d] + KW > q.dts[d]) return -1;
        change |= a0 ^ a1;
        m[d] = 0.5 * (d0 + d1);
        dl[d] = d1 - d0;
    }
    if (change) return 1;
    double M[3][K], D[3][K];
#pragma unroll
    for (int d = 0; d < 3; d++) {
        if (SHAPE == PK_CIC) {
            M[d][0] = 1.0 - m[d];
            M[d][1] = m[d];
            D[d][0] = -dl[d];
            D[d][1] = dl[d];
        } else {
            const double lo = 0.5 - m[d], hi = 0.5 + m[d], d8 = 0.125 * dl[d] * dl[d];
            M[d][0] = fma(0.5 * lo, lo, d8);
            M[d][1] = fma(-m[d], m[d], 0.75) - 2.0 * d8;
            M[d][K - 1] = fma(0.5 * hi, hi, d8);
            D[d][0] = -dl[d] * lo;
            D[d][1] = -2.0 * m[d] * dl[d];
            D[d][K - 1] = dl[d] * hi;
        }
    }
    const int st[3] = {q.dsx, q.dsy, 1};
    double* t0 = jt + w[0] * q.dsx + w[1] * q.dsy + w[2];
#pragma unroll
    for (int comp = 0; comp < 3; comp++) {
        const int d1 = (comp + 1) % 3, d2 = (comp + 2) % 3;
        const double k = qw * hdt[comp];
        const double f0 = -k * D[comp][0], f1 = k * D[comp][K - 1];      // CIC: one face, f0
        double* t = t0 + comp * q.dtn + st[comp];
#pragma unroll
        for (int p = 0; p < K; p++) {
            const double dp = (1.0 / 12.0) * D[d1][p];
#pragma unroll
            for (int r = 0; r < K; r++) {
                const double g = fma(M[d1][p], M[d2][r], dp * D[d2][r]);
                atomicAdd(&t[p * st[d1] + r * st[d2]], f0 * g);
                if (SHAPE == PK_TSC) atomicAdd(&t[st[comp] + p * st[d1] + r * st[d2]], f1 * g);
            }
        }
    }
    return 0;
}

// deposits a particle on the window of its old and new shape (a node changer)
template <int SHAPE>
__device__ __forceinline__ void esk_window(const ScGeom& q, double* jt, const double x0[3], const double x1[3], double qw,
                                           const double hdt[3])
{
    constexpr int KW = SHAPE == PK_CIC ? 3 : 4;
    double M[3][KW], D[3][KW];
    int w[3];
#pragma unroll
    for (int d = 0; d < 3; d++) {
        const double off = q.nom[d] + 0.5;
        double d0, d1, s0[3], s1[3];
        const int a0 = esk_node<SHAPE>(x0[d] * q.inv[d] - off, d0), a1 = esk_node<SHAPE>(x1[d] * q.inv[d] - off, d1);
        if (SHAPE == PK_CIC) {
            s0[0] = 1.0 - d0; s0[1] = d0;
            s1[0] = 1.0 - d1; s1[1] = d1;
        } else {
            tsc_w(d0, s0);
            tsc_w(d1, s1);
        }
        w[d] = a0 < a1 ? a0 : a1;
#pragma unroll
        for (int k = 0; k < KW; k++) {
            const double a = a0 > a1 ? (k ? s0[k - 1] : 0.0) : (k < KW - 1 ? s0[k] : 0.0);
            const double b = a1 > a0 ? (k ? s1[k - 1] : 0.0) : (k < KW - 1 ? s1[k] : 0.0);
            M[d][k] = 0.5 * (a + b);
            D[d][k] = b - a;
        }
    }
    const int st[3] = {q.dsx, q.dsy, 1};
    double* t0 = jt + w[0] * q.dsx + w[1] * q.dsy + w[2];
#pragma unroll
    for (int comp = 0; comp < 3; comp++) {
        const int d1 = (comp + 1) % 3, d2 = (comp + 2) % 3;
        double cum[KW - 1];
#pragma unroll
        for (int a = 0; a < KW - 1; a++) cum[a] = -qw * hdt[comp] * D[comp][a] + (a ? cum[a - 1] : 0.0);
        double* t = t0 + comp * q.dtn + st[comp];
#pragma unroll
        for (int p = 0; p < KW; p++) {
            const double dp = (1.0 / 12.0) * D[d1][p];
#pragma unroll
            for (int r = 0; r < KW; r++) {
                const double g = fma(M[d1][p], M[d2][r], dp * D[d2][r]);
                if (g == 0.0) continue;      // a node pair that only a change in these dimensions reaches
#pragma unroll
                for (int a = 0; a < KW - 1; a++) atomicAdd(&t[a * st[comp] + p * st[d1] + r * st[d2]], cum[a] * g);
            }
        }
    }
}

// a node changer by 16 lanes (every lane of the wavefront takes part; has = the lanes hold one): lane
// (p, r) of them adds the transverse node pair (p, r) of every component.  Each lane evaluates its node p
// of every dimension; node r's values come from the lane of the same four that holds it.
template <int SHAPE>
__device__ __forceinline__ void esk_change(const ScGeom& q, double* jt, bool has, const double x0[3], const double x1[3],
                                           double qw, const double hdt[3])
{
    constexpr int KW = SHAPE == PK_CIC ? 3 : 4;
    const int lane = threadIdx.x & 63, p = lane & 3, r = (lane >> 2) & 3, four = lane & ~3;
    double M[3], D[3], Mr[3], Dr[3], cum[3][KW - 1];
    int w[3];
#pragma unroll
    for (int d = 0; d < 3; d++) {
        const double off = q.nom[d] + 0.5, xi0 = x0[d] * q.inv[d] - off, xi1 = x1[d] * q.inv[d] - off;
        double e;
        const int a0 = esk_node<SHAPE>(xi0, e), a1 = esk_node<SHAPE>(xi1, e);
        w[d] = a0 < a1 ? a0 : a1;
        const double node = (double)(w[d] + p);
        const double s0 = esk_shape<SHAPE>(fabs(xi0 - node)), s1 = esk_shape<SHAPE>(fabs(xi1 - node));
        M[d] = 0.5 * (s0 + s1);
        D[d] = s1 - s0;
        Mr[d] = __shfl(M[d], four | r);
        Dr[d] = __shfl(D[d], four | r);
#pragma unroll
        for (int a = 0; a < KW - 1; a++) cum[d][a] = __shfl(D[d], four | a) + (a ? cum[d][a - 1] : 0.0);
    }
    if (!has || p >= KW || r >= KW) return;
    const int st[3] = {q.dsx, q.dsy, 1};
    double* t0 = jt + w[0] * q.dsx + w[1] * q.dsy + w[2];
#pragma unroll
    for (int comp = 0; comp < 3; comp++) {
        const int d1 = (comp + 1) % 3, d2 = (comp + 2) % 3;
        const double k = -qw * hdt[comp];
        const double g = k * fma(M[d1], Mr[d2], (1.0 / 12.0) * D[d1] * Dr[d2]);
        double* t = t0 + comp * q.dtn + st[comp] + p * st[d1] + r * st[d2];
#pragma unroll
        for (int a = 0; a < KW - 1; a++) atomicAdd(&t[a * st[comp]], cum[comp][a] * g);
    }
}

struct StepParams {
    double dt, coeff, q;
    double L[3], scinv[3], hdt[3];
    int mask_words;
    FlatLevels flat;
};

// all arguments of one ensemble's particle step (one kernel argument, or one entry of a batch)
struct F64Args {
    GridView<double> g;
    EnsGeom eg;
    PartF64 pm, po;
    uint8_t* odir;
    const int64_t* off;
    const int32_t* cnt;
    int32_t *nstay, *nmove, *mvc, *flags;
    StepParams sp;
};


template <int SHAPE, int DEP, int NC>
__global__ void __launch_bounds__(PK_BLOCK) k_particles(GridView<double> g, EnsGeom eg, PartF64 pm, PartF64 po,
                                                        uint8_t* __restrict__ odir, const int64_t* __restrict__ off,
                                                        const int32_t* __restrict__ cnt, int32_t* __restrict__ nstay,
                                                        int32_t* __restrict__ nmove, int32_t* __restrict__ mvc,
                                                        int32_t* __restrict__ flags, StepParams sp)
{
    const long s = pk_xcd_supercell(blockIdx.x, eg.xcd_chunk);
    if (s >= eg.nsct) return;
#include "pk_particles_f64_body.inc"
}

// many ensembles: a list of (ensemble, supercell) items; gridDim.x < nitems makes it persistent.  At least three
// wavefronts a SIMD with Esirkepov: the compiler takes 176 VGPRs for TSC otherwise, and two (64 plasmas of 16^3 to
// 32^3 cells at 4 and 8 ppc, a step: 1049 us with two, 877 us with three, which need no spill)
template <int SHAPE, int DEP, int NC>
__global__ void __launch_bounds__(PK_BLOCK, DEP == PK_ESIRKEPOV ? 3 : 1) k_particles_batch(const F64Args* __restrict__ jobs,
                                                              const int2* __restrict__ items, long nitems,
                                                              const int* __restrict__ halt)
{
    if (halt[PK_HALT_STOP]) return;
    for (long w = blockIdx.x; w < nitems; w += gridDim.x) {
        __syncthreads();
        const int2 it = items[w];
        const long s = it.y;
        const F64Args& A = jobs[it.x];      // arguments read in place (a copy would live in scratch)
        const GridView<double>& g = A.g;
        const EnsGeom& eg = A.eg;
        const PartF64& pm = A.pm;
        const PartF64& po = A.po;
        uint8_t* __restrict__ odir = A.odir;
        const int64_t* __restrict__ off = A.off;
        const int32_t* __restrict__ cnt = A.cnt;
        int32_t* __restrict__ nstay = A.nstay;
        int32_t* __restrict__ nmove = A.nmove;
        int32_t* __restrict__ mvc = A.mvc;
        int32_t* __restrict__ flags = A.flags;
        const StepParams& sp = A.sp;
#include "pk_particles_f64_body.inc"
    }
}

size_t f64_lds(const pk_ens* e, bool c4, int shape, int dep, int mask_words, FlatLevels flat);

StepParams step_params(const pk_ens* e, double dt, int shape, int dep)
{
    StepParams sp;
    sp.dt = dt;
    const double q = e->ctx->charge[e->type], m = e->ctx->mass[e->type];
    sp.coeff = q * dt / (2.0 * m * PK_C);        // BorisPusher.h:29
    sp.q = q;
    for (int d = 0; d < 3; d++) {
        sp.L[d] = (double)e->ncell[d] * e->step[d];
        const double cellSize = (sp.L[d] - 0.0) / (double)e->ncell[d];      // EnsembleSupercells.h:31-33
        sp.scinv[d] = 1.0 / ((double)e->ncps[d] * cellSize);
        sp.hdt[d] = e->step[d] / dt;
    }
    sp.mask_words = (e->maxcap + PK_BLOCK + 63) / 64 + 1;
    sp.flat = FlatLevels{0, 0};
    if (e->ncps[2] == 1)
        sp.flat = pk_flat_levels([&](FlatLevels f) { return f64_lds(e, false, shape, dep, sp.mask_words, f); },
                                 shape == PK_CIC && dep == PK_DIRECT ? 4 : 3, shape == PK_TSC);
    return sp;
}

// 4^3 supercells have their own kernels: their tile strides are constants, so that the 162 field reads and
// the deposits' atomics of a particle take one base address and immediate offsets (CIC direct at 128^3 x 16 ppc:
// 1.38 ms against 1.54 ms with strides read at run time)
bool cube4(const pk_ens* e) { return e->ncps[0] == 4 && e->ncps[1] == 4 && e->ncps[2] == 4; }

// dynamic LDS of k_particles (c4: its form for 4^3 supercells): field and J tiles, mover mask, counters, mask prefix
size_t f64_lds(const pk_ens* e, bool c4, int shape, int dep, int mask_words, FlatLevels flat)
{
    int its[3], dts[3];
    for (int d = 0; d < 3; d++) {
        its[d] = e->ncps[d] + (shape == PK_CIC ? 2 : 3);
        dts[d] = e->ncps[d] + ((shape == PK_CIC && dep == PK_DIRECT) ? 3 : 4);
    }
    const size_t ip = pk_flat_plane(flat.field, its[1], pk_flat_row(flat.field, its[2]), e->ncps[1], 16, 0);
    const size_t dp = pk_flat_plane(flat.j, dts[1], pk_flat_row(flat.j, dts[2]), e->ncps[1], 16, 0);
    const size_t tiles = 6 * its[0] * (c4 ? (size_t)ISX4 : ip) + 3 * dts[0] * (c4 ? (size_t)DSX4 : dp);
    return sizeof(double) * tiles + sizeof(uint64_t) * mask_words + sizeof(int) * 32 + sizeof(long) * (mask_words + 1) + 16;
}

F64Args f64_args(pk_ens* e, pk_grid* g, const EnsGeom& eg, const StepParams& sp)
{
    F64Args A;
    A.g = grid_view<double>(g);
    A.eg = eg;
    A.pm = part_f64(e, e->main);
    A.po = part_f64(e, e->outbox);
    A.odir = e->odir;
    A.off = e->off;
    A.cnt = e->cnt;
    A.nstay = e->nstay;
    A.nmove = e->nmove;
    A.mvc = e->mvc;
    A.flags = e->flags;
    A.sp = sp;
    return A;
}

template <int SHAPE, int DEP, int NC>
int launch(pk_ens* e, pk_grid* g, double dt)
{
    EnsGeom eg = ens_geom(e);
    const StepParams sp = step_params(e, dt, SHAPE, DEP);
    const size_t lds = f64_lds(e, NC == 4, SHAPE, DEP, sp.mask_words, sp.flat);
    if (lds > 160 * 1024)
        return pk_fail(e->ctx, PK_E_CAPACITY, "particle step: supercell too large for LDS");
    const unsigned nblocks = (unsigned)(PK_XCD * (long)eg.xcd_chunk);
    const F64Args A = f64_args(e, g, eg, sp);
    pk_ktimer tm(e->ctx, "particles");
    hipLaunchKernelGGL((k_particles<SHAPE, DEP, NC>), dim3(nblocks), dim3(PK_BLOCK), lds, e->ctx->stream, A.g, A.eg, A.pm,
                       A.po, A.odir, A.off, A.cnt, A.nstay, A.nmove, A.mvc, A.flags, A.sp);
    PK_HIP(e->ctx, hipGetLastError());
    return PK_OK;
}

// the items of one form factor (SHAPE) in one launch
template <int SHAPE, int DEP, int NC>
int batch_go(pk_batch* b, bool prepare)
{
    const void* fn = (const void*)k_particles_batch<SHAPE, DEP, NC>;
    const size_t lds = b->cplds[SHAPE];
    const long nitems = b->cnitems[SHAPE];
    if (nitems == 0) return PK_OK;
    if (prepare) {
        PK_HIP(b->ctx, hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        return PK_OK;
    }
    const long wg = b->knob[PK_BATCH_WG_PER_CU];
    const long nb = wg > 0 && wg * 256 < nitems ? wg * 256 : nitems;
    hipLaunchKernelGGL((k_particles_batch<SHAPE, DEP, NC>), dim3((unsigned)nb), dim3(PK_BLOCK), lds, b->ctx->stream,
                       (const F64Args*)b->pjobs, b->citems[SHAPE], nitems, b->halt);
    PK_HIP(b->ctx, hipGetLastError());
    return PK_OK;
}

template <int SHAPE, int DEP>
int launch_nc(pk_ens* e, pk_grid* g, double dt)
{
    return cube4(e) ? launch<SHAPE, DEP, 4>(e, g, dt) : launch<SHAPE, DEP, 0>(e, g, dt);
}

template <int SHAPE, int DEP>
int batch_go_nc(pk_batch* b, bool prepare)
{
    return pk_batch_cube(b) == 4 ? batch_go<SHAPE, DEP, 4>(b, prepare) : batch_go<SHAPE, DEP, 0>(b, prepare);
}

// every form factor present, one launch each
int batch_dispatch(pk_batch* b, int dep, bool prepare)
{
    int r;
    if (dep == PK_DIRECT) {
        if ((r = batch_go_nc<PK_CIC, PK_DIRECT>(b, prepare))) return r;
        return batch_go_nc<PK_TSC, PK_DIRECT>(b, prepare);
    }
    if (dep == PK_ESIRKEPOV) {
        if ((r = batch_go_nc<PK_CIC, PK_ESIRKEPOV>(b, prepare))) return r;
        return batch_go_nc<PK_TSC, PK_ESIRKEPOV>(b, prepare);
    }
    return pk_fail(b->ctx, PK_E_ARG, "particle step: unknown depositor");
}

}  // namespace

int pk_particles_f64(pk_ens* e, pk_grid* g, double dt, int shape, int dep)
{
    if (shape == PK_CIC && dep == PK_DIRECT) return launch_nc<PK_CIC, PK_DIRECT>(e, g, dt);
    if (shape == PK_CIC && dep == PK_ESIRKEPOV) return launch_nc<PK_CIC, PK_ESIRKEPOV>(e, g, dt);
    if (shape == PK_TSC && dep == PK_DIRECT) return launch_nc<PK_TSC, PK_DIRECT>(e, g, dt);
    if (shape == PK_TSC && dep == PK_ESIRKEPOV) return launch_nc<PK_TSC, PK_ESIRKEPOV>(e, g, dt);
    return pk_fail(e->ctx, PK_E_ARG, "particle step: unknown shape/depositor");
}

int pk_batch_f64_prepare(pk_batch* b, double dt, int shape, int dep)
{
    const int n = b->n();
    std::vector<F64Args> jobs(n);
    const bool c4 = pk_batch_cube(b) == 4;
    b->cplds[0] = b->cplds[1] = 0;
    for (int i = 0; i < n; i++) {
        pk_ens* e = b->ens[i];
        const int sh = pk_batch_shape_of(b, i, shape);
        const StepParams sp = step_params(e, dt, sh, dep);
        jobs[i] = f64_args(e, b->grids[i], ens_geom(e), sp);
        const size_t l = f64_lds(e, c4, sh, dep, sp.mask_words, sp.flat);
        if (l > b->cplds[sh]) b->cplds[sh] = l;
    }
    if (b->cplds[0] > 160 * 1024 || b->cplds[1] > 160 * 1024)
        return pk_fail(b->ctx, PK_E_CAPACITY, "particle step: supercell too large for LDS");
    if (int r = pk_batch_upload(b, &b->pjobs, jobs.data(), sizeof(F64Args) * n)) return r;
    return batch_dispatch(b, dep, true);
}

int pk_batch_f64_launch(pk_batch* b, int dep) { return batch_dispatch(b, dep, false); }
