// ALE layer-transport kernels (gfx950): the producer of the advection step's layer fluxes, all FP64 in the
// reference's per-element arithmetic (no contraction, IEEE divisions), so results are bit-identical.
//
//   transport velocity   u^θ and the free-surface flux Q_bt per face column   (core/vertical/ale.py:789-808)
//   transport thickness  q_e / q_w, the donor layer cut at the shallower bed  (core/vertical/ale.py:168-199)
//   PPM edges            limited slopes + positive-definite parabola per cell (core/vertical/ale.py:578-623)
//   PPM flux             swept-volume mean thickness, a Newton correction du per face column with the global stop
//                        of the reference, then the residual share             (core/vertical/ale.py:626-740)
//   outflow limiter      outflow > content check, cut, give-back passes       (core/vertical/ale.py:299-437)
//   Lagrangian step      h† = h - Δt ∇·Q / A, emptied-layer check, V0, V1, ok (core/vertical/ale.py:278-295)
//
// Faces of one direction are addressed in their natural layout: AX 0 the u-faces (n, ny, nx+1), AX 1 the v-faces
// (n, ny+1, nx).  A face column (a, f) is face f along the flux axis in row (AX 0) or column (AX 1) a; threads
// take face columns with the unit-stride index fastest, so every layer's loads are coalesced.  Each thread loops
// over the layers from the bed up, which is the order of every sum over k in the reference.
#pragma once
#include <float.h>

#include <type_traits>

#include "ocx_weno.hpp"

namespace ocx {
namespace ale {

constexpr double H_PPM_MIN = 2e-10;   // positive-definite floor of the PPM thickness [m] (core/vertical/ale.py:298)

// Python's min(a, b) / max(a, b) on floats: the first argument unless the second compares smaller / larger
__device__ __forceinline__ double amin(double a, double b) { return b < a ? b : a; }
__device__ __forceinline__ double amax(double a, double b) { return b > a ? b : a; }

// numpy.nan_to_num: NaN -> 0, +-inf -> +-largest finite
__device__ __forceinline__ double nan0(double x) {
    if (x != x) return 0.0;
    if (x == __builtin_inf()) return DBL_MAX;
    if (x == -__builtin_inf()) return -DBL_MAX;
    return x;
}

// numpy.minimum: the smaller, NaN if either is NaN
__device__ __forceinline__ double npmin(double a, double b) {
    if (a != a) return a;
    if (b != b) return b;
    return b < a ? b : a;
}

// numpy.maximum: the larger, NaN if either is NaN
__device__ __forceinline__ double npmax(double a, double b) {
    if (a != a) return a;
    if (b != b) return b;
    return b > a ? b : a;
}

// numpy.sign: -1, 0 (of the zero's sign) or 1; NaN stays NaN
__device__ __forceinline__ double sgn(double x) { return x > 0.0 ? 1.0 : (x < 0.0 ? -1.0 : x * 0.0); }

template <int AX>
struct Geo {
    int n, ny, nx;
    __host__ __device__ __forceinline__ int ncell() const { return AX == 0 ? nx : ny; }           // cells along the flux axis
    __host__ __device__ __forceinline__ long long cols() const {                                    // face columns
        return AX == 0 ? (long long)ny * (nx + 1) : (long long)(ny + 1) * nx;
    }
    __host__ __device__ __forceinline__ size_t pc() const { return (size_t)ny * nx; }               // cell plane
    __host__ __device__ __forceinline__ size_t pf() const { return (size_t)cols(); }                // face plane
    __host__ __device__ __forceinline__ void col(long long t, int& a, int& f) const {
        if (AX == 0) {
            a = (int)(t / (nx + 1));
            f = (int)(t - (long long)a * (nx + 1));
        } else {
            f = (int)(t / nx);
            a = (int)(t - (long long)f * nx);
        }
    }
    __host__ __device__ __forceinline__ size_t cell(int a, int c) const {
        return AX == 0 ? (size_t)a * nx + c : (size_t)c * nx + a;
    }
    __host__ __device__ __forceinline__ size_t face(int a, int f) const {
        return AX == 0 ? (size_t)a * (nx + 1) + f : (size_t)f * nx + a;
    }
};

// layers whose loads a column's thread issues together
constexpr int KB = 8;

__device__ __forceinline__ long long gtid() { return (long long)blockIdx.x * blockDim.x + threadIdx.x; }

// one lane per wave with `bad` set ORs 1 into *flag (a vector atomic)
__device__ __forceinline__ void wave_flag(bool bad, unsigned* flag) {
    const unsigned long long b = __ballot(bad);
    if (b && (threadIdx.x & 63) == (unsigned)(__ffsll((long long)b) - 1)) atomicOr(flag, 1u);
}

// ------------------------------------------------------------------------------------------ transport velocity
// u (n, M) columns; last_wet (M) bytes; w (n, M); L, D (M).  ut (n, M), Qb (M).  Columns of TV_MIN to TV_MAX layers.
//
// A workgroup holds 64 columns; its TV_W wavefronts share the layers, every one of them TV_L layers in registers, all
// loads in flight together, so that the column is read once (32 B a cell-layer with the result; a thread that walks
// its column twice fetched 54) and a small grid does not wait at every layer.  The sums run from the bed up as the
// reference adds: the products go to LDS as [layer][column] and one wavefront per sum adds them in order.  Layers
// w, w + TV_W, ... belong to wavefront w.  Dynamic LDS: 2 n * 64 doubles.  198 x 159 x 50 42 -> 17 us a direction,
// 384 x 384 x 50 79 -> 72.  Below TV_MIN layers the wavefronts have too little to share (us, shared / one thread a column:
// 1024 x 1024 1 layer 36 / 16, 3 layers 39 / 24, 5 48 / 45, 8 74 / 70, 10 89 / 87, 12 95 / 112, 20 145 / 202; 2000 x 2000
// 1 layer 127 / 34, 8 274 / 260, 10 309 / 327; grids up to 384 x 384 are level below 12 layers).
constexpr int TV_W = 4, TV_L = 16, TV_MIN = 10, TV_MAX = TV_W * TV_L;
__global__ __launch_bounds__(64 * TV_W) void k_transport_velocity(
    const double* __restrict__ u_new, const double* __restrict__ u_old, const uint8_t* __restrict__ last_wet,
    const double* __restrict__ w, const double* __restrict__ L, const double* __restrict__ D, double theta,
    double theta_bc, int n, long long M, double* __restrict__ ut, double* __restrict__ Qb) {
    extern __shared__ double tv_lds[];
    double* s1 = tv_lds;
    double* s0 = tv_lds + (size_t)n * 64;
    const int lane = threadIdx.x & 63, wv = wave_id();
    const long long p0 = block_id() * 64 + lane, p = p0 < M ? p0 : M - 1;
    const bool wet = last_wet[p] != 0;
    double un[TV_L], uo[TV_L], ww[TV_L];
#pragma unroll
    for (int q = 0; q < TV_L; ++q) {
        const int k = wv + q * TV_W;
        if (k < n) {
            const size_t x = (size_t)k * M + p;
            un[q] = u_new[x];
            ww[q] = w[x];
            uo[q] = wet ? u_old[x] : 0.0;
        }
    }
#pragma unroll
    for (int q = 0; q < TV_L; ++q) {
        const int k = wv + q * TV_W;
        if (k < n) {
            s1[k * 64 + lane] = ww[q] * un[q];
            s0[k * 64 + lane] = ww[q] * uo[q];
        }
    }
    __syncthreads();
    double m = 0.0;
    if (wv < 2) {
        const double* t = (wv == 0 ? s1 : s0) + lane;
        for (int k = 0; k < n; ++k) m += t[k * 64];
    }
    __syncthreads();
    if (wv < 2) tv_lds[wv * 64 + lane] = m;
    __syncthreads();
    const double d = (theta - theta_bc) * (tv_lds[lane] - tv_lds[64 + lane]);
    const double omt = 1.0 - theta_bc;
    __syncthreads();
#pragma unroll
    for (int q = 0; q < TV_L; ++q) {
        const int k = wv + q * TV_W;
        if (k < n) {
            const double v = theta_bc * un[q] + omt * uo[q] + d;
            if (p0 < M) ut[(size_t)k * M + p] = v;
            s1[k * 64 + lane] = ww[q] * v;
        }
    }
    __syncthreads();
    if (wv != 0 || p0 >= M) return;
    double s = 0.0;
    for (int k = 0; k < n; ++k) s += s1[k * 64 + lane];
    Qb[p] = L[p] * D[p] * s;
}

// The same for shorter and deeper columns: one thread per column, two walks over its layers.
__global__ void k_transport_velocity_walk(const double* __restrict__ u_new, const double* __restrict__ u_old,
                                          const uint8_t* __restrict__ last_wet, const double* __restrict__ w,
                                          const double* __restrict__ L, const double* __restrict__ D, double theta,
                                          double theta_bc, int n, long long M, double* __restrict__ ut,
                                          double* __restrict__ Qb) {
    const long long p = gtid();
    if (p >= M) return;
    const bool wet = last_wet[p] != 0;
    double m1 = 0.0, m0 = 0.0;
    for (int k = 0; k < n; ++k) {
        const size_t x = (size_t)k * M + p;
        const double un = wet ? u_old[x] : 0.0;
        m1 += w[x] * u_new[x];
        m0 += w[x] * un;
    }
    const double d = (theta - theta_bc) * (m1 - m0);
    const double omt = 1.0 - theta_bc;
    double s = 0.0;
    for (int k = 0; k < n; ++k) {
        const size_t x = (size_t)k * M + p;
        const double un = wet ? u_old[x] : 0.0;
        const double v = theta_bc * u_new[x] + omt * un + d;
        ut[x] = v;
        s += w[x] * v;
    }
    Qb[p] = L[p] * D[p] * s;
}

// ------------------------------------------------------------------------------------------ transport thickness
// q_e: from the low-side cell (flow towards +), q_w: from the high-side cell; the domain-edge faces use the inner
// cell, closed faces are 0.  clip: only the part of the donor layer above the shallower bed passes.
// NB layers' loads are in flight, the last one repeated beyond n: KB, and 1 (fewer registers) below KB / 2 layers (us, 1
// / KB: 2000 x 2000 1 layer 25 / 44, 3 layers 74 / 98, 4 103 / 112, 5 156 / 123, 8 304 / 215; 1024 x 1024 2 layers 14 /
// 18, 4 22 / 22, 8 54 / 44, 50 771 / 647; 198 x 159 x 50 23 / 18; up to 600 x 600 level below 5 layers).
template <int AX, int NB>
__global__ void k_face_thickness(const double* __restrict__ h, const double* __restrict__ H,
                                 const uint8_t* __restrict__ act, int clip, Geo<AX> g, double* __restrict__ qe,
                                 double* __restrict__ qw) {
    const long long t = gtid();
    if (t >= g.cols()) return;
    int a, f;
    g.col(t, a, f);
    const int nc = g.ncell();
    const size_t cw = g.cell(a, f > 0 ? f - 1 : 0), ce = g.cell(a, f < nc ? f : nc - 1);
    const size_t fo = g.face(a, f), PC = g.pc(), PF = g.pf();
    if (!(act[cw] && act[ce])) {
        for (int k = 0; k < g.n; ++k) {
            qe[k * PF + fo] = 0.0;
            qw[k * PF + fo] = 0.0;
        }
        return;
    }
    if (clip) {
        double Hw = H[cw], He = H[ce];
        Hw = Hw == Hw ? Hw : 0.0;
        He = He == He ? He : 0.0;
        const double z_bed = amax(-Hw, -He);
        double sw = 0.0, se = 0.0;
        for (int k = 0; k < g.n; k += NB) {
            double hw[NB], he[NB];
#pragma unroll
            for (int q = 0; q < NB; ++q) {
                const size_t x = (size_t)min(k + q, g.n - 1) * PC;
                hw[q] = h[x + cw];
                he[q] = h[x + ce];
            }
#pragma unroll
            for (int q = 0; q < NB; ++q) {
                if (k + q < g.n) {
                    const double a0 = hw[q] == hw[q] ? hw[q] : 0.0, a1 = he[q] == he[q] ? he[q] : 0.0;
                    sw += a0;
                    se += a1;
                    qe[(k + q) * PF + fo] = amin(a0, amax(0.0, (-Hw + sw) - z_bed));
                    qw[(k + q) * PF + fo] = amin(a1, amax(0.0, (-He + se) - z_bed));
                }
            }
        }
    } else {
        for (int k = 0; k < g.n; ++k) {
            const double hw = h[k * PC + cw], he = h[k * PC + ce];
            qe[k * PF + fo] = hw == hw ? hw : 0.0;
            qw[k * PF + fo] = he == he ? he : 0.0;
        }
    }
}

// ------------------------------------------------------------------------------------------ PPM edges
// limited slope of a cell from its neighbours' values (already the cell itself where the neighbour is land or
// outside) and its masks
__device__ __forceinline__ double ppm_slope(double hm1, double hc, double hp1, double mw, double me, double m) {
    double s = 0.5 * (hp1 - hm1);
    const double dmx = amax(amax(hp1, hm1), hc) - hc;
    const double dmn = hc - amin(amin(hp1, hm1), hc);
    const double a = amin(fabs(s), 2.0 * amin(dmx, dmn));
    s = s > 0.0 ? a : (s < 0.0 ? -a : 0.0);
    return mw * me * m > 0.0 ? s : 0.0;
}

// one thread per cell (natural index j * nx + i) and every gridDim.y-th layer, which no result of another layer enters:
// with all layers in one thread a small grid was one long chain of loads per wavefront (198 x 159 x 50: 78-110 us a
// direction -> 21).  The layers are split only as far as that gives EDGE_WAVES wavefronts, and into slices of at least
// EDGE_LAYERS layers: each slice reads the masks again and the layers in flight spread over memory (us, 1 / 2 / 4 / 13
// slices: 384 x 384 x 50 110 / 78 / 68 / 62, 512 x 512 x 50 167 / 131 / 131 / 135, 724 x 724 x 50 258 / 258 / 259 / 271,
// 1024 x 1024 x 50 504 / 510 / 512 / 528, 2000 x 2000 x 20 762 / 767 / 792 / 949).  The thickness is read as the flux
// passes it: inactive cells 0, NaN 0.  Edges: lo = the low-index (west / south) edge, hi = the high one.
constexpr int EDGE_LAYERS = 4;
constexpr long long EDGE_WAVES = 24576;
template <int AX>
__global__ void k_ppm_edges(const double* __restrict__ h, const uint8_t* __restrict__ act, double h_min, Geo<AX> g,
                            double* __restrict__ e_lo, double* __restrict__ e_hi) {
    const long long t = gtid();
    const size_t PC = g.pc();
    if (t >= (long long)PC) return;
    const int nx = g.nx;
    const int a = AX == 0 ? (int)(t / nx) : (int)(t % nx);
    const int c = AX == 0 ? (int)(t % nx) : (int)(t / nx);
    const int nc = g.ncell();
    // the five cells c-2 .. c+2 along the axis (clamped indices; existence flags decide)
    size_t o[5];
    bool ex[5];
    double m[5];
    for (int d = 0; d < 5; ++d) {
        const int cc = c + d - 2;
        ex[d] = cc >= 0 && cc < nc;
        o[d] = g.cell(a, ex[d] ? cc : c);
        m[d] = ex[d] && act[o[d]] ? 1.0 : 0.0;
    }
    const double r6 = 1.0 / 6.0;
    for (int k = (int)blockIdx.y; k < g.n; k += (int)gridDim.y) {
        double v[5];
        for (int d = 0; d < 5; ++d) v[d] = m[d] != 0.0 ? nan0(h[k * PC + o[d]]) : 0.0;
        // hm1 / hp1 / slope of the cell at offset d (1..3) with its neighbours d-1, d+1
        double hm1[5], hp1[5], slp[5];
        for (int d = 1; d <= 3; ++d) {
            const bool lo_ex = ex[d - 1], hi_ex = ex[d + 1];      // cell d has a low / high neighbour
            const double mw = lo_ex ? m[d - 1] : 0.0, me = hi_ex ? m[d + 1] : 0.0;
            hm1[d] = lo_ex ? mw * v[d - 1] + (1.0 - mw) * v[d] : v[d];
            hp1[d] = hi_ex ? me * v[d + 1] + (1.0 - me) * v[d] : v[d];
            slp[d] = ex[d] ? ppm_slope(hm1[d], v[d], hp1[d], mw, me, m[d]) : 0.0;
        }
        const double hc = v[2];
        const double sw = ex[1] ? slp[1] : 0.0, se = ex[3] ? slp[3] : 0.0;
        const double hw = 0.5 * (hm1[2] + hc) + div_const(sw - slp[2], 6.0, r6);
        const double he = 0.5 * (hp1[2] + hc) + div_const(slp[2] - se, 6.0, r6);
        const double curv = 3.0 * ((hw + he) - 2.0 * hc);
        const double dh = he - hw;
        const bool inside = curv > 0.0 && fabs(dh) < curv;
        double ow, oe;
        if (inside && hc <= h_min) {
            ow = hc;
            oe = hc;
        } else {
            double sc = 1.0;
            if (inside) {
                const double num = 12.0 * curv * (hc - h_min);
                const double den = curv * curv + 3.0 * dh * dh;
                if (num < den) sc = num / den;
            }
            ow = hc + sc * (hw - hc);
            oe = hc + sc * (he - hc);
        }
        e_lo[k * PC + t] = ow;
        e_hi[k * PC + t] = oe;
    }
}

// ------------------------------------------------------------------------------------------ PPM flux
template <int AX>
struct PpmArgs {
    const double *h, *e_lo, *e_hi, *ut, *L, *Qb, *qe, *qw, *dxt;
    const uint8_t* act;
    double dt;
    Geo<AX> g;
    double *du, *lo, *hi, *err, *dsum;   // state per face column
    unsigned* notconv;                   // notconv[m]: some column unconverged after iteration m
    double* hist;                        // du after each iteration of the last bundle (k_ppm_bundle), bundle x columns
    double* out;
    int single, bundle;                  // iterations with a launch of their own, and iterations in each launch after those
};

// the face column's geometry: donor cells on both sides and their widths
struct Column {
    size_t cw, ce, fo;
    double dxw, dxe, Lf, Qb;
    Recip rw, re;            // reciprocals of the widths (qdiv_r gives the IEEE quotient)
    bool open;
};

template <int AX>
__device__ __forceinline__ Column column(const PpmArgs<AX>& p, long long t) {
    Column c;
    int a, f;
    p.g.col(t, a, f);
    const int nc = p.g.ncell();
    c.cw = p.g.cell(a, f > 0 ? f - 1 : 0);
    c.ce = p.g.cell(a, f < nc ? f : nc - 1);
    c.fo = p.g.face(a, f);
    c.dxw = p.dxt[c.cw];
    c.dxe = p.dxt[c.ce];
    c.rw = recip_of(c.dxw);
    c.re = recip_of(c.dxe);
    c.Lf = p.L[c.fo];
    c.Qb = p.Qb[c.fo];
    c.open = p.act[c.cw] && p.act[c.ce];
    return c;
}

// The sums over the layers of a face column run from the bed up, in one chain of additions as the reference adds;
// everything before the additions is independent from layer to layer.  So a workgroup holds 64 face columns and its
// PPM_W wavefronts share the layers of a chunk, PPM_L each, with the loads of those layers in flight together; the
// terms go to LDS as [layer][column], and one wavefront per sum adds them in order while the others load the next
// chunk (two buffers, one barrier a chunk).  With one thread for a whole column a small grid had fewer wavefronts than
// SIMDs and waited twice per layer (198 x 159 x 50: a Newton pass 53 us -> 13, the fluxes 90 -> 26; 384 x 384 x 50: 90 -> 54
// and 155 -> 106; 1024 x 1024 x 50, where both stream, the whole transport 14.3 -> 12.4 ms).
constexpr int PPM_W = 4, PPM_L = 4, PPM_C = PPM_W * PPM_L;

// terms of the layers k .. k + NL - 1 (beyond n: repeated, not added): F and dF/du at velocity u^theta + du: the
// swept mean thickness of the donor parabola over the Courant fraction, capped by the transport thickness where that
// is below the donor layer.  u: the velocities u^theta of these layers.
template <int AX, int NL = PPM_L>
__device__ __forceinline__ void layer_fluxes(const PpmArgs<AX>& p, const Column& c, int k, const double* u, double* F,
                                             double* dF) {
    const size_t PC = p.g.pc(), PF = p.g.pf();
    double hu[NL], ww[NL], ee[NL], qq[NL];
#pragma unroll
    for (int q = 0; q < NL; ++q) {
        const size_t kk = (size_t)min(k + q, p.g.n - 1);
        const bool pos = u[q] >= 0.0;
        const size_t ci = kk * PC + (pos ? c.cw : c.ce);
        hu[q] = p.h[ci];
        ww[q] = p.e_lo[ci];
        ee[q] = p.e_hi[ci];
        qq[q] = (pos ? p.qe : p.qw)[kk * PF + c.fo];
    }
#pragma unroll
    for (int q = 0; q < NL; ++q) {
        const bool pos = u[q] >= 0.0;
        const double cr = amin(qdiv_r(fabs(u[q]) * p.dt, pos ? c.rw : c.re), 1.0);
        const double h0 = nan0(hu[q]);
        const double curv3 = (ww[q] + ee[q]) - 2.0 * h0;
        const double dh = pos ? ww[q] - ee[q] : ee[q] - ww[q];
        const double edge = pos ? ee[q] : ww[q];
        double mean = edge + cr * (0.5 * dh + curv3 * (cr - 1.5));
        double marg = edge + cr * (dh + 3.0 * curv3 * (cr - 1.0));
        if (qq[q] < h0) {
            mean = amin(mean, qq[q]);
            marg = amin(marg, qq[q]);
        }
        F[q] = c.Lf * u[q] * amax(mean, 0.0);
        dF[q] = c.Lf * amax(marg, 0.0);
    }
}

// adds the terms of layers [0, m) of one LDS chunk, in order
__device__ __forceinline__ double add_layers(double s, const double* t, int m) {
    if (m >= PPM_C) {
#pragma unroll
        for (int l = 0; l < PPM_C; ++l) s += t[l * 64];
    } else {
        for (int l = 0; l < m; ++l) s += t[l * 64];
    }
    return s;
}

// Newton state of a face column, and the step to the next du (bracketing bisection)
struct Newton {
    double du, lo, hi, err, dsum;
};
__device__ __forceinline__ void newton_step(Newton& s) {
    if (s.err > 0.0) s.hi = s.du;
    if (s.err < 0.0) s.lo = s.du;
    const double step = s.dsum > 0.0 ? -s.err / s.dsum : 0.0;
    double nw = s.du + step;
    if (step > 0.0 && nw >= s.hi) nw = 0.5 * (s.du + s.hi);
    if (step < 0.0 && nw <= s.lo) nw = 0.5 * (s.du + s.lo);
    s.du = nw;
}

// The column's sums of F (wavefront 0) and dF/du (wavefront 1) at u^theta + du.  Every wavefront of the workgroup calls
// it; sF, sD: two chunks each.
template <int AX>
__device__ __forceinline__ double column_sum(const PpmArgs<AX>& p, const Column& c, double du, int lane, int wv,
                                             double (*sF)[PPM_C * 64], double (*sD)[PPM_C * 64]) {
    const size_t PF = p.g.pf();
    const int n = p.g.n;
    double sum = 0.0;
    for (int kc = 0, b = 0; kc < n; kc += PPM_C, b ^= 1) {
        const int k = kc + wv * PPM_L;
        if (c.open) {
            double u[PPM_L], F[PPM_L], dF[PPM_L];
#pragma unroll
            for (int q = 0; q < PPM_L; ++q) u[q] = p.ut[(size_t)min(k + q, n - 1) * PF + c.fo];
#pragma unroll
            for (int q = 0; q < PPM_L; ++q) u[q] = u[q] + du;
            layer_fluxes(p, c, k, u, F, dF);
#pragma unroll
            for (int q = 0; q < PPM_L; ++q) {
                sF[b][(wv * PPM_L + q) * 64 + lane] = F[q];
                sD[b][(wv * PPM_L + q) * 64 + lane] = dF[q];
            }
        }
        __syncthreads();
        if (c.open) {
            if (wv == 0) sum = add_layers(sum, sF[b] + lane, n - kc);
            if (wv == 1) sum = add_layers(sum, sD[b] + lane, n - kc);
        }
    }
    return sum;
}

// INIT: the CFL bracket [lo, hi] of du and the uncorrected column sums (the reference evaluates at u^theta itself);
// block 0 also clears the convergence flags of the passes to come (m of them).
// Otherwise Newton iteration m (0-based) with bracketing bisection; runs only while the previous iteration left some
// column unconverged (every column iterates until all have converged, as the reference).
// Block 64 * PPM_W threads for 64 face columns.
template <int AX, bool INIT>
__global__ __launch_bounds__(64 * PPM_W) void k_ppm_pass(PpmArgs<AX> p, int m) {
    if (!INIT && m > 0 && p.notconv[m - 1] == 0u) return;
    __shared__ double sF[2][PPM_C * 64], sD[2][PPM_C * 64];
    const int lane = threadIdx.x & 63, wv = wave_id();
    if (INIT && block_id() == 0)
        for (int q = threadIdx.x; q < m; q += 64 * PPM_W) p.notconv[q] = 0u;
    const long long t0 = block_id() * 64 + lane;
    const bool in = t0 < p.g.cols();
    const long long t = in ? t0 : p.g.cols() - 1;
    const Column c = column(p, t);
    const size_t PF = p.g.pf();
    const int n = p.g.n;
    const double limw = 0.5 * c.dxw / p.dt, lime = 0.5 * c.dxe / p.dt;
    Newton s{0.0, 0.0, 0.0, 0.0, 0.0};
    double sum = 0.0;                       // wavefront 0: of F, 1: of dF/du
    if constexpr (INIT) {
        double mnw = __builtin_inf(), mxe = -__builtin_inf();
        for (int kc = 0, b = 0; kc < n; kc += PPM_C, b ^= 1) {
            const int k = kc + wv * PPM_L;
            double u[PPM_L], F[PPM_L], dF[PPM_L];
#pragma unroll
            for (int q = 0; q < PPM_L; ++q) u[q] = p.ut[(size_t)min(k + q, n - 1) * PF + c.fo];
#pragma unroll
            for (int q = 0; q < PPM_L; ++q) {          // (a repeated last layer changes no minimum or maximum)
                mnw = amin(mnw, limw - u[q]);
                mxe = amax(mxe, -(lime + u[q]));
            }
            if (c.open) {
                layer_fluxes(p, c, k, u, F, dF);
#pragma unroll
                for (int q = 0; q < PPM_L; ++q) {
                    sF[b][(wv * PPM_L + q) * 64 + lane] = F[q];
                    sD[b][(wv * PPM_L + q) * 64 + lane] = dF[q];
                }
            }
            __syncthreads();
            if (c.open) {
                if (wv == 0) sum = add_layers(sum, sF[b] + lane, n - kc);
                if (wv == 1) sum = add_layers(sum, sD[b] + lane, n - kc);
            }
        }
        // the wavefronts' brackets meet in LDS (the chunk buffers: every sum is done behind the barrier)
        __syncthreads();
        sF[0][wv * 64 + lane] = mnw;
        sD[0][wv * 64 + lane] = mxe;
        __syncthreads();
        if (wv == 0) {
            for (int q = 1; q < PPM_W; ++q) {
                mnw = amin(mnw, sF[0][q * 64 + lane]);
                mxe = amax(mxe, sD[0][q * 64 + lane]);
            }
            s.hi = amax(amin(limw, mnw), 0.0);
            s.lo = amin(amax(-lime, mxe), 0.0);
        }
    } else {
        s = Newton{p.du[t], p.lo[t], p.hi[t], p.err[t], p.dsum[t]};
        newton_step(s);
        sum = column_sum(p, c, s.du, lane, wv, sF, sD);
    }
    if (wv == 1 && in) p.dsum[t] = sum;
    if (wv == 0) {
        const double er = sum - c.Qb;
        if (in) {
            p.du[t] = s.du;
            p.hi[t] = s.hi;
            p.lo[t] = s.lo;
            p.err[t] = er;
        }
        if (!INIT) wave_flag(in && fabs(er) > 1e-12 * amax(fabs(c.Qb), 1.0), p.notconv + m);
    }
}

// The same with all layers of a column in one thread, PPM_L of them in flight, then the rest one by one, for short
// columns and for grids that fill the chip (ppm_walks has the line and both sides); state and results as k_ppm_pass.
template <int AX, bool INIT>
__global__ __launch_bounds__(256) void k_ppm_walk(PpmArgs<AX> p, int m) {
    if (!INIT && m > 0 && p.notconv[m - 1] == 0u) return;
    const long long t = gtid();
    if (INIT && blockIdx.x == 0)
        for (int q = threadIdx.x; q < m; q += 256) p.notconv[q] = 0u;
    bool bad = false;
    if (t < p.g.cols()) {
        const Column c = column(p, t);
        const size_t PF = p.g.pf();
        const int n = p.g.n;
        const double limw = 0.5 * c.dxw / p.dt, lime = 0.5 * c.dxe / p.dt;
        double mnw = __builtin_inf(), mxe = -__builtin_inf();
        Newton s{0.0, 0.0, 0.0, 0.0, 0.0};
        if constexpr (!INIT) {
            s = Newton{p.du[t], p.lo[t], p.hi[t], p.err[t], p.dsum[t]};
            newton_step(s);
        }
        double sum = 0.0, dsum = 0.0;
        auto layers = [&](auto count, int k) {
            constexpr int NL = decltype(count)::value;
            double u[NL], F[NL], dF[NL];
#pragma unroll
            for (int q = 0; q < NL; ++q) u[q] = p.ut[(size_t)(k + q) * PF + c.fo];
#pragma unroll
            for (int q = 0; q < NL; ++q) {
                if constexpr (INIT) {
                    mnw = amin(mnw, limw - u[q]);
                    mxe = amax(mxe, -(lime + u[q]));
                } else {
                    u[q] = u[q] + s.du;
                }
            }
            if (!c.open) return;
            layer_fluxes<AX, NL>(p, c, k, u, F, dF);
#pragma unroll
            for (int q = 0; q < NL; ++q) {
                sum += F[q];
                dsum += dF[q];
            }
        };
        if (INIT || c.open) {
            int k = 0;
            for (; k + PPM_L <= n; k += PPM_L) layers(std::integral_constant<int, PPM_L>{}, k);
            for (; k < n; ++k) layers(std::integral_constant<int, 1>{}, k);
        }
        if constexpr (INIT) {
            s.hi = amax(amin(limw, mnw), 0.0);
            s.lo = amin(amax(-lime, mxe), 0.0);
        }
        const double er = sum - c.Qb;
        p.du[t] = s.du;
        p.hi[t] = s.hi;
        p.lo[t] = s.lo;
        p.err[t] = er;
        p.dsum[t] = dsum;
        bad = fabs(er) > 1e-12 * amax(fabs(c.Qb), 1.0);
    }
    if constexpr (!INIT) wave_flag(bad, p.notconv + m);
}

// The iterations m .. m + count - 1 (count <= p.bundle) in one launch, without a look at the other columns in between:
// du after each of them goes to hist, so that the fluxes can take the one after which all columns had converged.  4 to
// 6 iterations converge every column of the grids measured, and a launch with nothing to do costs 2 to 5 us, so of the
// usual 20 iterations only the first PPM_SINGLE have launches of their own: 799 us to 716 for a transport of 198 x 159
// x 50 with the other 12 in one bundle.  But a bundle in which all columns converge has iterated on for nothing, up to
// bundle - 1 times, and from some 1000 workgroups on that costs more than the launches: a field of 512 x 512 x 50 that
// takes 9 iterations took 2.59 ms a direction with a bundle of 12, and 1.71 before the layers were shared.  So a bundle
// has at most PPM_BUNDLE iterations and at most 8192 workgroup-iterations (ppm_bundle_of), and above 4096 workgroups
// every iteration has a launch of its own.
constexpr int PPM_SINGLE = 8, PPM_BUNDLE = 12;
template <int AX>
__global__ __launch_bounds__(64 * PPM_W) void k_ppm_bundle(PpmArgs<AX> p, int m, int count) {
    // nothing to do once an iteration before this bundle has converged everywhere (flags of iterations that were not
    // run are 0 too)
    for (int q = m > p.single ? m - p.bundle : m - 1; q < m; ++q)
        if (p.notconv[q] == 0u) return;
    __shared__ double sF[2][PPM_C * 64], sD[2][PPM_C * 64], sS[2][64];
    const int lane = threadIdx.x & 63, wv = wave_id();
    const long long t0 = block_id() * 64 + lane;
    const bool in = t0 < p.g.cols();
    const long long t = in ? t0 : p.g.cols() - 1;
    const Column c = column(p, t);
    Newton s{p.du[t], p.lo[t], p.hi[t], p.err[t], p.dsum[t]};
    for (int q = 0; q < count; ++q) {
        newton_step(s);
        const double sum = column_sum(p, c, s.du, lane, wv, sF, sD);
        if (wv < 2) sS[wv][lane] = sum;
        __syncthreads();
        s.err = sS[0][lane] - c.Qb;
        s.dsum = sS[1][lane];
        if (wv == 0) {
            if (in) p.hist[(size_t)q * p.g.cols() + t] = s.du;
            wave_flag(in && fabs(s.err) > 1e-12 * amax(fabs(c.Qb), 1.0), p.notconv + m + q);
        }
        __syncthreads();                    // sS and the chunk buffers are read: the next iteration may write them
    }
    if (wv == 0 && in) {
        p.du[t] = s.du;
        p.hi[t] = s.hi;
        p.lo[t] = s.lo;
        p.err[t] = s.err;
        p.dsum[t] = s.dsum;
    }
}

// du after the first iteration after which every column had converged, or the last: the state's, or the history's if a
// bundle converged before its end
template <int AX>
__device__ __forceinline__ double final_du(const PpmArgs<AX>& p, long long t, int max_iter) {
    int it = 0;
    while (it < max_iter - 1 && p.notconv[it] != 0u) ++it;
    return it < p.single ? p.du[t] : p.hist[(size_t)((it - p.single) % p.bundle) * p.g.cols() + t];
}

// the residual's side: its thicknesses and their sum (1 where no side has any)
template <int AX>
__device__ __forceinline__ const double* residual_side(const PpmArgs<AX>& p, double R, double te, double tw, Recip& den) {
    bool use_e = R >= 0.0;
    double tot = use_e ? te : tw;
    if (tot <= 0.0) {
        use_e = !use_e;
        tot = use_e ? te : tw;
    }
    den = recip_of(tot > 0.0 ? tot : 1.0);
    return use_e ? p.qe : p.qw;
}

// the layer fluxes at u^theta + du plus the residual R = Q_bt - sum F shared in proportion to the transport thickness
// on R's side (the other side's where that column is empty); closed faces 0.  The layers are shared by the wavefronts
// as in k_ppm_pass; the sums of F, q_e and q_w are added by one wavefront each.  max_iter: the iterations allowed.
template <int AX>
__global__ __launch_bounds__(64 * PPM_W) void k_ppm_final(PpmArgs<AX> p, int max_iter) {
    __shared__ double sT[2][3][PPM_C * 64];
    const int lane = threadIdx.x & 63, wv = wave_id();
    const long long t0 = block_id() * 64 + lane;
    const bool in = t0 < p.g.cols();
    const long long t = in ? t0 : p.g.cols() - 1;
    const Column c = column(p, t);
    const size_t PF = p.g.pf();
    const int n = p.g.n;
    const bool run = in && c.open;
    const double du = final_du(p, t, max_iter);
    double sum = 0.0;                       // wavefront 0: of F, 1: of q_e, 2: of q_w
    for (int kc = 0, b = 0; kc < n; kc += PPM_C, b ^= 1) {
        const int k = kc + wv * PPM_L;
        if (run) {
            double u[PPM_L], F[PPM_L], dF[PPM_L], qe[PPM_L], qw[PPM_L];
#pragma unroll
            for (int q = 0; q < PPM_L; ++q) {
                const size_t x = (size_t)min(k + q, n - 1) * PF + c.fo;
                u[q] = p.ut[x];
                qe[q] = p.qe[x];
                qw[q] = p.qw[x];
            }
#pragma unroll
            for (int q = 0; q < PPM_L; ++q) u[q] = u[q] + du;
            layer_fluxes(p, c, k, u, F, dF);
#pragma unroll
            for (int q = 0; q < PPM_L; ++q) {
                const int l = (wv * PPM_L + q) * 64 + lane;
                if (k + q < n) p.out[(size_t)(k + q) * PF + c.fo] = F[q];
                sT[b][0][l] = F[q];
                sT[b][1][l] = qe[q];
                sT[b][2][l] = qw[q];
            }
        } else if (in) {
#pragma unroll
            for (int q = 0; q < PPM_L; ++q)
                if (k + q < n) p.out[(size_t)(k + q) * PF + c.fo] = 0.0;
        }
        __syncthreads();
        if (run && wv < 3) sum = add_layers(sum, sT[b][wv] + lane, n - kc);
    }
    __syncthreads();                        // every sum is done: the buffer takes the three results
    if (wv < 3) sT[0][wv][lane] = sum;
    __syncthreads();
    if (!run) return;
    const double R = c.Qb - sT[0][0][lane], te = sT[0][1][lane], tw = sT[0][2][lane];
    Recip den;
    const double* q = residual_side(p, R, te, tw, den);
    for (int kc = wv * PPM_L; kc < n; kc += PPM_C) {
        double f[PPM_L], qk[PPM_L];
#pragma unroll
        for (int l = 0; l < PPM_L; ++l) {
            const size_t x = (size_t)min(kc + l, n - 1) * PF + c.fo;
            f[l] = kc + l < n ? p.out[x] : 0.0;
            qk[l] = q[x];
        }
#pragma unroll
        for (int l = 0; l < PPM_L; ++l)
            if (kc + l < n) p.out[(size_t)(kc + l) * PF + c.fo] = f[l] + qdiv_r(R * qk[l], den);
    }
}

// The same with all layers of a column in one thread.
template <int AX>
__global__ __launch_bounds__(256) void k_ppm_walk_final(PpmArgs<AX> p, int max_iter) {
    const long long t = gtid();
    if (t >= p.g.cols()) return;
    const Column c = column(p, t);
    const size_t PF = p.g.pf();
    const int n = p.g.n;
    if (!c.open) {
        for (int k = 0; k < n; ++k) p.out[(size_t)k * PF + c.fo] = 0.0;
        return;
    }
    const double du = final_du(p, t, max_iter);
    double sum = 0.0, te = 0.0, tw = 0.0;
    auto layers = [&](auto count, int k) {
        constexpr int NL = decltype(count)::value;
        double u[NL], F[NL], dF[NL], qe[NL], qw[NL];
#pragma unroll
        for (int q = 0; q < NL; ++q) {
            const size_t x = (size_t)(k + q) * PF + c.fo;
            u[q] = p.ut[x];
            qe[q] = p.qe[x];
            qw[q] = p.qw[x];
        }
#pragma unroll
        for (int q = 0; q < NL; ++q) u[q] = u[q] + du;
        layer_fluxes<AX, NL>(p, c, k, u, F, dF);
#pragma unroll
        for (int q = 0; q < NL; ++q) {
            p.out[(size_t)(k + q) * PF + c.fo] = F[q];
            sum += F[q];
            te += qe[q];
            tw += qw[q];
        }
    };
    int k = 0;
    for (; k + PPM_L <= n; k += PPM_L) layers(std::integral_constant<int, PPM_L>{}, k);
    for (; k < n; ++k) layers(std::integral_constant<int, 1>{}, k);
    const double R = c.Qb - sum;
    Recip den;
    const double* q = residual_side(p, R, te, tw, den);
    for (k = 0; k < n; ++k) {
        const size_t x = (size_t)k * PF + c.fo;
        p.out[x] = p.out[x] + qdiv_r(R * q[x], den);
    }
}

// ------------------------------------------------------------------------------------------ upwind thickness flux
// upwind_transport_x (core/vertical/ale.py:233-251), one thread per face column: F_k = L u_k q_k with the transport
// thickness of the side the water comes from, R = Q_bt - sum_k F_k, and R shared in proportion to the transport
// thicknesses on R's side (the other side where that column's sum is not positive).  The sums run from layer 0
// up and start from the first term, as NumPy's sum over the first axis does.  Face arrays are indexed by the face
// column t directly (t is the face's index in its layer plane for both axes).
template <int AX>
__global__ void k_upwind_transport(const double* __restrict__ ut, const double* __restrict__ L,
                                   const double* __restrict__ Qb, const double* __restrict__ qe,
                                   const double* __restrict__ qw, Geo<AX> g, double* __restrict__ out) {
    const long long t = gtid();
    if (t >= g.cols()) return;
    const size_t PF = g.pf();
    const double Lf = L[t];
    double s = 0.0, se = 0.0, sw = 0.0;
    for (int k = 0; k < g.n; ++k) {
        const size_t x = k * PF + t;
        const double u = ut[x], e = qe[x], w = qw[x];
        const double F = Lf * u * (u >= 0.0 ? e : w);
        out[x] = F;
        s = k == 0 ? F : s + F;
        se = k == 0 ? e : se + e;
        sw = k == 0 ? w : sw + w;
    }
    const double R = Qb[t] - s;
    bool use_e = R >= 0.0;
    if (!((use_e ? se : sw) > 0.0)) use_e = !use_e;
    const double tot = use_e ? se : sw;
    const double den = tot > 0.0 ? tot : 1.0;
    const double* q = use_e ? qe : qw;
    for (int k = 0; k < g.n; ++k) {
        const size_t x = k * PF + t;
        out[x] = out[x] + R * q[x] / den;
    }
}

// ------------------------------------------------------------------------------------------ open-edge faces
// open_face_transport (core/vertical/ale.py:841-861) on the m faces of one open edge, one thread per face: the
// layer fluxes (h_k / sum h) Q_bt + L h_k (tb u'_new + (1 - tb) u'_old) of the interior cell's thicknesses,
// written where the face depth D > 0 (open_boundary.py:350-351).  Every array is addressed by an offset, a layer
// stride and a face stride, so the four edges of the u- and v-face arrays share the kernel.
struct EdgeArgs {
    double* Q;                       // face fluxes
    const double *h, *un, *uo;       // interior cells; new and old velocities at the faces
    const double *D, *Qo, *L;        // one layer of faces
    long long q0, qk, qf;            // Q, un, uo: offset, layer stride, face stride
    long long h0, hk, hf;            // h
    long long f0, ff;                // D, Qo, L
    int n, m;
    double tb;
};

__global__ void k_open_face_transport(EdgeArgs e) {
    const long long f = gtid();
    if (f >= e.m) return;
    const long long fq = e.q0 + f * e.qf, fh = e.h0 + f * e.hf, fo = e.f0 + f * e.ff;
    if (!(e.D[fo] > 0.0)) return;
    double tot = 0.0;
    for (int k = 0; k < e.n; ++k) {
        const double hk = e.h[fh + k * e.hk];
        tot = k == 0 ? hk : tot + hk;
    }
    const bool wet = tot > 0.0;
    const double den = wet ? tot : 1.0;
    double sn = 0.0, so = 0.0;
    for (int k = 0; k < e.n; ++k) {
        const double w = wet ? e.h[fh + k * e.hk] / den : 0.0;
        const double an = w * e.un[fq + k * e.qk], ao = w * e.uo[fq + k * e.qk];
        sn = k == 0 ? an : sn + an;
        so = k == 0 ? ao : so + ao;
    }
    const double Qb = e.Qo[fo], Lf = e.L[fo], tb = e.tb;
    for (int k = 0; k < e.n; ++k) {
        const double hk = e.h[fh + k * e.hk];
        const double w = wet ? hk / den : 0.0;
        const double pn = e.un[fq + k * e.qk] - sn, po = e.uo[fq + k * e.qk] - so;
        const double q = w * Qb + Lf * hk * (tb * pn + (1.0 - tb) * po);
        e.Q[fq + k * e.qk] = wet ? q : 0.0;
    }
}

// ------------------------------------------------------------------------------------------ freshwater
// One lane per wavefront with `hit` set adds the wavefront's count of set lanes to *count (a vector atomic).
__device__ __forceinline__ void wave_count(bool hit, unsigned long long* count) {
    const unsigned long long b = __ballot(hit);
    if (b && (threadIdx.x & 63) == (unsigned)(__ffsll((long long)b) - 1))
        atomicAdd(count, (unsigned long long)__popcll(b));
}

// freshwater_volumes (core/components/freshwater.py:31-58), one thread per column of M: the volume scale dV joins
// the top layer; a removal that would take it below the floor is taken from the original layers top-down, first
// keeping each at the floor, then down to zero.  Columns where that happens are counted.  With area, the volumes
// out A are written to Vout as well (layer_volumes of the thicknesses).
__global__ void k_freshwater_volumes(const double* __restrict__ V, const double* __restrict__ dV, double scale,
                                     const double* __restrict__ floor_c, double floor_s,
                                     const double* __restrict__ area, int n, long long M, double* __restrict__ out,
                                     double* __restrict__ Vout, unsigned long long* count) {
    const long long c = gtid();
    bool spill = false;
    if (c < M) {
        const double d = scale * dV[c];
        const double fl = floor_c ? floor_c[c] : floor_s;
        for (int k = 0; k < n - 1; ++k) out[(size_t)k * M + c] = V[(size_t)k * M + c];
        const size_t top = (size_t)(n - 1) * M + c;
        const double vt = V[top] + d;
        out[top] = vt;
        spill = d < 0.0 && vt < fl;
        if (spill) {
            double deficit = -d;
            out[top] = V[top];
            for (int pass = 0; pass < 2; ++pass) {
                const double keep = pass == 0 ? fl : 0.0;
                for (int k = n - 1; k >= 0; --k) {
                    const size_t x = (size_t)k * M + c;
                    const double col = out[x];
                    const double take = npmin(deficit, npmax(col - keep, 0.0));
                    out[x] = col - take;
                    deficit = deficit - take;
                }
            }
        }
        if (Vout) {
            const double A = area[c];
            for (int k = 0; k < n; ++k) Vout[(size_t)k * M + c] = out[(size_t)k * M + c] * A;
        }
    }
    wave_count(spill, count);
}

// apply_freshwater (core/components/freshwater.py:61-122), one thread per column, in place on the stack (nt, n, M):
// every member but T (t_index) and T^2 (t2_index) takes c V_adv / V_fw where the column has freshwater; in a
// column whose volume changed below the top layer the touched layers (from the lowest changed one up) share
// sum V_adv c / sum V_fw.  var_surf (n, M), for member s_index: (V_fw S_new^2 - V_adv S_old^2) / dt where the
// column has freshwater, else 0.  The sums run from layer 0 up and start from the first term (NumPy's sum over
// the first axis).  Columns with a change below the top layer are counted.
struct FreshArgs {
    double* stack;
    const double *Va, *Vf, *fwa;
    double* var_surf;
    int nt, n, t_index, t2_index, s_index;
    long long M;
    double dt;
    unsigned long long* count;
};

__global__ void k_apply_freshwater(FreshArgs a) {
    const long long c = gtid();
    bool spill = false;
    if (c < a.M) {
        const int n = a.n;
        const long long M = a.M;
        const bool cols = a.fwa[c] != 0.0;
        int kmin = -1;
        for (int k = 0; k < n; ++k) {
            const bool ch = a.Va[(size_t)k * M + c] != a.Vf[(size_t)k * M + c];
            if (ch && kmin < 0) kmin = k;
            if (ch && k < n - 1) spill = true;
        }
        if (kmin < 0) kmin = 0;
        double vsum = 0.0;
        if (spill)
            for (int k = 0; k < n; ++k) {
                const double v = k >= kmin ? a.Vf[(size_t)k * M + c] : 0.0;
                vsum = k == 0 ? v : vsum + v;
            }
        const bool has_water = vsum > 0.0;
        for (int i = 0; i < a.nt; ++i) {
            if (i == a.t_index || i == a.t2_index) continue;
            double* st = a.stack + (size_t)i * n * M + c;
            double cbar = 0.0;
            if (spill) {
                double num = 0.0;
                for (int k = 0; k < n; ++k) {
                    const double v = k >= kmin ? a.Va[(size_t)k * M + c] * st[(size_t)k * M] : 0.0;
                    num = k == 0 ? v : num + v;
                }
                cbar = has_water ? num / vsum : 0.0;
            }
            for (int k = 0; k < n; ++k) {
                const size_t x = (size_t)k * M;
                const double va = a.Va[x + c], vf = a.Vf[x + c], s = st[x];
                const double ratio = (cols && vf > 0.0) ? va / vf : 1.0;
                double cv = cols ? s * ratio : s;
                if (spill && k >= kmin && has_water) cv = cbar;
                if (i == a.s_index && a.var_surf) a.var_surf[x + c] = cols ? (vf * (cv * cv) - va * (s * s)) / a.dt : 0.0;
                st[x] = cv;
            }
        }
    }
    wave_count(spill, a.count);
}

// ------------------------------------------------------------------------------------------ outflow limiter
struct OutArgs {
    const double *h, *area;
    const uint8_t* act;
    double *Qx, *Qy;
    int n, ny, nx;
    double dt, h_floor;
    double *r, *room;                    // (n, ny, nx)
    double* delta;                       // per face column of the current axis
    unsigned long long* count;           // cell-layers over the bound
    unsigned* wild;                      // some cell-layer's room0 is not finite
    unsigned long long* bad_face;        // first face of the current axis whose cut cannot be given back (linear
                                         // index), else ~0; bad_face[-1]: the u-faces' while the v-faces run
};

// Both axes of a pass run before the host looks at the flags.  The v-faces leave everything as it is where a u-face
// could not place its cut: the call then ends with that face, and Qy keeps what the passes before gave it.
template <int AX>
__device__ __forceinline__ bool pass_ended(const OutArgs& o) {
    return AX == 1 && o.bad_face[-1] != ~0ull;
}

// what a cell-layer can give in Δt, (h - h_floor)+ A / Δt with A = 0 on land
__device__ __forceinline__ double room0(const OutArgs& o, size_t x, size_t c) {
    const double A = o.act[c] ? o.area[c] : 0.0;
    return amax(o.h[x] - o.h_floor, 0.0) * A / o.dt;
}

// outgoing flux of cell-layer (k, j, i) over its four faces
__device__ __forceinline__ double outflow(const OutArgs& o, int k, int j, int i) {
    const size_t fx = ((size_t)k * o.ny + j) * (o.nx + 1) + i;
    const size_t fy = ((size_t)k * (o.ny + 1) + j) * o.nx + i;
    return amax(o.Qx[fx + 1], 0.0) - amin(o.Qx[fx], 0.0) + amax(o.Qy[fy + o.nx], 0.0) - amin(o.Qy[fy], 0.0);
}

// over = active & O > room0 x factor; r = room0 / O where over, else 1; counts the cells over
__global__ void k_out_over(OutArgs o, double factor, int first) {
    const long long t = gtid();
    const size_t PC = (size_t)o.ny * o.nx;
    bool over = false, wild = false;
    if (t < (long long)(PC * o.n)) {
        const int k = (int)(t / PC);
        const size_t c = (size_t)t - (size_t)k * PC;
        const int j = (int)(c / o.nx), i = (int)(c - (size_t)j * o.nx);
        const double O = outflow(o, k, j, i);
        const double r0 = room0(o, t, c);
        over = o.act[c] && (first ? O > r0 : O > r0 * factor);
        o.r[t] = over ? r0 / (O > 0.0 ? O : 1.0) : 1.0;
        wild = !(fabs(r0) <= DBL_MAX);
    }
    wave_flag(wild, o.wild);
    const unsigned long long b = __ballot(over);
    if (b && (threadIdx.x & 63) == (unsigned)(__ffsll((long long)b) - 1))
        atomicAdd(o.count, (unsigned long long)__popcll(b));
}

// room = room0 - outflow with the current Qx, Qy
__global__ void k_out_room(OutArgs o) {
    const long long t = gtid();
    const size_t PC = (size_t)o.ny * o.nx;
    if (t >= (long long)(PC * o.n)) return;
    const int k = (int)(t / PC);
    const size_t c = (size_t)t - (size_t)k * PC;
    const int j = (int)(c / o.nx), i = (int)(c - (size_t)j * o.nx);
    o.room[t] = room0(o, t, c) - outflow(o, k, j, i);
}

// the face arrays of one axis and the donor cells of face column (a, f): lo = the low-index side (the donor of
// flow towards +), hi = the high-index side; the edge faces take the cell across the wrap on a periodic axis
template <int AX>
struct OutFace {
    size_t fo, PF, clo, chi;
    bool has_lo, has_hi;
};

template <int AX>
__device__ __forceinline__ OutFace<AX> out_face(const OutArgs& o, long long t, int wrap) {
    Geo<AX> g{o.n, o.ny, o.nx};
    int a, f;
    g.col(t, a, f);
    const int nc = g.ncell();
    OutFace<AX> r;
    r.fo = g.face(a, f);
    r.PF = g.pf();
    r.has_lo = f > 0 || wrap;
    r.has_hi = f < nc || wrap;
    r.clo = g.cell(a, f > 0 ? f - 1 : nc - 1);
    r.chi = g.cell(a, f < nc ? f : 0);
    return r;
}

// cut every layer's flux by the ratio of its donor cell; delta = Σ_k (Q - Q_cut), the net cut of the face
template <int AX>
__global__ void k_out_cut(OutArgs o, int wrap) {
    const long long t = gtid();
    Geo<AX> g{o.n, o.ny, o.nx};
    if (t >= g.cols() || pass_ended<AX>(o)) return;
    const OutFace<AX> fc = out_face<AX>(o, t, wrap);
    double* Q = AX == 0 ? o.Qx : o.Qy;
    const size_t PC = g.pc();
    double d = 0.0;
    for (int k = 0; k < o.n; k += KB) {
        double q[KB], rlo[KB], rhi[KB];
#pragma unroll
        for (int l = 0; l < KB; ++l) {
            const size_t kk = (size_t)min(k + l, o.n - 1);
            q[l] = Q[kk * fc.PF + fc.fo];
            rlo[l] = fc.has_lo ? o.r[kk * PC + fc.clo] : 1.0;
            rhi[l] = fc.has_hi ? o.r[kk * PC + fc.chi] : 1.0;
        }
#pragma unroll
        for (int l = 0; l < KB; ++l) {
            if (k + l < o.n) {
                const double nw = q[l] > 0.0 ? q[l] * rlo[l] : (q[l] < 0.0 ? q[l] * rhi[l] : q[l]);
                d += q[l] - nw;
                if (nw != q[l]) Q[(size_t)(k + l) * fc.PF + fc.fo] = nw;
            }
        }
    }
    o.delta[t] = d;
}

// give the net cut back to the face's layers: same-way layers by donor room, then counter-flowing layers by |Q|
// (never past 0), then the donor's layers by content; a face that needs the last step out of an empty donor column
// is recorded (the reference raises there)
template <int AX>
__global__ void k_out_give(OutArgs o, int wrap) {
    const long long t = gtid();
    Geo<AX> g{o.n, o.ny, o.nx};
    if (t >= g.cols() || pass_ended<AX>(o)) return;
    const OutFace<AX> fc = out_face<AX>(o, t, wrap);
    double* Q = AX == 0 ? o.Qx : o.Qy;
    const size_t PC = g.pc();
    const double delta = o.delta[t];
    const double s = sgn(delta);
    // Most faces have no cut.  There (and where no room0 is infinite or NaN, whose product with 0 would be NaN) the
    // steps below add +0 to each flux and nothing else: a zero loses its sign.
    const bool plain = *o.wild == 0u;
    if (delta == 0.0 && plain) {
        for (int k = 0; k < o.n; k += KB) {
            double q[KB];
#pragma unroll
            for (int l = 0; l < KB; ++l) q[l] = Q[(size_t)min(k + l, o.n - 1) * fc.PF + fc.fo];
#pragma unroll
            for (int l = 0; l < KB; ++l)
                if (k + l < o.n && q[l] == 0.0 && __double_as_longlong(q[l]) < 0)
                    Q[(size_t)(k + l) * fc.PF + fc.fo] = 0.0;
        }
        return;
    }
    // the donor of the cut's direction: the low side for s > 0, else the high side
    const bool lo_side = s > 0.0, has = lo_side ? fc.has_lo : fc.has_hi;
    const size_t dc = lo_side ? fc.clo : fc.chi;
    double q[KB], rm[KB];
    // fluxes and donor rooms of the layers k .. k + KB - 1 (rm: 0 where a layer takes nothing back)
    auto load = [&](int k) {
#pragma unroll
        for (int l = 0; l < KB; ++l) {
            const size_t kk = (size_t)min(k + l, o.n - 1);
            q[l] = Q[kk * fc.PF + fc.fo];
            rm[l] = has ? o.room[kk * PC + dc] : 0.0;
        }
#pragma unroll
        for (int l = 0; l < KB; ++l) rm[l] = (sgn(q[l]) == s) && (q[l] != 0.0) && (s != 0.0) ? amax(rm[l], 0.0) : 0.0;
    };
    double tot = 0.0;
    for (int k = 0; k < o.n; k += KB) {
        load(k);
#pragma unroll
        for (int l = 0; l < KB; ++l)
            if (k + l < o.n) tot += rm[l];
    }
    const double need_ = fabs(delta);
    const double give = npmin(need_, tot);
    const double gq = tot > 0.0 ? give / tot : 0.0;
    double cap = 0.0;
    for (int k = 0; k < o.n; k += KB) {
        load(k);
#pragma unroll
        for (int l = 0; l < KB; ++l) {
            if (k + l < o.n) {
                const double nq = q[l] + s * rm[l] * gq;
                Q[(size_t)(k + l) * fc.PF + fc.fo] = nq;
                const bool opp = (sgn(nq) == -s) && (s != 0.0);
                cap += opp ? fabs(nq) : 0.0;
            }
        }
    }
    double rest = need_ - give;
    if (rest == 0.0 && plain) return;       // what follows would take and add zeros of the fluxes' own signs
    const double take = npmin(rest, cap);
    const double frac = cap > 0.0 ? take / cap : 0.0;
    rest = rest - take;
    const double on = rest > 0.0 ? 1.0 : 0.0;
    double tot2 = 0.0;
    for (int k = 0; k < o.n; ++k) {
        const size_t x = k * fc.PF + fc.fo;
        const double qk = Q[x];
        const bool opp = (sgn(qk) == -s) && (s != 0.0);
        Q[x] = qk - (opp ? qk * frac : 0.0);
        const double full = has ? room0(o, k * PC + dc, dc) : 0.0;
        tot2 += full * on;
    }
    if (rest > 0.0 && tot2 <= 0.0) atomicMin(o.bad_face, (unsigned long long)t);
    const double gr = tot2 > 0.0 ? rest / tot2 : 0.0;
    for (int k = 0; k < o.n; ++k) {
        const size_t x = k * fc.PF + fc.fo;
        const double full = has ? room0(o, k * PC + dc, dc) : 0.0;
        Q[x] = Q[x] + s * (full * on) * gr;
    }
}

// ------------------------------------------------------------------------------------------ Lagrangian step
// h† = h - Δt div / A (A = 1 where area <= 0), div = ∇·Q from divq or from Qx, Qy; the first cell-layer below
// -tol is recorded (linear index, atomicMin); h† = max(h†, 0).  With V0: V0 = h A, V1 = h† A, ok = active & V1 > 0.
__global__ void k_lagrangian(const double* __restrict__ h, const double* __restrict__ divq,
                             const double* __restrict__ Qx, const double* __restrict__ Qy,
                             const double* __restrict__ area, const uint8_t* __restrict__ act, int n, int ny,
                             int nx, double dt, double tol, double* __restrict__ out, double* __restrict__ V0,
                             double* __restrict__ V1, uint8_t* __restrict__ ok, unsigned long long* bad) {
    const long long t = gtid();
    const size_t PC = (size_t)ny * nx;
    if (t >= (long long)(PC * n)) return;
    const int k = (int)(t / PC);
    const size_t c = (size_t)t - (size_t)k * PC;
    double dv;
    if (divq) {
        dv = divq[t];
    } else {
        const int j = (int)(c / nx), i = (int)(c - (size_t)j * nx);
        const size_t fx = ((size_t)k * ny + j) * (nx + 1) + i;
        const size_t fy = ((size_t)k * (ny + 1) + j) * nx + i;
        dv = Qx[fx + 1] - Qx[fx] + Qy[fy + nx] - Qy[fy];
    }
    const double ar = area[c];
    const double hk = h[t];
    double v = hk - dt * dv / (ar > 0.0 ? ar : 1.0);
    if (v < -tol) atomicMin(bad, (unsigned long long)t);
    v = v < 0.0 ? 0.0 : v;
    out[t] = v;
    if (V0) {
        const double a1 = hk * ar, a2 = v * ar;
        V0[t] = a1;
        V1[t] = a2;
        ok[t] = (act[c] && a2 > 0.0) ? 1 : 0;
    }
}

// h_dag = active ? h - Δt div / A : 0 (A = area on active cells, 1 elsewhere); min over all cell-layers as an
// order-preserving u64 key (atomicMin), then the first index holding that minimum
__device__ __forceinline__ unsigned long long order_key(double x) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(x);
    return (b >> 63) ? ~b : (b | 0x8000000000000000ull);
}

__device__ __forceinline__ double h_dag(const OutArgs& o, long long t) {
    const size_t PC = (size_t)o.ny * o.nx;
    const int k = (int)(t / PC);
    const size_t c = (size_t)t - (size_t)k * PC;
    if (!o.act[c]) return 0.0;
    const int j = (int)(c / o.nx), i = (int)(c - (size_t)j * o.nx);
    const size_t fx = ((size_t)k * o.ny + j) * (o.nx + 1) + i;
    const size_t fy = ((size_t)k * (o.ny + 1) + j) * o.nx + i;
    const double div = o.Qx[fx + 1] - o.Qx[fx] + o.Qy[fy + o.nx] - o.Qy[fy];
    const double A = o.area[c];
    return o.h[t] - o.dt * div / (A > 0.0 ? A : 1.0);
}

__global__ void k_hdag_min(OutArgs o, unsigned long long* key) {
    const long long t = gtid();
    const long long N = (long long)o.n * o.ny * o.nx;
    if (t >= N) return;
    atomicMin(key, order_key(h_dag(o, t)));
}

__global__ void k_hdag_where(OutArgs o, const unsigned long long* key, unsigned long long* idx) {
    const long long t = gtid();
    const long long N = (long long)o.n * o.ny * o.nx;
    if (t >= N) return;
    if (order_key(h_dag(o, t)) == *key) atomicMin(idx, (unsigned long long)t);
}

}  // namespace ale
}  // namespace ocx
