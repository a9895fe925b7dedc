// budget.hip -- per-snapshot turbulence statistics and kinetic-energy budget on the
// device (dnsg_budget2d).
//
// The reference computes them offline, one snapshot at a time, with its TKE-budget
// tool (TKE-budget/computations/budget2D.c:13-1736, reading.c, uv_fluc.c) from the
// vel-* and den-* files.  Here the same pass runs on the current state:
//   1. k_bud_fill    velocity and density of every node of the three grids, formed as
//                    vel_print does, in planes [u v w rho][layer][y][x] (x fastest, as in
//                    the lattices, so every pass reads and writes whole lines: in the
//                    tool's [x][y][z] order the fill alone took 10.7 ms at the Re_tau=180
//                    size, now 1.0), and the per-layer sums of u, v, w, rho/3
//                    (budget2D.c:177-244);
//   2. k_bud_nodes   the 44 per-node products and derivative terms of :449-987 of the
//                    fluctuations, formed at each read (value - layer mean, :265-309), and
//                    summed per layer; the tool's periodic x ghost planes are index wraps,
//                    and where its one-sided z stencil reaches past a layer stack into the
//                    next row of its array, the same element is read here (bud_at);
//   3. the O(NZ) tail on the host: dU/dz, normalisation, production, transport,
//      dissipation (:311-444, :1003-1547).
// Each node's terms are formed exactly as the tool forms them; the sums over a
// layer are taken in another order, so the profiles agree with the tool's to
// rounding (1e-12 relative), not bit for bit.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <type_traits>
#include <vector>

#include "budget_split.hpp"
#include "internal.hpp"
#include "lattice.hpp"

namespace dnsg {

namespace {

// the per-node accumulators (budget2D.c:449-617), in this order in every table
enum {
    A_UU, A_UV, A_UW, A_VV, A_VW, A_WW, A_SKU, A_SKV, A_SKW, A_SKP, A_SKUW, A_SKUV, A_SKVW,
    A_KUU, A_KUV, A_KUW, A_KUP, A_KUUW, A_KUVW, A_KUUV, A_DD, A_UUW, A_VVW, A_WWW, A_UWW,
    A_PU, A_PV, A_PW, A_WX, A_WY, A_WZ, A_PAIUU, A_PAIVV, A_PAIWW, A_PAIUW,
    A_USUW, A_VSVW, A_WSWW, A_WSUW, A_USWW, A_EPUU, A_EPVV, A_EPWW, A_EPUW, NACC
};

// one grid of the snapshot: planes [4][Z][Y][X] of u, v, w, rho
struct BudGrid {
    double *v;
    int X, Y, Z;
    int k0, k1;         // layers taking part in the statistics
    int m0, m1;         // layers whose mean is taken (and subtracted)
    int base;           // profile index of layer 0
    int rows;           // rows a thread takes (bud_rows)
};

struct BudArgs {
    BudGrid g[3];       // coarse, lower band, upper band
    int GR;
    double coef;
    const double *mean; // [4][NZ]: U, V, W, rho/3
    int NZ;
};

// velocity and density of one node as vel_print.c:86-117 forms them
struct Vel {
    double u, v, w, rho;
};
__device__ __forceinline__ Vel node_vel(const double *f) {
    Vel r = {0., 0., 0., 0.};
    unroll<0, Q>([&](auto qq) {
        constexpr int q = decltype(qq)::value;
        r.u += (double)EX[q] * f[q];
        r.v += (double)EY[q] * f[q];
        r.w += (double)EZ[q] * f[q];
        r.rho += f[q];
    });
    if (r.rho > 0.) { r.u /= r.rho; r.v /= r.rho; r.w /= r.rho; }
    else r = {0., 0., 0., 0.};
    return r;
}
// node (x, y, k) of a grid whose stored layers start at file layer zlo and whose wall
// layer kwall (-1: none) comes from the wall-layer copy [X][Y][19]
template <class S>
__device__ __forceinline__ Vel file_vel(const S *__restrict__ lat, const double *__restrict__ wall, int X, int Y, int zlo,
                                        int kwall, int x, int y, int k) {
    double f[Q];
    if (k == kwall) {
        const double *w = wall + ((size_t)x * Y + y) * Q;
        unroll<0, Q>([&](auto qq) { f[decltype(qq)::value] = w[decltype(qq)::value]; });
    } else {
        const size_t row = (size_t)(k - zlo) * Y + y;
        unroll<0, Q>([&](auto qq) {
            constexpr int q = decltype(qq)::value;
            f[q] = (double)load_s(lat + lat_at(q, row, x, X));
            if constexpr (sizeof(S) != 8) f[q] += WQ[q];
        });
    }
    return node_vel(f);
}

// sum of W values over a workgroup into out[0..W) (fixed order: lanes, then waves)
template <int W>
__device__ __forceinline__ void wg_sum(double *v, double *out) {
    __shared__ double l[BT / 64][W];
#pragma unroll
    for (int c = 0; c < W; c++)
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) v[c] += __shfl_down(v[c], o, 64);
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    if (lane == 0)
#pragma unroll
        for (int c = 0; c < W; c++) l[wv][c] = v[c];
    __syncthreads();
    for (int c = threadIdx.x; c < W; c += BT) {
        double s = l[0][c];
#pragma unroll
        for (int w = 1; w < BT / 64; w++) s += l[w][c];
        out[c] = s;
    }
}

// 1. planes of one grid, and per-(layer, chunk) sums of u, v, w, rho/3
template <class S>
__global__ __launch_bounds__(BT) void k_bud_fill(const S *__restrict__ lat, const double *__restrict__ wall, BudGrid G,
                                                 int zlo, int kwall, double *__restrict__ part) {
    const int nch = bud_chunks(G.X, G.Y, G.rows);
    const int k = (int)blockIdx.x / nch;
    int x, y0;
    bud_column(G.X, G.rows, (int)blockIdx.x % nch, threadIdx.x, x, y0);
    double v[4] = {0., 0., 0., 0.};
    for (int y = y0; y < min(y0 + G.rows, G.Y); y++) {
        const Vel r = file_vel(lat, wall, G.X, G.Y, zlo, kwall, x, y, k);
        const size_t plane = (size_t)G.Z * G.Y * G.X, e = ((size_t)k * G.Y + y) * G.X + x;
        G.v[e] = r.u;
        G.v[plane + e] = r.v;
        G.v[2 * plane + e] = r.w;
        G.v[3 * plane + e] = r.rho;
        v[0] += r.u;
        v[1] += r.v;
        v[2] += r.w;
        v[3] += (1. / 3.) * r.rho;
    }
    wg_sum<4>(v, part + (size_t)blockIdx.x * 4);
}

// sums of nch consecutive partial records of w values, one wave per (segment, value)
__global__ __launch_bounds__(BT) void k_bud_segsum(const double *__restrict__ part, int nseg, int nch, int w,
                                                   double *__restrict__ out) {
    const int t = (int)(blockIdx.x * (BT / 64) + (threadIdx.x >> 6)), lane = threadIdx.x & 63;
    if (t >= nseg * w) return;  // uniform over the wave
    const int s = t / w, c = t % w;
    double a = 0.;
    for (int i = lane; i < nch; i += 64) a += part[((size_t)s * nch + i) * w + c];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) a += __shfl_down(a, o, 64);
    if (lane == 0) out[t] = a;
}

// Fluctuation of velocity component c at element (i, j, k) of the tool's array of grid g,
// [x][y][k] behind two ghost planes in x: k outside the layers is the element that lies
// there, in the next or previous row (j) or plane (i); i is periodic
__device__ __forceinline__ double bud_at(const BudArgs &A, int g, int i, int j, int k, int c) {
    const BudGrid &G = A.g[g];
    while (k >= G.Z) { k -= G.Z; j++; }
    while (k < 0) { k += G.Z; j--; }
    if (j >= G.Y) { j -= G.Y; i++; }
    if (j < 0) { j += G.Y; i--; }
    i = i < 0 ? i + G.X : (i >= G.X ? i - G.X : i);
    const double u = G.v[(((size_t)c * G.Z + k) * G.Y + j) * G.X + i];
    return (k >= G.m0 && k < G.m1) ? u - A.mean[c * A.NZ + G.base + k] : u;
}

// z derivative of component c at (i, j, k) of grid g (budget2D.c:539-593 lower band,
// :720-748 coarse, :904-940 upper band)
__device__ __forceinline__ double bud_ddz(const BudArgs &A, int g, int i, int j, int k, int c) {
    const BudGrid &G = A.g[g];
    const int GR = A.GR;
    const double coef = A.coef;
    auto V = [&](int kk) { return bud_at(A, g, i, j, kk, c); };
    if (g == 1) {
        if (k == 1) {
            const double tmp = (2. / 3.) * (V(k + 3) - V(k + 1)) - (1. / 12.) * (V(k + 4) - V(k));
            return -(7. / 3.) * V(k) + 6. * V(k + 1) - 3. * V(k + 2) - (2. / 3.) * V(k + 3) + 3. * tmp;
        }
        if (k == G.Z - 1) {
            const double cc = bud_at(A, 0, i / GR, j / GR, 2, c);
            return (coef * (cc - V(k)) + GR * (V(k) - V(k - 1))) * 1. / (1. + GR);
        }
        return 0.5 * (V(k + 1) - V(k - 1));
    }
    if (g == 0) {
        if (k == 2) return 0.5 * coef * (V(k + 1) - bud_at(A, 1, i * GR, j * GR, A.g[1].Z - 1, c));
        if (k == 3 || k == G.Z - 4) return 0.5 * coef * (V(k + 1) - V(k - 1));
        if (k == G.Z - 3) return 0.5 * coef * (bud_at(A, 2, i * GR, j * GR, 0, c) - V(k - 1));
        return 0.5 * coef * (V(k + 1) - V(k - 1));
    }
    if (k == 0) {
        const double cc = bud_at(A, 0, i / GR, j / GR, A.g[0].Z - 3, c);
        return (GR * (V(k + 1) - V(k)) + coef * (V(k) - cc)) * 1. / (1. + GR);
    }
    if (k == G.Z - 2) {
        const double tmp = (2. / 3.) * (V(k - 1) - V(k - 3)) - (1. / 12.) * (V(k) - V(k - 4));
        return (7. / 3.) * V(k) - 6. * V(k - 1) + 3. * V(k - 2) + (2. / 3.) * V(k - 3) + 3. * tmp;
    }
    return 0.5 * (V(k + 1) - V(k - 1));
}

// 2. the per-node terms of grid g (budget2D.c:449-617, :636-797, :800-987), summed
//    per (layer, chunk) -> part[(k - k0) * chunks + chunk][NACC]
__global__ __launch_bounds__(BT) void k_bud_nodes(BudArgs A, int g, double *__restrict__ part) {
    const BudGrid &G = A.g[g];
    const int X = G.X, Y = G.Y, nch = bud_chunks(X, Y, G.rows);
    const int k = G.k0 + (int)blockIdx.x / nch;
    int i, y0;
    bud_column(X, G.rows, (int)blockIdx.x % nch, threadIdx.x, i, y0);
    double a[NACC];
#pragma unroll
    for (int c = 0; c < NACC; c++) a[c] = 0.;
    const int im = i == 0 ? X - 1 : i - 1, imm = im == 0 ? X - 1 : im - 1;
    const int ip = i == X - 1 ? 0 : i + 1, ipp = ip == X - 1 ? 0 : ip + 1;
    const size_t plane = (size_t)Y * X;
    for (int j = y0; j < min(y0 + G.rows, Y); j++) {
        const int jp = j == 0 ? Y - 1 : j - 1, jpp = jp == 0 ? Y - 1 : jp - 1;
        const int jn = j == Y - 1 ? 0 : j + 1, jnn = jn == Y - 1 ? 0 : jn + 1;
        double w0[3], d[3][3];
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const double *p = G.v + ((size_t)c * G.Z + k) * plane;
            const double m = (k >= G.m0 && k < G.m1) ? A.mean[c * A.NZ + G.base + k] : 0.;
            auto at = [&](int ii, int jj) { return p[(size_t)jj * X + ii] - m; };
            const double gx = (2. / 3.) * (at(ip, j) - at(im, j)) - (1. / 12.) * (at(ipp, j) - at(imm, j));
            const double gy = (2. / 3.) * (at(i, jn) - at(i, jp)) - (1. / 12.) * (at(i, jnn) - at(i, jpp));
            w0[c] = at(i, j);
            d[c][0] = g == 0 ? A.coef * gx : gx;
            d[c][1] = g == 0 ? A.coef * gy : gy;
            d[c][2] = bud_ddz(A, g, i, j, k, c);
        }
        const double u = w0[0], vv = w0[1], w = w0[2];
        const double dfl = (1. / 3.) * G.v[((size_t)3 * G.Z + k) * plane + (size_t)j * X + i] - A.mean[3 * A.NZ + G.base + k];
        const double dudx = d[0][0], dudy = d[0][1], dudz = d[0][2];
        const double dvdx = d[1][0], dvdy = d[1][1], dvdz = d[1][2];
        const double dwdx = d[2][0], dwdy = d[2][1], dwdz = d[2][2];
        const double ox = (dwdy - dvdz), oy = (dudz - dwdx), oz = (dvdx - dudy);
        a[A_UU] += u * u; a[A_UV] += u * vv; a[A_UW] += u * w; a[A_VV] += vv * vv; a[A_VW] += vv * w; a[A_WW] += w * w;
        a[A_SKU] += u * u * u; a[A_SKV] += vv * vv * vv; a[A_SKW] += w * w * w; a[A_SKP] += dfl * dfl * dfl;
        a[A_SKUW] += u * u * u * w * w * w; a[A_SKUV] += u * u * u * vv * vv * vv; a[A_SKVW] += vv * vv * vv * w * w * w;
        a[A_KUU] += u * u * u * u; a[A_KUV] += vv * vv * vv * vv; a[A_KUW] += w * w * w * w;
        a[A_KUP] += dfl * dfl * dfl * dfl;
        a[A_KUUW] += u * u * u * u * w * w * w * w; a[A_KUVW] += vv * vv * vv * vv * w * w * w * w;
        a[A_KUUV] += u * u * u * u * vv * vv * vv * vv;
        a[A_DD] += dfl * dfl;
        a[A_UUW] += u * u * w; a[A_VVW] += vv * vv * w; a[A_WWW] += w * w * w; a[A_UWW] += u * w * w;
        a[A_PU] += u * dfl; a[A_PV] += vv * dfl; a[A_PW] += w * dfl;
        a[A_WX] += ox * ox; a[A_WY] += oy * oy; a[A_WZ] += oz * oz;
        a[A_PAIUU] += dfl * dudx; a[A_PAIVV] += dfl * dvdy; a[A_PAIWW] += dfl * dwdz; a[A_PAIUW] += dfl * (dudz + dwdx);
        a[A_USUW] += 0.5 * u * (dudz + dwdx); a[A_VSVW] += 0.5 * vv * (dvdz + dwdy);
        a[A_WSWW] += 0.5 * w * (dwdz + dwdz); a[A_WSUW] += 0.5 * w * (dudz + dwdx); a[A_USWW] += 0.5 * u * (dwdz + dwdz);
        a[A_EPUU] += dudx * (dudx + dudx) + dudy * (dudy + dvdx) + dudz * (dudz + dwdx);
        a[A_EPVV] += dvdx * (dvdx + dudy) + dvdy * (dvdy + dvdy) + dvdz * (dvdz + dwdy);
        a[A_EPWW] += dwdx * (dwdx + dudz) + dwdy * (dwdy + dvdz) + dwdz * (dwdz + dwdz);
        a[A_EPUW] += dudx * (dwdx + dudz) + dudy * (dwdy + dvdz) + dudz * (dwdz + dwdz) + dwdx * (dudx + dudx) +
                     dwdy * (dudy + dvdx) + dwdz * (dudz + dwdx);
    }
    wg_sum<NACC>(a, part + (size_t)blockIdx.x * NACC);
}

// the lower band's u', v' at k = 4 (uv_fluc.c:25-33), [Xf][Yf]
__global__ __launch_bounds__(BT) void k_bud_plane(BudArgs A, int k, double *__restrict__ uo, double *__restrict__ vo) {
    const int n = blockIdx.x * BT + threadIdx.x;
    if (n >= A.g[1].X * A.g[1].Y) return;
    uo[n] = bud_at(A, 1, n / A.g[1].Y, n % A.g[1].Y, k, 0);
    vo[n] = bud_at(A, 1, n / A.g[1].Y, n % A.g[1].Y, k, 1);
}

// 3. dU/dz of the mean profile (budget2D.c:311-444)
void bud_dudz(const double *U, int zdf, int zdc, int GR, double *dUdz) {
    const double coef = (1. / ((double)GR));
    const int zd = zdf;
    for (int k = 1; k < zd; k++) {
        const double *a = U;
        if (k == 1) {
            const double tmp = (2. / 3.) * (a[k + 3] - a[k + 1]) - (1. / 12.) * (a[k + 4] - a[k]);
            dUdz[k] = -(7. / 3.) * a[k] + 6. * a[k + 1] - 3. * a[k + 2] - (2. / 3.) * a[k + 3] + 3. * tmp;
        } else if (k == zd - 1) {
            dUdz[k] = (coef * (a[k + 1] - a[k]) + GR * (a[k] - a[k - 1])) * 1. / (1. + GR);
        } else if (k == 2 || k == zd - 2) {
            dUdz[k] = 0.5 * (a[k + 1] - a[k - 1]);
        } else {
            dUdz[k] = (2. / 3.) * (a[k + 1] - a[k - 1]) - (1. / 12.) * (a[k + 2] - a[k - 2]);
        }
    }
    for (int k = 2; k < zdc - 2; k++) {
        const double *a = U + zdf - 2;
        if (k == 2 || k == 3 || k == zdc - 4 || k == zdc - 3) dUdz[zdf - 2 + k] = 0.5 * coef * (a[k + 1] - a[k - 1]);
        else dUdz[zdf - 2 + k] = coef * ((2. / 3.) * (a[k + 1] - a[k - 1]) - (1. / 12.) * (a[k + 2] - a[k - 2]));
    }
    double *o = dUdz + zdf + zdc - 4;
    const double *a = U + zdf + zdc - 4;
    for (int k = 0; k < zd - 1; k++) {
        if (k == 0) {
            o[k] = (GR * (a[k + 1] - a[k]) + coef * (a[k] - a[k - 1])) * 1. / (1. + GR);
        } else if (k == zd - 2) {
            const double tmp = (2. / 3.) * (a[k - 1] - a[k - 3]) - (1. / 12.) * (a[k] - a[k - 4]);
            o[k] = (7. / 3.) * a[k] - 6. * a[k - 1] + 3. * a[k - 2] + (2. / 3.) * a[k - 3] + 3. * tmp;
        } else if (k == 1 || k == zd - 3) {
            o[k] = 0.5 * (a[k + 1] - a[k - 1]);
        } else {
            o[k] = (2. / 3.) * (a[k + 1] - a[k - 1]) - (1. / 12.) * (a[k + 2] - a[k - 2]);
        }
    }
}

// 3. normalisation and the derived profiles (budget2D.c:1003-1547)
void bud_finish(const dnsg_params &p, const double *Um, const double *dUdz, std::vector<double> &a, double *turb,
                double *vort, double *ke) {
    const int GR = p.gratio, zdf = p.zds + 1, zdc = p.zdv;
    const int NZ = 2 * zdf + (zdc - 4), NZs = 2 * zdf + GR * (zdc - 4) + GR - 1;
    const double tauf = (3. / p.Rebs) * p.ub * (NZs - 2.) + 0.5;  // :55-58
    const double nu = (1. / 6.) * (2. * tauf - 1.), coef = (1. / ((double)GR));
    const double nf = (double)(GR * p.xdv) * (GR * p.ydv), nc = (double)p.xdv * p.ydv;
    auto S = [&](int n) { return a.data() + (size_t)n * NZ; };
    std::memset(turb, 0, (size_t)19 * NZ * 8);
    std::memset(vort, 0, (size_t)3 * NZ * 8);
    std::memset(ke, 0, (size_t)30 * NZ * 8);
    double *UTIN = turb + 3 * NZ, *VTIN = turb + 4 * NZ, *WTIN = turb + 5 * NZ, *DTIN = turb + 8 * NZ;
    double *Pii = ke, *Puu = ke + NZ, *Pvv = ke + 2 * NZ, *Pww = ke + 3 * NZ, *Puw = ke + 4 * NZ;
    double *Tiir = ke + 5 * NZ, *Tuur = ke + 6 * NZ, *Tvvr = ke + 7 * NZ, *Twwr = ke + 8 * NZ, *Tuwr = ke + 9 * NZ;
    double *Tiipai = ke + 10 * NZ, *Tuupai = ke + 11 * NZ, *Tvvpai = ke + 12 * NZ, *Twwpai = ke + 13 * NZ;
    double *Tuwpai = ke + 14 * NZ, *Tiis = ke + 19 * NZ, *Tuus = ke + 20 * NZ, *Tvvs = ke + 21 * NZ;
    double *Twws = ke + 22 * NZ, *Tuws = ke + 23 * NZ, *Epii = ke + 24 * NZ, *KE = ke + 29 * NZ;
    for (int k = 0; k < NZ; k++) {  // :1003-1058
        const double num = k < zdf ? nf : ((k < zdf + zdc - 4 && k >= zdf) ? nc : nf);
        for (int n = 0; n < NACC; n++) S(n)[k] /= num;
    }
    for (int k = 1; k < NZ - 1; k++) {  // :1201-1237
        const double siu = UTIN[k] = std::sqrt(S(A_UU)[k]), siv = VTIN[k] = std::sqrt(S(A_VV)[k]);
        const double siw = WTIN[k] = std::sqrt(S(A_WW)[k]), sip = DTIN[k] = std::sqrt(S(A_DD)[k]);
        KE[k] += (S(A_UU)[k] + S(A_VV)[k] + S(A_WW)[k]);
        S(A_WX)[k] = std::sqrt(S(A_WX)[k]);
        S(A_WY)[k] = std::sqrt(S(A_WY)[k]);
        S(A_WZ)[k] = std::sqrt(S(A_WZ)[k]);
        S(A_SKU)[k] /= (siu * siu * siu);
        S(A_SKV)[k] /= (siv * siv * siv);
        S(A_SKW)[k] /= (siw * siw * siw);
        S(A_SKP)[k] /= (sip * sip * sip);
        S(A_SKUW)[k] /= (siu * siu * siu * siw * siw * siw);
        S(A_SKVW)[k] /= (siv * siv * siv * siw * siw * siw);
        S(A_SKUV)[k] /= (siu * siu * siu * siv * siv * siv);
        S(A_KUU)[k] /= (siu * siu * siu * siu);
        S(A_KUV)[k] /= (siv * siv * siv * siv);
        S(A_KUW)[k] /= (siw * siw * siw * siw);
        S(A_KUP)[k] /= (sip * sip * sip * sip);
        S(A_KUUW)[k] /= (siu * siu * siu * siu * siw * siw * siw * siw);
        S(A_KUUV)[k] /= (siu * siu * siu * siu * siv * siv * siv * siv);
        S(A_KUVW)[k] /= (siv * siv * siv * siv * siw * siw * siw * siw);
        S(A_EPUU)[k] *= nu;
        S(A_EPVV)[k] *= nu;
        S(A_EPWW)[k] *= nu;
        S(A_EPUW)[k] *= (2. * nu);
        Epii[k] = (S(A_EPUU)[k]) + (S(A_EPVV)[k]) + (S(A_EPWW)[k]);
    }
    // production and transport (:1238-1547); the z differences of the tool's
    // DDZ1F, DDZ1B, DDZ2C, DDZ2CNUl and DDZ2CNUu
    enum { D1F, D1B, D2C, NUL, NUU };
    auto D = [&](int op, int s, int k) {
        const double *x = S(s);
        switch (op) {
        case D1F: return (x[k + 1]) - (x[k]);
        case D1B: return (x[k]) - (x[k - 1]);
        case D2C: return ((x[k + 1]) - (x[k - 1])) * 0.5;
        case NUL: return (1. / (1. + GR)) * ((1. / GR) * ((x[k + 1]) - (x[k])) + GR * ((x[k]) - (x[k - 1])));
        default: return (1. / (1. + GR)) * ((1. / GR) * ((x[k]) - (x[k - 1])) + GR * ((x[k + 1]) - (x[k])));
        }
    };
    auto terms = [&](int q, int op, double m, double m2, double cs, double half) {
        Tuur[q] = half * D(op, A_UUW, q);
        Tvvr[q] = half * D(op, A_VVW, q);
        Twwr[q] = half * D(op, A_WWW, q);
        Tuwr[q] = m * D(op, A_UWW, q);
        Tiipai[q] = m * D(op, A_PW, q);
        Twwpai[q] = m2 * D(op, A_PW, q);
        Tuwpai[q] = m * D(op, A_PU, q);
        Tuus[q] = cs * D(op, A_USUW, q);
        Tvvs[q] = cs * D(op, A_VSVW, q);
        Twws[q] = cs * D(op, A_WSWW, q);
        Tuws[q] = cs * D(op, A_WSUW, q) + cs * D(op, A_WSWW, q);
    };
    auto common = [&](int q) {
        Pii[q] = -(S(A_UW)[q]) * (dUdz[q]);
        Puu[q] = 2. * (Pii[q]);
        Pvv[q] = 0.;
        Pww[q] = 0.;
        Puw[q] = -(S(A_WW)[q]) * (dUdz[q]);
        Tuupai[q] = 0.;
        Tvvpai[q] = 0.;
    };
    auto sums = [&](int q) {
        Tiis[q] = 0.5 * (Tuus[q] + Tvvs[q] + Twws[q]);
        Tiir[q] = 0.5 * (Tuur[q] + Tvvr[q] + Twwr[q]);
    };
    for (int k = 1; k < zdf; k++) {
        const int q = k;
        common(q);
        if (k == 1) terms(q, D1F, -1., -2., 2. * nu, -1.);
        else if (k == zdf - 1) terms(q, NUL, -1., -2., 2. * nu, -1.);
        else if (k == 2 || k == zdf - 2) terms(q, D2C, -1., -2., 2. * nu, -1.);
        else terms(q, D2C, -1., -2., 2. * nu, -0.5);
        sums(q);
    }
    for (int k = 2; k < zdc - 2; k++) {
        const int q = zdf - 2 + k;
        common(q);
        if (k == 2 || k == 3 || k == zdc - 4 || k == zdc - 3) terms(q, D2C, -coef, -2. * coef, 2. * nu * coef, -coef);
        else terms(q, D2C, -coef, -2. * coef, coef * 2. * nu, -coef * 0.5);
        sums(q);
    }
    for (int k = 0; k < zdf - 1; k++) {
        const int q = zdf + zdc - 4 + k;
        common(q);
        if (k == 0) terms(q, NUU, -1., -2., 2. * nu, -1.);
        else if (k == zdf - 2) terms(q, D1B, -1., -2., 2. * nu, -1.);
        else if (k == 2 || k == zdf - 3) terms(q, D2C, -1., -2., 2. * nu, -1.);
        else terms(q, D2C, -1., -2., 2. * nu, -0.5);
        sums(q);
    }
    // the files' profiles (:1553-1636)
    std::memcpy(turb, Um, (size_t)3 * NZ * 8);
    std::memcpy(turb + 6 * NZ, S(A_UW), NZ * 8);
    std::memcpy(turb + 7 * NZ, Um + 3 * NZ, NZ * 8);
    const int tsrc[10] = {A_SKU, A_SKV, A_SKW, A_SKUW, A_SKP, A_KUU, A_KUV, A_KUW, A_KUUW, A_KUP};
    for (int t = 0; t < 10; t++) std::memcpy(turb + (9 + t) * NZ, S(tsrc[t]), NZ * 8);
    for (int t = 0; t < 3; t++) std::memcpy(vort + t * NZ, S(A_WX + t), NZ * 8);
    for (int t = 0; t < 4; t++) std::memcpy(ke + (15 + t) * NZ, S(A_PAIUU + t), NZ * 8);
    for (int t = 0; t < 4; t++) std::memcpy(ke + (25 + t) * NZ, S(A_EPUU + t), NZ * 8);
}

}  // namespace

// A snapshot's tile: SX columns x by SZ layers of one row y.  The lattice is read along x
// and the file order [x][y][k][3] written along k, through LDS (written node by node
// from threads along k, each of the 19 reads of a node was a line of its own: 0.25 ms for
// a 420 x 252 x 12 band against 0.05).
constexpr int SX = 32, SZ = 8;
template <class S>
__global__ __launch_bounds__(SX *SZ) void k_snapshot(const S *__restrict__ lat, const double *__restrict__ wall, int X,
                                                      int Y, int Z, int zlo, int kwall, double *__restrict__ vel,
                                                      double *__restrict__ den) {
    __shared__ double sv[SX][3 * SZ + 1], sd[SX][SZ + 1];
    const int nxc = (X + SX - 1) / SX, nzc = (Z + SZ - 1) / SZ;
    const int bx = blockIdx.x % nxc, bz = blockIdx.x / nxc % nzc, y = blockIdx.x / (nxc * nzc);
    const int x0 = bx * SX, z0 = bz * SZ, tx = threadIdx.x % SX, tz = threadIdx.x / SX;
    if (x0 + tx < X && z0 + tz < Z) {
        const Vel r = file_vel(lat, wall, X, Y, zlo, kwall, x0 + tx, y, z0 + tz);
        sv[tx][3 * tz] = r.u;
        sv[tx][3 * tz + 1] = r.v;
        sv[tx][3 * tz + 2] = r.w;
        sd[tx][tz] = r.rho;
    }
    __syncthreads();
    const int nz = min(SZ, Z - z0), nx = min(SX, X - x0);
    for (int t = threadIdx.x; t < nx * 3 * nz; t += SX * SZ) {
        const int xx = t / (3 * nz), e = t % (3 * nz);
        vel[(((size_t)(x0 + xx) * Y + y) * Z + z0) * 3 + e] = sv[xx][e];
    }
    for (int t = threadIdx.x; t < nx * nz; t += SX * SZ) {
        const int xx = t / nz, e = t % nz;
        den[((size_t)(x0 + xx) * Y + y) * Z + z0 + e] = sd[xx][e];
    }
}

// a grid as vel_print sees it: its lattice, extents, first stored file layer, wall layer
struct FileGrid {
    const Grid *lat;
    int X, Y, Z, zlo, kwall;
    const double *wall;
};
FileGrid file_grid(const dnsg_ctx *h, int g) {
    const dnsg_dims &d = h->d;
    if (g == 0) return {&h->coarse, d.Xc, d.Yc, d.zdc, 0, -1, h->fwall};
    if (g == 1) return {&h->lower, d.Xf, d.Yf, d.zdf, 1, 0, h->fwall};
    return {&h->upper, d.Xf, d.Yf, d.zdf, 0, d.zdf - 1, h->fwall + (size_t)d.Xf * d.Yf * 19};
}

template <class F>
auto by_storage(const dnsg_ctx *h, const void *lat, F f) {
    if (h->p.precision == DNSG_PREC_FP64) return f((const double *)lat);
    if (h->p.precision == DNSG_PREC_FP32) return f((const float *)lat);
    return f((const __half *)lat);
}

hipError_t launch_snapshot(dnsg_ctx *h, int g, double *vel, double *den) {
    const FileGrid F = file_grid(h, g);
    const dim3 grd((unsigned)(((F.X + SX - 1) / SX) * ((F.Z + SZ - 1) / SZ)) * (unsigned)F.Y), blk(SX * SZ);
    by_storage(h, F.lat->c(), [&](auto *lat) {
        using S = std::remove_const_t<std::remove_pointer_t<decltype(lat)>>;
        hipLaunchKernelGGL(k_snapshot<S>, grd, blk, 0, h->stream, lat, F.wall, F.X, F.Y, F.Z, F.zlo, F.kwall, vel, den);
    });
    return hipGetLastError();
}

}  // namespace dnsg

using namespace dnsg;

constexpr size_t BUD_SMALL = (size_t)1 << 20;

#define BCHK(h, expr)                                                                       \
    do {                                                                                    \
        hipError_t e_ = (expr);                                                             \
        if (e_ != hipSuccess) {                                                             \
            (h)->err = std::string(#expr) + ": " + hipGetErrorString(e_);                   \
            rc = e_ == hipErrorOutOfMemory ? DNSG_ERR_OOM : DNSG_ERR_HIP;                   \
            goto done;                                                                      \
        }                                                                                   \
    } while (0)

extern "C" int dnsg_budget2d(dnsg_t *h, double *turb, double *vort, double *ke, double *ufl, double *vfl) {
    if (!h || !h->stream || !turb || !vort || !ke || (!ufl) != (!vfl)) return DNSG_ERR_ARG;
    if (!h->have_state) {
        h->err = "no state: call dnsg_init_state or dnsg_upload_state first";
        return DNSG_ERR_STATE;
    }
    const dnsg_dims &d = h->d;
    if (d.Yc < 4 || d.zdc < 6) {  // the tool's periodic y stencil and its coarse z branches
        h->err = "the budget needs ydv >= 4 and zdv >= 6";
        return DNSG_ERR_ARG;
    }
    int rc = ensure_fwall(h);
    if (rc) return rc;
    const int zdf = d.zdf, zdc = d.zdc, NZ = 2 * zdf + (zdc - 4), GR = d.GR;
    BudArgs A{};
    A.GR = GR;
    A.coef = (1. / ((double)GR));
    A.NZ = NZ;
    const int k0[3] = {2, 1, 0}, k1[3] = {zdc - 2, zdf, zdf - 1};    // node passes
    const int m0[3] = {2, 0, 0}, m1[3] = {zdc - 2, zdf, zdf};        // means and subtraction
    const int base[3] = {zdf - 2, 0, zdf + zdc - 4};
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, h->device) != hipSuccess) cus = 0;
    size_t npart = 0, nv[3], off[3][2], n4 = 0, nacc = 0;  // off: of a grid's sums, layer means and node terms
    std::vector<double> mean(4 * (size_t)NZ, 0.), acc((size_t)NACC * NZ, 0.), dUdz(NZ, 0.), lay;
    double *dmean = nullptr, *dpart = nullptr, *dsum = nullptr, *dpl = nullptr, *dv[3] = {nullptr, nullptr, nullptr};
    for (int g = 0; g < 3; g++) {
        const FileGrid F = file_grid(h, g);
        const int rows = bud_rows(F.X, F.Y, k1[g] - k0[g], cus);
        A.g[g] = BudGrid{nullptr, F.X, F.Y, F.Z, k0[g], k1[g], m0[g], m1[g], base[g], rows};
        npart = std::max(npart, (size_t)bud_chunks(F.X, F.Y, rows) * F.Z * NACC);
        off[g][0] = n4;
        off[g][1] = nacc;
        n4 += (size_t)F.Z * 4;
        nacc += (size_t)(k1[g] - k0[g]) * NACC;
        nv[g] = 4 * (size_t)F.X * F.Y * F.Z;
    }
    // one block for the planes of all grids, or one a grid where each is below 1 MiB: the
    // runtime cuts those from a larger one, while a block of its own takes 0.3 ms or more
    // (the first budget of a 32 x 24 x 16 handle 560 us with one block, 280 with three)
    if (nv[0] * 8 < BUD_SMALL && nv[1] * 8 < BUD_SMALL) {
        for (int g = 0; g < 3; g++) {
            BCHK(h, scratch_get(&dv[g], nv[g] * 8));
            A.g[g].v = dv[g];
        }
    } else {
        BCHK(h, scratch_get(&dv[0], (nv[0] + nv[1] + nv[2]) * 8));
        for (int g = 0; g < 3; g++) A.g[g].v = g == 0 ? dv[0] : A.g[g - 1].v + nv[g - 1];
    }
    BCHK(h, scratch_get(&dmean, 4 * (size_t)NZ * 8));
    BCHK(h, scratch_get(&dpart, npart * 8));
    // the sums lie end to end: copies of up to 16 KiB to the host are made by a kernel, larger
    // ones by the DMA engines, which also clear freed memory and may be busy with that (a
    // small budget took 260 us for 12 ms after another handle's 300 MB were freed, now 155)
    BCHK(h, scratch_get(&dsum, std::max(n4, nacc) * 8));
    lay.resize(std::max(n4, nacc));
    // 1. snapshot planes and layer means
    for (int g = 0; g < 3; g++) {
        const FileGrid F = file_grid(h, g);
        const BudGrid &G = A.g[g];
        const int nch = bud_chunks(G.X, G.Y, G.rows);
        by_storage(h, F.lat->c(), [&](auto *lat) {
            using S = std::remove_const_t<std::remove_pointer_t<decltype(lat)>>;
            hipLaunchKernelGGL(k_bud_fill<S>, dim3((unsigned)(G.Z * nch)), dim3(BT), 0, h->stream, lat, F.wall, G, F.zlo,
                               F.kwall, dpart);
        });
        hipLaunchKernelGGL(k_bud_segsum, dim3((unsigned)((G.Z * 4 + 3) / 4)), dim3(BT), 0, h->stream,
                           (const double *)dpart, G.Z, nch, 4, dsum + off[g][0]);
        BCHK(h, hipGetLastError());
    }
    BCHK(h, hipMemcpyAsync(lay.data(), dsum, n4 * 8, hipMemcpyDeviceToHost, h->stream));
    BCHK(h, hipStreamSynchronize(h->stream));
    for (int g = 0; g < 3; g++) {
        const BudGrid &G = A.g[g];
        for (int k = G.m0; k < G.m1; k++)
            for (int c = 0; c < 4; c++)
                mean[(size_t)c * NZ + G.base + k] = lay[off[g][0] + (size_t)k * 4 + c] / (double)(G.X * G.Y);
    }
    BCHK(h, hipMemcpyAsync(dmean, mean.data(), mean.size() * 8, hipMemcpyHostToDevice, h->stream));
    // 2. per-node terms over the layers of the node passes
    A.mean = dmean;
    for (int g = 0; g < 3; g++) {
        const BudGrid &G = A.g[g];
        const int nch = bud_chunks(G.X, G.Y, G.rows), nk = G.k1 - G.k0;
        hipLaunchKernelGGL(k_bud_nodes, dim3((unsigned)(nk * nch)), dim3(BT), 0, h->stream, A, g, dpart);
        hipLaunchKernelGGL(k_bud_segsum, dim3((unsigned)((nk * NACC + 3) / 4)), dim3(BT), 0, h->stream,
                           (const double *)dpart, nk, nch, (int)NACC, dsum + off[g][1]);
        BCHK(h, hipGetLastError());
    }
    BCHK(h, hipMemcpyAsync(lay.data(), dsum, nacc * 8, hipMemcpyDeviceToHost, h->stream));
    BCHK(h, hipStreamSynchronize(h->stream));
    for (int g = 0; g < 3; g++) {
        const BudGrid &G = A.g[g];
        for (int k = G.k0; k < G.k1; k++)
            for (int c = 0; c < NACC; c++)
                acc[(size_t)c * NZ + G.base + k] = lay[off[g][1] + (size_t)(k - G.k0) * NACC + c];
    }
    if (ufl) {
        const size_t np = (size_t)A.g[1].X * A.g[1].Y;
        BCHK(h, scratch_get(&dpl, 2 * np * 8));
        hipLaunchKernelGGL(k_bud_plane, dim3((unsigned)((np + BT - 1) / BT)), dim3(BT), 0, h->stream, A, 4, dpl, dpl + np);
        BCHK(h, hipGetLastError());
        BCHK(h, hipMemcpyAsync(ufl, dpl, np * 8, hipMemcpyDeviceToHost, h->stream));
        BCHK(h, hipMemcpyAsync(vfl, dpl + np, np * 8, hipMemcpyDeviceToHost, h->stream));
        BCHK(h, hipStreamSynchronize(h->stream));
    }
    // 3. the profile tail
    bud_dudz(mean.data(), zdf, zdc, GR, dUdz.data());
    bud_finish(h->p, mean.data(), dUdz.data(), acc, turb, vort, ke);
done:
    (void)scratch_put(h->stream, {dv[0], dv[1], dv[2], dmean, dpart, dsum, dpl});
    return rc;
}

// ---- time averages of the per-snapshot profiles ----------------------------------------
// The reference averages the per-snapshot files afterwards with its serial
// post-processor: time_stat.c:132-210 (turb-fld-2d: the mean of every profile except
// UTIN, VTIN, WTIN and DTIN, whose squares it averages), vorticity.c:73-98 (the
// squares of the three vorticity rms) and Ebudget.c:184-300 (the mean of every budget
// term).  Here the same sums are folded at each snapshot, in FP64, in the handle: the
// per-snapshot pass over the lattices is the device's work; the fold adds 52 profiles
// of NZ values per snapshot.
namespace {
constexpr int BUD_ROWS = 19 + 3 + 30;
// turb rows averaged as squares: UTIN VTIN WTIN (3..5) and DTIN (8); every vort row
inline bool bud_squared(int row) { return row == 3 || row == 4 || row == 5 || row == 8 || (row >= 19 && row < 22); }
}  // namespace

extern "C" int dnsg_budget2d_accumulate(dnsg_t *h, double *turb, double *vort, double *ke) {
    if (!h || !h->stream) return DNSG_ERR_ARG;
    const int NZ = h->d.NZ;
    std::vector<double> prof((size_t)BUD_ROWS * NZ);
    double *t = prof.data(), *v = t + 19 * (size_t)NZ, *k = v + 3 * (size_t)NZ;
    int rc = dnsg_budget2d(h, t, v, k, nullptr, nullptr);
    if (rc) return rc;
    if (h->bud_acc.size() != prof.size()) {
        h->bud_acc.assign(prof.size(), 0.);
        h->bud_count = 0;
    }
    for (int r = 0; r < BUD_ROWS; r++)
        for (int z = 0; z < NZ; z++) {
            const double x = prof[(size_t)r * NZ + z];
            h->bud_acc[(size_t)r * NZ + z] += bud_squared(r) ? x * x : x;
        }
    h->bud_count++;
    if (turb) memcpy(turb, t, 19 * (size_t)NZ * 8);
    if (vort) memcpy(vort, v, 3 * (size_t)NZ * 8);
    if (ke) memcpy(ke, k, 30 * (size_t)NZ * 8);
    return DNSG_OK;
}

extern "C" int dnsg_budget2d_average(dnsg_t *h, double *turb, double *vort, double *ke, long *count) {
    if (!h || !turb || !vort || !ke) return DNSG_ERR_ARG;
    const int NZ = h->d.NZ;
    if (count) *count = h->bud_count;
    if (h->bud_count == 0) {
        h->err = "no snapshot folded: call dnsg_budget2d_accumulate first";
        return DNSG_ERR_STATE;
    }
    double *dst[3] = {turb, vort, ke};
    const int rows[3] = {19, 3, 30};
    int r0 = 0;
    for (int g = 0; g < 3; g++) {
        for (size_t i = 0; i < (size_t)rows[g] * NZ; i++) dst[g][i] = h->bud_acc[(size_t)r0 * NZ + i] / h->bud_count;
        r0 += rows[g];
    }
    return DNSG_OK;
}

extern "C" int dnsg_budget2d_reset(dnsg_t *h) {
    if (!h) return DNSG_ERR_ARG;
    h->bud_acc.clear();
    h->bud_count = 0;
    return DNSG_OK;
}
