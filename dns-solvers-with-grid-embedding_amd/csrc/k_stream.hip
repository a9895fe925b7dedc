// k_stream.hip -- fused BGK collide + push-stream on the coarse grid and the
// wall bands, the initial-state kernel and the AoS <-> SoA transposes.
//
// A workgroup owns CS_THREADS nodes of a row (two chunks of them in the paired form, a run
// of consecutive nodes of the layer in the flat form): its reads are 19 contiguous vectors
// of the row block, its writes the same vectors of the 9 neighbouring rows shifted by e_x.
//
// Boundary rules at the stored z ends (xfcomputations.c:215-442):
//   BOUND_DROP  populations leaving the lattice are not written (the bounded
//               layers of the reference: coarse k = 0, zdc-1 and the band
//               interface layers, which the interface transfer rewrites)
//   BOUND_WALL  the target is a wall node with code s(t) in {-1, -2}; with
//               s1 the code below the source node:
//                 s(t) = -1 and s1 = -1  -> halfway bounce-back  f(x, opp q)
//                 otherwise              -> specular reflection  f(x + e_xy, mirror q)
#include "internal.hpp"
#include "lattice.hpp"
#include "stream_common.hpp"

namespace dnsg {

// Sums of a node's stores by the layer step k = -1, 0, 1 of their destination; the layer
// weights are applied once at the end (LatArgs::dsum).  Every direction is added at its
// own step, stored or not: the layers that take no store (beyond an end, or rewritten by
// an interface transfer) have weight 0.  The sums stay in registers only while no branch
// chooses between two of them, so the wall rules select values, not members.
struct DestSums {
    double dl = 0., dc = 0., dh = 0., xl = 0., xc = 0., xh = 0.;
    template <int k>
    __device__ __forceinline__ void mass(double v) {
        if constexpr (k < 0) dl += v;
        if constexpr (k == 0) dc += v;
        if constexpr (k > 0) dh += v;
    }
    template <int k, int ex>
    __device__ __forceinline__ void mom(double v) {
        const double e = ex > 0 ? v : -v;
        if constexpr (ex != 0 && k < 0) xl += e;
        if constexpr (ex != 0 && k == 0) xc += e;
        if constexpr (ex != 0 && k > 0) xh += e;
    }
    __device__ __forceinline__ void into(RowSums &rs, const LatArgs &L, int z) const {
        const double wl = dest_w(L, z - 1), wc = dest_w(L, z), wh = dest_w(L, z + 1);
        rs.dd += weighted(wl, dl) + weighted(wc, dc) + weighted(wh, dh);
        rs.dm += weighted(wl, xl) + weighted(wc, xc) + weighted(wh, xh);
    }
};

// Scatter form for the node at x of row (y, z): collide, then write each direction to its
// target (x + e_x, y + e_y, z + e_z) with the boundary rules above.  With DS, the
// destination-weighted sums of the writes go into rs.
template <class S, bool DS, class T>
__device__ __forceinline__ void cs_scatter(const LatArgs &L, const S *__restrict__ cur, S *__restrict__ nxt, int row,
                                           int x, T G, T om, bool red, RowSums &rs) {
    const int nx = L.nx, ny = L.ny, nz = L.nz;
    T f[Q];
    unroll<0, Q>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        f[q] = load_s(cur + (size_t)q * nx + x);
    });
    const auto pre = collide_any(f, G, om);
    if (red) rs.add<S>(pre);
    const int y = row % ny, z = row / ny;
    const bool lo_edge = (z == 0), hi_edge = (z == nz - 1);
    const int ym = (y == 0) ? ny - 1 : y - 1, yp = (y == ny - 1) ? 0 : y + 1;
    const int xm = (x == 0) ? nx - 1 : x - 1, xp = (x == nx - 1) ? 0 : x + 1;
    DestSums dst;
    unroll<0, Q>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        if constexpr (DS) {
            dst.mass<EZ[q]>(read_back<S, q>(f[q]));
            dst.mom<EZ[q], EX[q]>(read_back<S, q>(f[q]));
        }
        const int xt = (EX[q] > 0) ? xp : (EX[q] < 0 ? xm : x);
        const int yt = (EY[q] > 0) ? yp : (EY[q] < 0 ? ym : y);
        if constexpr (EZ[q] != 0) {
            const bool at_end = (EZ[q] < 0) ? lo_edge : hi_edge;
            if (at_end) {
                const int kind = (EZ[q] < 0) ? L.lo_kind : L.hi_kind;
                if (kind == BOUND_WALL) {
                    const int8_t *wc = (EZ[q] < 0) ? L.wlo : L.whi;
                    const bool bb = wc[(size_t)yt * nx + xt] == -1 && wc[(size_t)y * nx + x] == -1;
                    if (bb) store_s(nxt + lat_at(OPP[q], (size_t)row, x, nx), f[q]);
                    else store_s(nxt + lat_at(MIR[q], (size_t)z * ny + yt, xt, nx), f[q]);
                    if constexpr (DS) {  // it lands in this layer
                        const double v = read_back<S, q>(f[q]);
                        dst.mass<0>(v);
                        dst.mom<0, EX[q]>(bb ? -v : v);
                    }
                }
                return;
            }
        }
        const int zt = z + EZ[q];
        if ((zt == 0 && L.skip_lo) || (zt == nz - 1 && L.skip_hi)) return;
        store_s(nxt + lat_at(q, (size_t)zt * ny + yt, xt, nx), f[q]);
    });
    if constexpr (DS) dst.into(rs, L, z);
}

// Aligned form for chunk x0 .. x0 + CS_THREADS - 1 of row (y, z) (nx a multiple of
// CS_THREADS): the workgroup also collides the two nodes just outside its chunk
// and passes the e_x != 0 values one lane along (shuffles within a wave, LDS
// between waves), so that every store of direction q lands on the workgroup's own
// positions of the target row: whole cache lines, written once.  Each thread
// stores, at its own x, the value arriving there from x - e_x; the set of writes
// is exactly the scatter form's.
// The nine rows (y + e_y, z + e_z) that a row's values go to, each a buffer resource of its
// own, so that layers of any size can be addressed: what is kept is the addresses of the
// three layers and the row offsets, uniform over the workgroup.
template <class S>
struct RowTargets {
    const char *lo, *mid, *hi;
    size_t ym, yc, yp;
    unsigned line, row;
    __device__ __forceinline__ RowTargets(const LatArgs &L, const S *nxt, int y, int z) {
        line = __builtin_amdgcn_readfirstlane(L.nx * (int)sizeof(S));
        y = __builtin_amdgcn_readfirstlane(y);
        row = Q * line;
        const size_t bytes = (size_t)row * L.ny;
        mid = reinterpret_cast<const char *>(nxt) + z * bytes;
        lo = mid - bytes;  // beyond an end: takes no stores
        hi = mid + bytes;
        ym = (size_t)row * (y == 0 ? L.ny - 1 : y - 1);
        yc = (size_t)row * y;
        yp = (size_t)row * (y == L.ny - 1 ? 0 : y + 1);
    }
    template <int ey, int ez>
    __device__ __forceinline__ Rsrc at() const {
        return buf_rsrc((ez < 0 ? lo : (ez > 0 ? hi : mid)) + (ey < 0 ? ym : (ey > 0 ? yp : yc)), row);
    }
    template <int ey>
    __device__ __forceinline__ unsigned off(unsigned q_line) const { return q_line; }
};

// The three layers a layer's values go to, as buffer resources (layers below 2 GiB)
template <class S>
struct LayerTargets {
    Rsrc lo, mid, hi;
    __device__ __forceinline__ LayerTargets(const LatArgs &L, const S *nxt, int z) {
        const unsigned bytes = Q * (unsigned)L.nx * sizeof(S) * (unsigned)L.ny;
        const char *m = reinterpret_cast<const char *>(nxt) + (size_t)z * bytes;
        lo = buf_rsrc(z > 0 ? m - bytes : m, bytes);  // the layer beyond an end takes no stores
        mid = buf_rsrc(m, bytes);
        hi = buf_rsrc(z < L.nz - 1 ? m + bytes : m, bytes);
    }
    template <int ez>
    __device__ __forceinline__ Rsrc layer() const { return ez < 0 ? lo : (ez > 0 ? hi : mid); }
};

// The nine rows as offsets into the three layers' resources (layers below 2 GiB): 46 scalar
// instructions fewer a wave than a resource for each row.  It shows where instructions bound
// the launch, in FP16: a Re_tau=180 step 880 us against 886 (flux control 966 against 975).
// FP64 and FP32 take the rows in all sizes (no difference).
template <class S>
struct LayerRowTargets : LayerTargets<S> {
    unsigned ym, yc, yp;
    __device__ __forceinline__ LayerRowTargets(const LatArgs &L, const S *nxt, int y, int z) : LayerTargets<S>(L, nxt, z) {
        y = __builtin_amdgcn_readfirstlane(y);
        const unsigned row = Q * __builtin_amdgcn_readfirstlane(L.nx * (int)sizeof(S));
        ym = row * (unsigned)(y == 0 ? L.ny - 1 : y - 1);
        yc = row * (unsigned)y;
        yp = row * (unsigned)(y == L.ny - 1 ? 0 : y + 1);
    }
    template <int ey, int ez>
    __device__ __forceinline__ Rsrc at() const { return this->template layer<ez>(); }
    template <int ey>
    __device__ __forceinline__ unsigned off(unsigned q_line) const { return (ey < 0 ? ym : (ey > 0 ? yp : yc)) + q_line; }
};

// Flat form: the workgroup takes CS_THREADS consecutive nodes of layer z, from node n0 on,
// so every lane has a node whatever the row length (by rows, a 144-node row filled 144 of
// 256 lanes and a 285-node one 285 of 512).  A lane's row is its own, so its offsets are
// per lane, 32 bits each; layer and direction stay scalar.  The writes are the scatter
// form's.
template <class S, bool DS, class T>
__device__ __forceinline__ void cs_flat(const LatArgs &L, const S *__restrict__ lat, S *__restrict__ nxt, int z, int n0,
                                        T G, T om, bool red, RowSums &rs) {
    const int nx = L.nx, ny = L.ny, nz = L.nz, n = nx * ny;
    const bool ok = n0 + (int)threadIdx.x < n;
    const unsigned id = ok ? n0 + threadIdx.x : n0;
    const int y = (int)(id / (unsigned)nx), x = (int)id - y * nx;
    constexpr unsigned ES = sizeof(S);
    const unsigned line = __builtin_amdgcn_readfirstlane(nx * (int)ES), row = Q * line;
    const LayerTargets<S> in(L, lat, z), to(L, nxt, z);
    T f[Q];
    unroll<0, Q>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        f[q] = buf_load(in.mid, y * row + x * ES, q * line, lat);
    });
    const auto pre = collide_any(f, G, om);
    if (red && ok) rs.add<S>(pre);
    const bool lo_edge = (z == 0), hi_edge = (z == nz - 1);
    const int ym = (y == 0) ? ny - 1 : y - 1, yp = (y == ny - 1) ? 0 : y + 1;
    const int xm = (x == 0) ? nx - 1 : x - 1, xp = (x == nx - 1) ? 0 : x + 1;
    // a lane without a node: every offset at or past DROP
    const unsigned om_ = ok ? ym * row : DROP, oc = ok ? y * row : DROP, op = ok ? yp * row : DROP;
    DestSums dst;
    unroll<0, Q>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        if constexpr (DS) {
            dst.mass<EZ[q]>(read_back<S, q>(f[q]));
            dst.mom<EZ[q], EX[q]>(read_back<S, q>(f[q]));
        }
        const int xt = (EX[q] > 0) ? xp : (EX[q] < 0 ? xm : x);
        if constexpr (EZ[q] != 0) {
            const bool at_end = (EZ[q] < 0) ? lo_edge : hi_edge;
            if (at_end) {  // uniform over the workgroup
                const int kind = (EZ[q] < 0) ? L.lo_kind : L.hi_kind;
                if (kind == BOUND_WALL && ok) {
                    const int yt = (EY[q] > 0) ? yp : (EY[q] < 0 ? ym : y);
                    const int8_t *wc = (EZ[q] < 0) ? L.wlo : L.whi;
                    const bool bb = wc[(size_t)yt * nx + xt] == -1 && wc[(size_t)y * nx + x] == -1;
                    if (bb) store_s(nxt + lat_at(OPP[q], (size_t)z * ny + y, x, nx), f[q]);
                    else store_s(nxt + lat_at(MIR[q], (size_t)z * ny + yt, xt, nx), f[q]);
                    if constexpr (DS) {  // it lands in this layer
                        const double v = read_back<S, q>(f[q]);
                        dst.mass<0>(v);
                        dst.mom<0, EX[q]>(bb ? -v : v);
                    }
                }
                return;
            }
        }
        const int zt = z + EZ[q];
        if ((zt == 0 && L.skip_lo) || (zt == nz - 1 && L.skip_hi)) return;
        const unsigned o = ((EY[q] > 0) ? op : (EY[q] < 0 ? om_ : oc)) + xt * ES;
        buf_store<0>(to.template layer<EZ[q]>(), o, q * line, nxt, f[q]);
    });
    if (DS && ok) dst.into(rs, L, z);
}

template <class S, bool DS, class T>
__device__ __forceinline__ void cs_aligned_chunk(const LatArgs &L, const S *__restrict__ cur, S *__restrict__ nxt,
                                                 int row, int x0, T G, T om, bool red, RowSums &rs) {
    constexpr int NW = CS_THREADS / 64;
    __shared__ T hb[2][Q];      // post-collision halo nodes x0 - 1, x0 + CS_THREADS
    __shared__ T wb[NW][2][Q];  // per wave: last lane's e_x > 0, first lane's e_x < 0 values
    const int nx = L.nx, ny = L.ny, nz = L.nz;
    const int y = row % ny, z = row / ny;
    const bool lo_edge = (z == 0), hi_edge = (z == nz - 1);
    const int ym = (y == 0) ? ny - 1 : y - 1, yp = (y == ny - 1) ? 0 : y + 1;
    const int t = threadIdx.x, lane = t & 63, w = t >> 6, x = x0 + t;
    constexpr unsigned ES = sizeof(S);
    constexpr int NT = 2;
    const unsigned vx = (unsigned)x * ES, lb = __builtin_amdgcn_readfirstlane(nx * (int)ES);
    const Rsrc in = buf_rsrc(cur, Q * lb);
    if (t == 0 || t == CS_THREADS - 1) {
        const int side = t == 0 ? 0 : 1;
        int xh = side == 0 ? x0 - 1 : x0 + CS_THREADS;
        xh = xh < 0 ? xh + nx : (xh >= nx ? xh - nx : xh);
        T g[Q];
        unroll<0, Q>([&](auto qc) {
            constexpr int q = decltype(qc)::value;
            g[q] = load_s(cur + (size_t)q * nx + xh);
        });
        collide_any(g, G, om);
        unroll<0, Q>([&](auto qc) {
            constexpr int q = decltype(qc)::value;
            if constexpr (EX[q] != 0) hb[side][q] = g[q];
        });
    }
    T f[Q];
    unroll<0, Q>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        f[q] = buf_load(in, vx, q * lb, cur);
    });
    const auto pre = collide_any(f, G, om);
    if (red) rs.add<S>(pre);
    unroll<0, Q>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        if constexpr (EX[q] > 0) {
            if (lane == 63) wb[w][0][q] = f[q];
        } else if constexpr (EX[q] < 0) {
            if (lane == 0) wb[w][1][q] = f[q];
        }
    });
    __syncthreads();
    DestSums dst;
    const RowTargets<S> to(L, nxt, y, z);
    const int xm = (x == 0) ? nx - 1 : x - 1, xp = (x == nx - 1) ? 0 : x + 1;
    unroll<0, Q>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        T v = f[q];  // the value arriving at x: post-collision f_q of node x - e_x
        if constexpr (EX[q] > 0) {
            v = __shfl_up(f[q], 1, 64);
            if (lane == 0) v = (w == 0) ? hb[0][q] : wb[w - 1][0][q];
        } else if constexpr (EX[q] < 0) {
            v = __shfl_down(f[q], 1, 64);
            if (lane == 63) v = (w == NW - 1) ? hb[1][q] : wb[w + 1][1][q];
        }
        if constexpr (DS) {
            dst.mass<EZ[q]>(read_back<S, q>(v));
            dst.mom<EZ[q], EX[q]>(read_back<S, q>(v));
        }
        const int yt = (EY[q] > 0) ? yp : (EY[q] < 0 ? ym : y);
        if constexpr (EZ[q] != 0) {
            const bool at_end = (EZ[q] < 0) ? lo_edge : hi_edge;
            if (at_end) {
                const int kind = (EZ[q] < 0) ? L.lo_kind : L.hi_kind;
                if (kind == BOUND_WALL) {
                    const int8_t *wc = (EZ[q] < 0) ? L.wlo : L.whi;
                    // specular reflection of the source x - e_x into (x, yt), unless it bounces back
                    const int xs = (EX[q] > 0) ? xm : (EX[q] < 0 ? xp : x);
                    const bool spec = !(wc[(size_t)yt * nx + x] == -1 && wc[(size_t)y * nx + xs] == -1);
                    if (spec) store_s(nxt + lat_at(MIR[q], (size_t)z * ny + yt, x, nx), v);
                    // halfway bounce-back of this node's own value
                    const int xt = (EX[q] > 0) ? xp : (EX[q] < 0 ? xm : x);
                    const bool bb = wc[(size_t)yt * nx + xt] == -1 && wc[(size_t)y * nx + x] == -1;
                    if (bb) store_s(nxt + lat_at(OPP[q], (size_t)row, x, nx), f[q]);
                    if constexpr (DS) {  // both land in this layer
                        const double a = spec ? read_back<S, q>(v) : 0., b = bb ? read_back<S, q>(f[q]) : 0.;
                        dst.mass<0>(a + b);
                        dst.mom<0, EX[q]>(a - b);
                    }
                }
                return;
            }
        }
        const int zt = z + EZ[q];
        if ((zt == 0 && L.skip_lo) || (zt == nz - 1 && L.skip_hi)) return;
        buf_store<NT>(to.template at<EY[q], EZ[q]>(), vx, to.template off<EY[q]>(q * lb), nxt, v);
    });
    if constexpr (DS) dst.into(rs, L, z);
}

// Paired form (FP32 / FP16 storage, nx a multiple of 2 CS_THREADS): the workgroup
// takes nodes x0 .. x0 + 2 CS_THREADS - 1, thread t the pair x = x0 + 2t, x + 1, read
// and written as one 2-value access per direction.  As in the aligned form, the
// workgroup also collides the nodes x0 - 1 and x0 + 2 CS_THREADS, and each thread
// stores at (x, x + 1) the values arriving there from (x, x + 1) - e_x: for e_x = +1
// the pair (f(x - 1), f(x)), f(x - 1) being the previous thread's second node; for
// e_x = -1 the pair (f(x + 1), f(x + 2)).  At a wall end the pair's two positions
// take the wall rules one value at a time.  The writes are exactly the scatter
// form's.  Threads below / from CS_THREADS / 2 hold the first / second chunk's nodes.
// Paired stores are non-temporal, like the aligned form's.  Measured on the
// Re_tau=180 lattices: FP32 coarse 0.952 -> 0.938 ms and band 0.479 -> 0.472 ms; FP16
// within 1%.
template <class S, bool DS, template <class> class Targets, class T>
__device__ __forceinline__ void cs_paired_chunk(const LatArgs &L, const S *__restrict__ cur, S *__restrict__ nxt,
                                                int row, int x0, T G, T om, bool red, RowSums &rs) {
    constexpr int NW = CS_THREADS / 64, NP = 2 * CS_THREADS;
    __shared__ T hb[2][Q];      // post-collision nodes x0 - 1, x0 + NP
    __shared__ T wb[NW][2][Q];  // per wave: last lane's second node e_x > 0, first lane's first node e_x < 0
    const int nx = L.nx, ny = L.ny, nz = L.nz;
    const int y = row % ny, z = row / ny;
    const bool lo_edge = (z == 0), hi_edge = (z == nz - 1);
    const int ym = (y == 0) ? ny - 1 : y - 1, yp = (y == ny - 1) ? 0 : y + 1;
    const int t = threadIdx.x, lane = t & 63, w = t >> 6, x = x0 + 2 * t;
    constexpr unsigned ES = sizeof(S);
    const unsigned vx = (unsigned)x * ES, lb = __builtin_amdgcn_readfirstlane(nx * (int)ES);
    const Rsrc in = buf_rsrc(cur, Q * lb);
    if (t == 0 || t == CS_THREADS - 1) {
        const int side = t == 0 ? 0 : 1;
        int xh = side == 0 ? x0 - 1 : x0 + NP;
        xh = xh < 0 ? xh + nx : (xh >= nx ? xh - nx : xh);
        T g[Q];
        unroll<0, Q>([&](auto qc) {
            constexpr int q = decltype(qc)::value;
            g[q] = load_s(cur + (size_t)q * nx + xh);
        });
        collide_any(g, G, om);
        unroll<0, Q>([&](auto qc) {
            constexpr int q = decltype(qc)::value;
            if constexpr (EX[q] != 0) hb[side][q] = g[q];
        });
    }
    T f0[Q], f1[Q];
    unroll<0, Q>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        buf_load_pair(in, vx, q * lb, cur, f0[q], f1[q]);
    });
    const auto p0 = collide_any(f0, G, om);
    if (red) rs.add<S>(p0);
    // one collision after the other: interleaved by the scheduler they take 102 VGPRs (FP32)
    __builtin_amdgcn_sched_barrier(0);
    const auto p1 = collide_any(f1, G, om);
    if (red) rs.add<S>(p1);
    unroll<0, Q>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        if constexpr (EX[q] > 0) {
            if (lane == 63) wb[w][0][q] = f1[q];
        } else if constexpr (EX[q] < 0) {
            if (lane == 0) wb[w][1][q] = f0[q];
        }
    });
    __syncthreads();
    DestSums dst;
    const Targets<S> to(L, nxt, y, z);
    unroll<0, Q>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        // the values arriving at x and x + 1, and the sources they leave from
        T va = f0[q], vb = f1[q];
        if constexpr (EX[q] > 0) {
            T s = __shfl_up(f1[q], 1, 64);
            if (lane == 0) s = (w == 0) ? hb[0][q] : wb[w - 1][0][q];
            va = s;
            vb = f0[q];
        } else if constexpr (EX[q] < 0) {
            T s = __shfl_down(f0[q], 1, 64);
            if (lane == 63) s = (w == NW - 1) ? hb[1][q] : wb[w + 1][1][q];
            va = f1[q];
            vb = s;
        }
        if constexpr (DS) {
            const double a = read_back<S, q>(va) + read_back<S, q>(vb);
            dst.mass<EZ[q]>(a);
            dst.mom<EZ[q], EX[q]>(a);
        }
        const int yt = (EY[q] > 0) ? yp : (EY[q] < 0 ? ym : y);
        if constexpr (EZ[q] != 0) {
            const bool at_end = (EZ[q] < 0) ? lo_edge : hi_edge;
            if (at_end) {
                const int kind = (EZ[q] < 0) ? L.lo_kind : L.hi_kind;
                if (kind == BOUND_WALL) {
                    const int8_t *wc = (EZ[q] < 0) ? L.wlo : L.whi;
                    // positions x + i (i = 0, 1): the arriving value (source x + i - e_x)
                    // is reflected specularly into (x + i, yt) unless it bounces back,
                    // and the node's own value bounces back where its target is no-slip
                    unroll<0, 2>([&](auto ic) {
                        constexpr int i = decltype(ic)::value;
                        const int xi = x + i;
                        const int xm = (xi == 0) ? nx - 1 : xi - 1, xp = (xi == nx - 1) ? 0 : xi + 1;
                        const T v = i == 0 ? va : vb, own = i == 0 ? f0[q] : f1[q];
                        const int xs = (EX[q] > 0) ? xm : (EX[q] < 0 ? xp : xi);
                        const bool spec = !(wc[(size_t)yt * nx + xi] == -1 && wc[(size_t)y * nx + xs] == -1);
                        if (spec) store_s(nxt + lat_at(MIR[q], (size_t)z * ny + yt, xi, nx), v);
                        const int xt = (EX[q] > 0) ? xp : (EX[q] < 0 ? xm : xi);
                        const bool bb = wc[(size_t)yt * nx + xt] == -1 && wc[(size_t)y * nx + xi] == -1;
                        if (bb) store_s(nxt + lat_at(OPP[q], (size_t)row, xi, nx), own);
                        if constexpr (DS) {
                            const double a = spec ? read_back<S, q>(v) : 0., b = bb ? read_back<S, q>(own) : 0.;
                            dst.mass<0>(a + b);
                            dst.mom<0, EX[q]>(a - b);
                        }
                    });
                }
                return;
            }
        }
        const int zt = z + EZ[q];
        if ((zt == 0 && L.skip_lo) || (zt == nz - 1 && L.skip_hi)) return;
        buf_store_pair<2>(to.template at<EY[q], EZ[q]>(), vx, to.template off<EY[q]>(q * lb), nxt, va, vb);
    });
    if constexpr (DS) dst.into(rs, L, z);
}

__device__ __forceinline__ void write_sums(double *red, size_t e, const RowSums &s) {
    red[e + 0] = s.rho;
    red[e + 1] = s.mom;
    red[e + 2] = s.u;
}

// Workgroup sums of the fused reductions (wave shuffles, then LDS over the waves), written
// as `parts` consecutive partials from e on, each over CS_THREADS / parts threads.
template <bool DS>
__device__ __forceinline__ void write_block_sums(const LatArgs &L, const RowSums &s, size_t e, int parts) {
    constexpr int NW = CS_THREADS / 64;
    __shared__ double lds[5][NW];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const bool red = L.red != nullptr, ds = DS && L.dsum != nullptr;
    if (red) {
        const double a = wave_sum64(s.rho), b = wave_sum64(s.mom), c = wave_sum64(s.u);
        if (lane == 0) { lds[0][wid] = a; lds[1][wid] = b; lds[2][wid] = c; }
    }
    if (ds) {
        const double a = wave_sum64(s.dm), b = wave_sum64(s.dd);
        if (lane == 0) { lds[3][wid] = a; lds[4][wid] = b; }
    }
    __syncthreads();
    if ((int)threadIdx.x < parts) {
        RowSums t;
        const int nw = NW / parts;
        for (int w = threadIdx.x * nw; w < (int)(threadIdx.x + 1) * nw; w++) {
            if (red) { t.rho += lds[0][w]; t.mom += lds[1][w]; t.u += lds[2][w]; }
            if (ds) { t.dm += lds[3][w]; t.dd += lds[4][w]; }
        }
        e += threadIdx.x;
        if (red) write_sums(L.red, e * RED_W, t);
        if (ds) { L.dsum[2 * e] = t.dm; L.dsum[2 * e + 1] = t.dd; }
    }
}

template <class S, bool DS, template <class> class PairedTargets>
__device__ __forceinline__ void collide_stream(const Batch<LatArgs> &P) {
    using T = typename ComputeOf<S>::T;
    if (halted(P.halt)) return;
    const int bg = xcd_remap(blockIdx.x, gridDim.x);
    const int it = batch_find(P.first, P.n, bg);
    const LatArgs &L = P.it[it];
    const int nx = L.nx, ny = L.ny;
    const int b = bg - P.first[it];
    const S *__restrict__ base = static_cast<const S *>(L.cur);
    S *__restrict__ nxt = static_cast<S *>(L.nxt);
    const T G = (T)(L.gscale * L.force[0]);
    const T om = (T)L.omega;
    const bool red = L.red != nullptr;
    RowSums rs;
    size_t e;       // first partial of this workgroup
    int parts = 1;  // ... and how many it writes
    if (L.form == CS_FLAT) {
        const int ppl = cs_parts(CS_FLAT, nx, ny), z = b / ppl;
        cs_flat<S, DS, T>(L, base, nxt, z, (b - z * ppl) * CS_THREADS, G, om, red, rs);
        e = b;
    } else if constexpr (sizeof(S) == 8) {
        // CS_ALIGNED, one (row, chunk) per workgroup: row, y and z are uniform over the workgroup
        const int cpr = cs_chunks(nx), row = b / cpr, chunk = b % cpr;
        cs_aligned_chunk<S, DS, T>(L, base + (size_t)row * Q * nx, nxt, row, chunk * CS_THREADS, G, om, red, rs);
        e = b;
    } else {
        // CS_PAIRED, two chunks of one row per workgroup, two nodes per thread; the
        // workgroup's halves are the two chunks' partials
        const int cpr = cs_chunks(nx), ppr = cpr / 2, row = b / ppr, pc = b % ppr;
        cs_paired_chunk<S, DS, PairedTargets>(L, base + (size_t)row * Q * nx, nxt, row, pc * 2 * CS_THREADS, G, om, red,
                                              rs);
        e = (size_t)row * cpr + 2 * pc;
        parts = 2;
    }
    if (red || (DS && L.dsum)) write_block_sums<DS>(L, rs, e, parts);  // uniform per workgroup
}

template <class S, bool DS>
__global__ __launch_bounds__(CS_THREADS) void k_collide_stream(Batch<LatArgs> P) {
    if constexpr (sizeof(S) == 2) collide_stream<S, DS, LayerRowTargets>(P);
    else collide_stream<S, DS, RowTargets>(P);
}
// FP16 where a paired lattice has layers of 2 GiB and more
template <bool DS>
__global__ __launch_bounds__(CS_THREADS) void k_collide_half_rows(Batch<LatArgs> P) {
    collide_stream<__half, DS, RowTargets>(P);
}

// CS_WIDE: one (row, chunk) of one lattice per workgroup in the scatter form
template <class S, bool DS>
__global__ __launch_bounds__(CS_THREADS) void k_collide_wide(LatArgs L, const int *halt) {
    using T = typename ComputeOf<S>::T;
    if (halted(halt)) return;
    const int cpr = cs_chunks(L.nx), row = blockIdx.x / cpr, x = (blockIdx.x % cpr) * CS_THREADS + threadIdx.x;
    RowSums rs;
    if (x < L.nx)
        cs_scatter<S, DS, T>(L, static_cast<const S *>(L.cur) + (size_t)row * Q * L.nx, static_cast<S *>(L.nxt), row, x,
                             (T)(L.gscale * L.force[0]), (T)L.omega, L.red != nullptr, rs);
    if (L.red || (DS && L.dsum)) write_block_sums<DS>(L, rs, blockIdx.x, 1);
}

template <class S>
static void launch_wide(hipStream_t s, const LatArgs &L, const int *halt) {
    const dim3 g((unsigned)(L.nz * cs_blocks(CS_WIDE, L.nx, L.ny))), b(CS_THREADS);
    if (L.dsum) hipLaunchKernelGGL((k_collide_wide<S, true>), g, b, 0, s, L, halt);
    else hipLaunchKernelGGL((k_collide_wide<S, false>), g, b, 0, s, L, halt);
}

hipError_t launch_collide_stream(hipStream_t s, const LatArgs *lats, int nlat, int prec, const int *halt) {
    for (int i = 0; i < nlat;) {
        Batch<LatArgs> P;
        P.halt = halt;
        P.n = 0;
        bool ds = false, rows = false;
        int blocks = 0;
        for (; i < nlat && P.n < BATCH_MAX; i++) {
            const LatArgs &L = lats[i];
            if (L.form == CS_WIDE) {
                if (prec == DNSG_PREC_FP64) launch_wide<double>(s, L, halt);
                else if (prec == DNSG_PREC_FP32) launch_wide<float>(s, L, halt);
                else launch_wide<__half>(s, L, halt);
                const hipError_t e = hipGetLastError();
                if (e != hipSuccess) return e;
                continue;
            }
            ds = ds || L.dsum != nullptr;
            rows = rows || (L.form == CS_PAIRED && !buf_fits(L.nx, L.ny, sizeof(__half)));
            P.it[P.n] = L;
            P.first[P.n++] = blocks;
            blocks += L.nz * cs_blocks(L.form, L.nx, L.ny);
        }
        for (int k = P.n; k <= BATCH_MAX; k++) P.first[k] = blocks;
        if (blocks == 0) continue;
        const dim3 g(blocks), b(CS_THREADS);
        if (prec == DNSG_PREC_FP64) {
            if (ds) hipLaunchKernelGGL((k_collide_stream<double, true>), g, b, 0, s, P);
            else hipLaunchKernelGGL((k_collide_stream<double, false>), g, b, 0, s, P);
        } else if (prec == DNSG_PREC_FP32) {
            if (ds) hipLaunchKernelGGL((k_collide_stream<float, true>), g, b, 0, s, P);
            else hipLaunchKernelGGL((k_collide_stream<float, false>), g, b, 0, s, P);
        } else if (rows) {
            if (ds) hipLaunchKernelGGL(k_collide_half_rows<true>, g, b, 0, s, P);
            else hipLaunchKernelGGL(k_collide_half_rows<false>, g, b, 0, s, P);
        } else {
            if (ds) hipLaunchKernelGGL((k_collide_stream<__half, true>), g, b, 0, s, P);
            else hipLaunchKernelGGL((k_collide_stream<__half, false>), g, b, 0, s, P);
        }
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

// ---- initial state --------------------------------------------------------------
// Counter-based PRNG (splitmix64 finaliser) over (seed, grid, component, node):
// independent of the traversal order, so every node's noise is fixed by its
// global index in the reference layout [x][y][k] of that grid.
__device__ __forceinline__ uint64_t mix64(uint64_t z) {
    z += 0x9E3779B97F4A7C15ULL;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
    return z ^ (z >> 31);
}
__device__ __forceinline__ double prng_sym(uint64_t seed, int grid, int comp, uint64_t node) {
    const uint64_t b =
        mix64(mix64(seed) ^ mix64(((uint64_t)(grid & 0xff) << 56) ^ ((uint64_t)(comp & 0xff) << 48) ^ node));
    const double u = (double)(b >> 11) * 0x1.0p-53;
    return 2. * u - 1.;
}

struct InitArgs {
    void *dst;
    int nx, ny, nz;     // stored extents
    int zdf_or_zdc;     // reference z extent of this grid
    int kofs;           // reference k = stored z + kofs
    int grid;           // 0 coarse, 1 lower, 2 upper (PRNG stream)
    int kind;           // DNSG_INIT_*
    int GR, zdf, zdc, NZs;
    uint64_t seed;
    double u_max, noise;
};

template <class S>
__global__ __launch_bounds__(256) void k_init(InitArgs A) {
    const size_t n = (size_t)A.nx * A.ny * A.nz;
    const size_t id = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= n) return;
    const int x = (int)(id % A.nx), y = (int)((id / A.nx) % A.ny), z = (int)(id / ((size_t)A.nx * A.ny));
    const int k = z + A.kofs;
    S *dst = static_cast<S *>(A.dst);
    double f[Q];
    if (A.kind == DNSG_INIT_REST) {
        unroll<0, Q>([&](auto qc) { f[decltype(qc)::value] = WQ[decltype(qc)::value]; });
    } else {
        double dist;
        if (A.grid == 0) dist = A.GR * (k - 1) + (A.zdf - 1 - 0.5);
        else if (A.grid == 1) dist = k - 0.5;
        else dist = k + A.GR * (A.zdc - 3) + A.zdf - 1. - 0.5;
        const double zeta = dist / ((double)(A.NZs - 2));
        const double amp = A.noise * A.u_max;
        const uint64_t node = ((uint64_t)x * A.ny + y) * A.zdf_or_zdc + k;
        const double u0 = 4. * A.u_max * zeta * (1. - zeta) + amp * prng_sym(A.seed, A.grid, 0, node);
        const double u1 = amp * prng_sym(A.seed, A.grid, 1, node);
        const double u2 = amp * prng_sym(A.seed, A.grid, 2, node);
        const double v = u0 * u0 + u1 * u1 + u2 * u2;
        unroll<0, Q>([&](auto qc) {
            constexpr int q = decltype(qc)::value;
            f[q] = feq64<q>(1., u0, u1, u2, v);
        });
    }
    const size_t row = (size_t)z * A.ny + y;
    unroll<0, Q>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        if constexpr (sizeof(S) == 8) store_s((double *)dst + lat_at(q, row, x, A.nx), f[q]);
        else store_s(dst + lat_at(q, row, x, A.nx), (float)(f[q] - WQ[q]));
    });
}

hipError_t launch_init_lattice(hipStream_t s, dnsg_ctx *h, int grid, void *dst) {
    InitArgs A;
    const Grid &g = grid == 0 ? h->coarse : (grid == 1 ? h->lower : h->upper);
    A.dst = dst;
    A.nx = g.nx; A.ny = g.ny; A.nz = g.nz;
    A.zdf_or_zdc = grid == 0 ? h->d.zdc : h->d.zdf;
    A.kofs = grid == 1 ? 1 : 0;
    A.grid = grid;
    A.kind = h->p.init_kind;
    A.GR = h->d.GR; A.zdf = h->d.zdf; A.zdc = h->d.zdc; A.NZs = h->d.NZs;
    A.seed = h->p.seed; A.u_max = h->p.u_max; A.noise = h->p.noise;
    const size_t n = g.nodes();
    dim3 grd((unsigned)((n + 255) / 256)), blk(256);
    if (h->p.precision == DNSG_PREC_FP64) hipLaunchKernelGGL(k_init<double>, grd, blk, 0, s, A);
    else if (h->p.precision == DNSG_PREC_FP32) hipLaunchKernelGGL(k_init<float>, grd, blk, 0, s, A);
    else hipLaunchKernelGGL(k_init<__half>, grd, blk, 0, s, A);
    return hipGetLastError();
}

// ---- AoS (reference layouts [x][y][k][19]) <-> SoA ----------------------------------
// gl = 0: the file layout [nx][ny][nz_aos][19]; gl = 1: the in-memory layout
// [nx+1][ny+1][nz_aos][19] whose last x-plane and y-row are ghost cells.
template <class S>
__global__ __launch_bounds__(256) void k_aos_to_soa(const double *__restrict__ aos, S *__restrict__ soa, int nx,
                                                    int ny, int nz_aos, int z0, int nz, int gl) {
    const size_t n = (size_t)nx * ny * nz * Q;
    const size_t id = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= n) return;
    const int x = (int)(id % nx), q = (int)((id / nx) % Q);
    const size_t row = id / ((size_t)nx * Q);
    const int y = (int)(row % ny), z = (int)(row / ny);
    const double v = aos[(((size_t)x * (ny + gl) + y) * nz_aos + (z + z0)) * Q + q];
    if constexpr (sizeof(S) == 8) soa[id] = v;
    else store_s(soa + id, (float)(v - WQ[q]));
}

// every node of the host layout, ghost cells as their periodic images
template <class S>
__global__ __launch_bounds__(256) void k_soa_to_aos(const S *__restrict__ soa, double *__restrict__ aos, int nx,
                                                    int ny, int nz_aos, int z0, int nz, int gl) {
    const int mx = nx + gl, my = ny + gl;
    const size_t n = (size_t)mx * my * nz * Q;
    const size_t id = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= n) return;
    const int x = (int)(id % mx), q = (int)((id / mx) % Q);
    const size_t r = id / ((size_t)mx * Q);
    const int y = (int)(r % my), z = (int)(r / my);
    const int xs = x < nx ? x : x - nx, ys = y < ny ? y : y - ny;
    const size_t src = lat_at(q, (size_t)z * ny + ys, xs, nx);
    double v;
    if constexpr (sizeof(S) == 8) v = soa[src];
    else v = (double)load_s(soa + src) + WQ[q];
    aos[(((size_t)x * my + y) * nz_aos + (z + z0)) * Q + q] = v;
}

hipError_t launch_aos_to_soa(hipStream_t s, const double *aos, void *soa, int nx, int ny, int nz_aos, int z0, int nz,
                             int prec, int gl) {
    const size_t n = (size_t)nx * ny * nz * Q;
    dim3 grd((unsigned)((n + 255) / 256)), blk(256);
    if (prec == DNSG_PREC_FP64)
        hipLaunchKernelGGL(k_aos_to_soa<double>, grd, blk, 0, s, aos, (double *)soa, nx, ny, nz_aos, z0, nz, gl);
    else if (prec == DNSG_PREC_FP32)
        hipLaunchKernelGGL(k_aos_to_soa<float>, grd, blk, 0, s, aos, (float *)soa, nx, ny, nz_aos, z0, nz, gl);
    else
        hipLaunchKernelGGL(k_aos_to_soa<__half>, grd, blk, 0, s, aos, (__half *)soa, nx, ny, nz_aos, z0, nz, gl);
    return hipGetLastError();
}

hipError_t launch_soa_to_aos(hipStream_t s, const void *soa, double *aos, int nx, int ny, int nz_aos, int z0, int nz,
                             int prec, int gl) {
    const size_t n = (size_t)(nx + gl) * (ny + gl) * nz * Q;
    dim3 grd((unsigned)((n + 255) / 256)), blk(256);
    if (prec == DNSG_PREC_FP64)
        hipLaunchKernelGGL(k_soa_to_aos<double>, grd, blk, 0, s, (const double *)soa, aos, nx, ny, nz_aos, z0, nz, gl);
    else if (prec == DNSG_PREC_FP32)
        hipLaunchKernelGGL(k_soa_to_aos<float>, grd, blk, 0, s, (const float *)soa, aos, nx, ny, nz_aos, z0, nz, gl);
    else
        hipLaunchKernelGGL(k_soa_to_aos<__half>, grd, blk, 0, s, (const __half *)soa, aos, nx, ny, nz_aos, z0, nz, gl);
    return hipGetLastError();
}

}  // namespace dnsg
