// k_band2.hip -- both band substeps of a gratio-2 coarse step in one pass over the
// band lattices.
//
// With gratio 2 a coarse step runs xfcomputations twice on each band, with the
// coarse->fine fill of the interface layer between them (main:1347-1365), so a
// two-launch step reads and writes every band value twice.  The first substep's
// result feeds only the second: the first fill writes just the interface layer,
// which the first substep does not store (it is rewritten by the transfer), and the
// fill reads only the interface planes.  So the fill runs first, into the output
// lattice's interface layer, and one workgroup then carries a tile of the band
// through both substeps, keeping the intermediate state on chip:
//   * a workgroup has NR waves, one per row of the tile and its ring; a lane holds NPL
//     adjacent nodes of its row.  The first substep is collided on all 64 NPL columns
//     and NR rows, the second on all but the outermost lane and row on each side (the
//     ring), so a tile is 62 NPL columns by NR - 2 rows, all layers.  Large tiles have 12
//     waves and two nodes per lane (FP64 one), small ones 8 waves and one node, which
//     halves a layer's chain and leaves fewer CUs idle on small lattices (band2_pick.hpp);
//     huge ones are large tiles whose buffer resources are rows, for layers of 2 GiB and more
//     (a resource for each row costs the FP64 launch 9 more spilled registers and 3%);
//   * the workgroup marches through the layers from the interface towards the wall.
//     At layer t it collides the first substep's input and puts the 18 streamed
//     values of each node into LDS; after a barrier every node of the tile takes the
//     values that arrive at it from layer t toward the interface, has everything that
//     streams into layer t-1 (the rest was kept in registers from earlier layers),
//     collides that again (the second substep) and pushes the result to its targets
//     in the output lattice with the wall rules; then it takes the values that stay in
//     layer t or go on toward the wall out of LDS, and a second barrier frees it;
//   * the interface layer (t = 0) takes the first fill's values from the output
//     lattice; the layer next to the wall (t = nz-1) takes its values coming from
//     the wall by the wall rules in pull form: for a direction b leaving the wall,
//     halfway bounce-back of the node's own opp(b) value when the wall cells at
//     (x, y) and (x, y) - e_b (in plane) are both no-slip (-1), else specular
//     reflection of mirror(b) from the node (x, y) - e_b, exactly the writes of
//     xfcomputations.c:230-239 seen from the receiving node.
// Every collision and store is the two-launch path's on the same inputs, so the
// result is bit for bit the same.  HBM traffic per band node and coarse step drops
// from 2 x (19 reads + 19 writes) to 19 reads (+ the ring, largely from L2) and 19
// writes.
//
// The same launch sums, per row and tile of b2_cols() columns, the first substep's
// pre-collision moments for encalc2 and wshearstr (LatArgs::red, B2_RED doubles) or, in
// flux mode, the destination-weighted sums of the second substep's writes
// (LatArgs::dsum, 2 doubles) beside the wall-stress part.  A lane adds up its layers and
// a wave reduces once per tile: reduced at every layer, the sums took 4% of the launch.
#include <algorithm>

#include "internal.hpp"
#include "lattice.hpp"
#include "stream_common.hpp"

namespace dnsg {

namespace {

template <class S, int TILE>
constexpr int npl() { return b2_npl(TILE, sizeof(S)); }  // nodes per lane
template <class S, int TILE>
constexpr bool early() { return npl<S, TILE>() == 1; }  // when the next layer is loaded (band2_tile)

// March coordinate t: 0 at the interface layer, nz-1 next to the wall.  A direction
// moves t by ez for the upper band (interface = stored layer 0) and by -ez for the
// lower band (interface = stored layer nz-1).
template <int SIDE>
constexpr int ezt(int q) { return SIDE ? EZ[q] : -EZ[q]; }
// class of a direction: 0 along the layer, 1 toward the wall, 2 toward the interface
template <int SIDE>
constexpr int cls(int q) { return ezt<SIDE>(q) == 0 ? 0 : (ezt<SIDE>(q) > 0 ? 1 : 2); }
// register slot of a direction within its class: along the layer (EZ = 0) q = 0..4 ->
// 0..4, 7..10 -> 5..8; out of the layer by in-plane offset
constexpr int slot(int q) {
    if (EZ[q] == 0) return q < 5 ? q : q - 2;
    return EX[q] > 0 ? 1 : EX[q] < 0 ? 2 : EY[q] > 0 ? 3 : EY[q] < 0 ? 4 : 0;
}

// LDS plane of a direction: 10 out of the layer, then 8 along it, which are kept twice
// (even and odd layers): those of a layer are read one layer later
constexpr int plane(int q) { return EZ[q] != 0 ? (q < 7 ? q - 5 : q - 9) : (q < 5 ? q + 9 : q + 7); }
constexpr int ALONG = 8, NPLANES = 10 + 2 * ALONG;

// NPL adjacent values of a lane: one value (FP64) or a pair
__device__ __forceinline__ void load_n(Rsrc R, unsigned v, unsigned s, const double *p, double (&o)[1]) { o[0] = buf_load(R, v, s, p); }
template <class S>
__device__ __forceinline__ void load_n(Rsrc R, unsigned v, unsigned s, const S *p, float (&o)[2]) { buf_load_pair(R, v, s, p, o[0], o[1]); }

template <class S>
__device__ __forceinline__ void load_n(Rsrc R, unsigned v, unsigned s, const S *p, float (&o)[1]) { o[0] = buf_load(R, v, s, p); }

template <class S, int TILE, int SIDE, bool DS>
__device__ __forceinline__ void band2_tile(const LatArgs &L, int tile, typename ComputeOf<S>::T *lds, int8_t *wcl) {
    using T = typename ComputeOf<S>::T;
    constexpr int NR = b2_rows(TILE), TY = NR - 2;  // rows of the workgroup, one wave each, and of the tile
    constexpr int NPL = npl<S, TILE>(), CW = 64 * NPL, OX = 62 * NPL;
    auto each_n = [](auto &&f) __attribute__((always_inline)) { unroll<0, NPL>(f); };
    const int nx = L.nx, ny = L.ny, nz = L.nz;
    const int tilesx = (nx + OX - 1) / OX;
    const int tx = tile % tilesx, ty = tile / tilesx;
    const int x0 = tx * OX, y0 = ty * TY;
    const int w = min(OX, nx - x0), th = min(TY, ny - y0);
    // the wave index as a scalar: row addresses and row conditions are wave-uniform
    const int r = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const S *__restrict__ cur = static_cast<const S *>(L.cur);
    S *__restrict__ nxt = static_cast<S *>(L.nxt);
    const T G = (T)(L.gscale * L.force[0]);
    const T om = (T)L.omega;
    const int8_t *__restrict__ wc = SIDE ? L.whi : L.wlo;
    const bool rowok = r < th + 2, core_row = r >= 1 && r <= th;
    const int ya = y0 - 1 + r, y = ya < 0 ? ya + ny : (ya >= ny ? ya - ny : ya);
    const int ym = y == 0 ? ny - 1 : y - 1, yp = y == ny - 1 ? 0 : y + 1;
    // this lane's first column; lanes past the right ring column repeat it
    const int lc = min(lane, w / NPL + 1);
    const int xa = x0 - NPL + NPL * lc, x = xa < 0 ? xa + nx : (xa >= nx ? xa - nx : xa);
    const bool core = core_row && lane >= 1 && lane <= w / NPL;
    // byte offsets in a row: this lane's nodes (loads), and the targets of e_x = 0, +1, -1
    constexpr unsigned ES = sizeof(S);
    const unsigned vx = (unsigned)x * ES;
    const unsigned vs0 = core ? vx : DROP;
    unsigned vsp = DROP, vsm = DROP;
    if (core && (NPL == 1 || x + NPL != nx)) vsp = x + 1 == nx ? 0 : vx + ES;
    if (core && (NPL == 1 || x != 0)) vsm = x == 0 ? (unsigned)(nx - 1) * ES : vx - ES;
    // a pair of targets across the periodic edge is stored one value at a time
    const bool edge = NPL == 2 && (x0 == 0 || x0 + w == nx);
    const bool ep = core && x + NPL == nx, em = core && x == 0;
    // a resource is a layer, or a row where layers are too large for one
    constexpr bool ROWS = TILE == B2_HUGE;
    const unsigned layer_bytes = ROWS ? (unsigned)Q * nx * ES : (unsigned)ny * Q * nx * ES;
    // scalar offset of direction q of row yy within it
    auto soff = [&](int yy, int q) { return ROWS ? (unsigned)q * nx * ES : (unsigned)(yy * Q + q) * nx * ES; };
    // LDS: plane q-1 of [NR][CW]; this lane's place in it
    T *const me = lds + r * CW + NPL * lane;
    constexpr int PL = NR * CW;

    T fin[NPL][Q];                       // first-substep input of the next layer
    T q0[NPL];                           // rest direction of layer t-1
    T wo[NPL][5], wn[NPL][5];            // arrived toward the wall: from layer t-2, t-1
    double srho = 0., smom = 0.;         // layer-weighted sums of the first substep's input (encalc2)
    double sdm = 0., sdd = 0.;           // ... and of the second substep's writes (flux controller)
    each_n([&](auto nc) {
        constexpr int n = decltype(nc)::value;
        q0[n] = T(0);
#pragma unroll
        for (int k = 0; k < 5; k++) wo[n][k] = wn[n][k] = T(0);
    });

    auto row_rsrc = [&](const S *lat, int t, int yy) {
        return buf_rsrc(lat + ((size_t)(SIDE ? t : nz - 1 - t) * ny + yy) * Q * nx, layer_bytes);
    };
    auto layer_rsrc = [&](const S *lat, int t) {  // ... of layer t, or of its row y
        if constexpr (ROWS) return row_rsrc(lat, t, y);
        else return buf_rsrc(lat + (size_t)(SIDE ? t : nz - 1 - t) * ny * Q * nx, layer_bytes);
    };
    auto load_q = [&](Rsrc R, int q, T (&v)[NPL]) __attribute__((always_inline)) { load_n(R, vx, soff(y, q), cur, v); };
    auto load_layer = [&](Rsrc R, T (&f)[NPL][Q]) __attribute__((always_inline)) {
        unroll<0, Q>([&](auto qc) {
            constexpr int q = decltype(qc)::value;
            T v[NPL];
            load_q(R, q, v);
            each_n([&](auto nc) { constexpr int n = decltype(nc)::value; f[n][q] = v[n]; });
        });
    };
    // value of direction q arriving at node n of this lane, from the layer whose values are
    // at m (me, for the directions along a layer plus that layer's copy)
    auto arrive = [&](auto qc, int n, const T *m) {
        constexpr int q = decltype(qc)::value;
        return m[plane(q) * PL - EY[q] * CW + n - EX[q]];
    };
    auto collide_all = [&](T (&g)[NPL][Q]) __attribute__((always_inline)) {
        unroll<0, NPL>([&](auto nc) { collide_any(g[decltype(nc)::value], G, om); });
    };

    // push of the second substep's result at layer t
    auto push = [&](int t, const T (&g)[NPL][Q]) __attribute__((always_inline)) {
        const int m = SIDE ? t : nz - 1 - t;
        double sd[3] = {0., 0., 0.}, sx[3] = {0., 0., 0.};  // per class: sums of f and of e_x f
        auto put = [&](Rsrc R, auto qc) {  // R: the target layer
            constexpr int q = decltype(qc)::value;
            const unsigned so = soff(EY[q] > 0 ? yp : (EY[q] < 0 ? ym : y), q);
            if constexpr (ROWS && EY[q] != 0)
                R = row_rsrc(nxt, cls<SIDE>(q) == 1 ? t + 1 : (cls<SIDE>(q) == 2 ? t - 1 : t), EY[q] > 0 ? yp : ym);
            const unsigned vo = EX[q] > 0 ? vsp : (EX[q] < 0 ? vsm : vs0);
            if constexpr (NPL == 1) {
                buf_store<0>(R, vo, so, nxt, g[0][q]);
            } else {
                // e_x = +-1: a dword-aligned 8-byte store in FP32; FP16 has no such store, so two
                if constexpr (EX[q] == 0 || sizeof(S) == 4) {
                    buf_store_pair<0>(R, vo, so, nxt, g[0][q], g[1][q]);
                } else {
                    buf_store<0>(R, vo, so, nxt, g[0][q]);
                    buf_store<0>(R, vo == DROP ? DROP : vo + ES, so, nxt, g[1][q]);
                }
                if constexpr (EX[q] != 0) {
                    if (edge) {
                        const bool e = EX[q] > 0 ? ep : em;
                        buf_store<0>(R, e ? (unsigned)(nx - 1) * ES : DROP, so, nxt, g[0][q]);
                        buf_store<0>(R, e ? 0u : DROP, so, nxt, g[1][q]);
                    }
                }
            }
            if constexpr (DS) {
                each_n([&](auto nc) {
                    constexpr int n = decltype(nc)::value;
                    const double v = read_back<S, q>(g[n][q]);
                    sd[cls<SIDE>(q)] += v;
                    if constexpr (EX[q] > 0) sx[cls<SIDE>(q)] += v;
                    if constexpr (EX[q] < 0) sx[cls<SIDE>(q)] -= v;
                });
            }
        };
        if (t >= 1) {  // along the interface layer: rewritten by the next fill
            const Rsrc R = layer_rsrc(nxt, t);
            unroll<0, Q>([&](auto qc) {
                if constexpr (cls<SIDE>(decltype(qc)::value) == 0) put(R, qc);
            });
        }
        if (t >= 2) {  // into the interface layer (t = 1) or out of the band (t = 0): not written
            const Rsrc R = layer_rsrc(nxt, t - 1);
            unroll<0, Q>([&](auto qc) {
                if constexpr (cls<SIDE>(decltype(qc)::value) == 2) put(R, qc);
            });
        }
        if (t < nz - 1) {
            const Rsrc R = layer_rsrc(nxt, t + 1);
            unroll<0, Q>([&](auto qc) {
                if constexpr (cls<SIDE>(decltype(qc)::value) == 1) put(R, qc);
            });
        } else if (core) {
            // onto the wall (xfcomputations.c:230-239): halfway bounce-back where both wall
            // cells are no-slip, else specular reflection
            unroll<0, Q>([&](auto qc) {
                constexpr int q = decltype(qc)::value;
                if constexpr (cls<SIDE>(q) == 1) {
                    const int yt = EY[q] > 0 ? yp : (EY[q] < 0 ? ym : y);
                    unroll<0, NPL>([&](auto nc) {
                        constexpr int n = decltype(nc)::value;
                        const int c = NPL * lane + n;
                        const bool bb = wcl[r * CW + c] == -1 && wcl[(r + EY[q]) * CW + c + EX[q]] == -1;
                        const int xn = x + n, xt = EX[q] > 0 ? (xn + 1 == nx ? 0 : xn + 1)
                                                             : (EX[q] < 0 ? (xn == 0 ? nx - 1 : xn - 1) : xn);
                        if (bb) store_s(nxt + lat_at(OPP[q], (size_t)m * ny + y, xn, nx), g[n][q]);
                        else store_s(nxt + lat_at(MIR[q], (size_t)m * ny + yt, xt, nx), g[n][q]);
                        if constexpr (DS) {  // lands in this layer
                            const double v = read_back<S, q>(g[n][q]);
                            sd[0] += v;
                            if constexpr (EX[q] > 0) sx[0] += bb ? -v : v;
                            if constexpr (EX[q] < 0) sx[0] += bb ? v : -v;
                        }
                    });
                }
            });
        }
        if constexpr (DS) {
            if (core) {
                constexpr int up = SIDE ? 1 : -1;  // stored-layer step toward the wall
                const double w0 = dest_w(L, m), w1 = t < nz - 1 ? dest_w(L, m + up) : 0., w2 = t >= 1 ? dest_w(L, m - up) : 0.;
                sdm += weighted(w0, sx[0]) + weighted(w1, sx[1]) + weighted(w2, sx[2]);
                sdd += weighted(w0, sd[0]) + weighted(w1, sd[1]) + weighted(w2, sd[2]);
            }
        }
    };

    if (rowok) {
        if (NPL * lane < w + 2 * NPL)  // the tile's wall codes, ring included
            each_n([&](auto nc) { constexpr int n = decltype(nc)::value; wcl[r * CW + NPL * lane + n] = wc[(size_t)y * nx + x + n]; });
        load_layer(layer_rsrc(cur, 0), fin);
    }
    double *const rec = L.red ? L.red + ((size_t)y * tilesx + tx) * B2_RED : nullptr;
    for (int t = 0; t < nz; t++) {
        T *const me0 = me + (t & 1) * ALONG * PL;               // along-layer copy of layer t
        const T *const me1 = me + ((t & 1) ^ 1) * ALONG * PL;   // ... of layer t-1
        // The next layer's loads: issued here, before this layer's collision, with one node
        // per lane, so they have the whole iteration to arrive (FP64 Re_tau=180 launch 1.250
        // -> 1.203 ms, FP32 small tiles on 512 x 256 x 8 bands 99 -> 86 us); with two, which
        // would spill (FP32 0.749 -> 0.812 ms), after it, into the registers it frees.
        T f[NPL][Q];
        T(&F)[NPL][Q] = early<S, TILE>() ? f : fin;
        if constexpr (early<S, TILE>()) {
            unroll<0, Q>([&](auto qc) {
                constexpr int q = decltype(qc)::value;
                each_n([&](auto nc) { f[decltype(nc)::value][q] = fin[decltype(nc)::value][q]; });
            });
            if (rowok && t + 1 < nz) load_layer(layer_rsrc(cur, t + 1), fin);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (rowok) {
            // ---- first substep at layer t: collide, sum, share
            PreSums<T> ps[NPL];
            each_n([&](auto nc) { ps[decltype(nc)::value] = collide_any(F[decltype(nc)::value], G, om); });
            if (L.red) {
                const double wt = DS ? 0. : dest_w(L, SIDE ? t : nz - 1 - t);  // flux control: encalc2 comes from the writes
                if (wt != 0. && core)
                    each_n([&](auto nc) {
                        srho += wt * pre_rho(ps[decltype(nc)::value]);
                        smom += wt * (double)ps[decltype(nc)::value].mx;
                    });
                if (t >= nz - 3 && core_row) {  // the layers of the wall-stress stencil
                    double u = 0., d = 0.;
                    if (core)
                        each_n([&](auto nc) {
                            u += pre_u(ps[decltype(nc)::value]);
                            d += pre_rho(ps[decltype(nc)::value]);
                        });
                    u = wave_sum64(u);
                    if (lane == 0) rec[3 + (nz - 1 - t)] = u;
                    if (t == (SIDE ? nz - 3 : nz - 1)) {
                        d = wave_sum64(d);
                        if (lane == 0) rec[2] = d;
                    }
                }
            }
            each_n([&](auto nc) {
                constexpr int n = decltype(nc)::value;
                // FP16 storage: one launch per substep stores this result in FP16 and the
                // second substep reads it back; round it the same way here
                if constexpr (sizeof(S) == 2)
                    unroll<0, Q>([&](auto qc) {
                        constexpr int q = decltype(qc)::value;
                        F[n][q] = __half2float(__float2half(F[n][q]));
                    });
                unroll<1, Q>([&](auto qc) {
                    constexpr int q = decltype(qc)::value;
                    (EZ[q] == 0 ? me0 : me)[plane(q) * PL + n] = F[n][q];
                });
            });
        }
        T f0[NPL];
        each_n([&](auto nc) { f0[decltype(nc)::value] = F[decltype(nc)::value][0]; });
        __syncthreads();
        if constexpr (!early<S, TILE>()) {
            if (rowok && t + 1 < nz) load_layer(layer_rsrc(cur, t + 1), fin);
        }
        __builtin_amdgcn_sched_barrier(0);
        // ---- second substep at layer t-1
        T g[NPL][Q];
        if (t >= 1 && core_row) {
            unroll<0, Q>([&](auto qc) {
                constexpr int q = decltype(qc)::value;
                each_n([&](auto nc) {
                    constexpr int n = decltype(nc)::value;
                    if constexpr (q == 0) g[n][q] = q0[n];
                    else if constexpr (cls<SIDE>(q) == 0) g[n][q] = arrive(qc, n, me1);
                    else if constexpr (cls<SIDE>(q) == 1) g[n][q] = wo[n][slot(q)];
                    else g[n][q] = arrive(qc, n, me);
                });
            });
            if (t == 1) {  // the interface layer: the first fill's values (those toward the wall are in wo)
                const Rsrc R = layer_rsrc(nxt, 0);
                unroll<0, Q>([&](auto qc) {
                    constexpr int q = decltype(qc)::value;
                    if constexpr (cls<SIDE>(q) != 1) {
                        T v[NPL];
                        load_q(R, q, v);
                        each_n([&](auto nc) { g[decltype(nc)::value][q] = v[decltype(nc)::value]; });
                    }
                });
            }
            collide_all(g);
        }
        // every wave waits here for the next layer's loads and the previous layer's stores,
        // so that the pushes below are the only vector memory operations in flight when the
        // loaded values are first used
        __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0), no wait on expcnt / lgkmcnt
        __builtin_amdgcn_sched_barrier(0);
        if (t >= 1 && core_row) push(t - 1, g);
        if (core_row) {
            each_n([&](auto nc) {
                constexpr int n = decltype(nc)::value;
#pragma unroll
                for (int k = 0; k < 5; k++) wo[n][k] = wn[n][k];
                q0[n] = f0[n];
                unroll<1, Q>([&](auto qc) {
                    constexpr int q = decltype(qc)::value;
                    if constexpr (cls<SIDE>(q) == 1) wn[n][slot(q)] = arrive(qc, n, me);
                });
            });
            if (t == 0) {  // the interface layer: the first fill's values
                const Rsrc R = layer_rsrc(nxt, 0);
                unroll<0, Q>([&](auto qc) {
                    constexpr int q = decltype(qc)::value;
                    if constexpr (cls<SIDE>(q) == 1) {
                        T v[NPL];
                        load_q(R, q, v);
                        each_n([&](auto nc) { wo[decltype(nc)::value][slot(q)] = v[decltype(nc)::value]; });
                    }
                });
            }
        }
        if (t + 1 < nz) __syncthreads();
    }
    // ---- second substep at the layer next to the wall; the directions leaving the wall
    // from this layer's toward-the-wall values (wn, and LDS at this node)
    if (core_row) {
        T g[NPL][Q];
        each_n([&](auto nc) {
            constexpr int n = decltype(nc)::value;
            const int c = NPL * lane + n;
            const bool own = wcl[r * CW + c] == -1;
            unroll<0, Q>([&](auto qc) {
                constexpr int q = decltype(qc)::value;
                if constexpr (q == 0) g[n][q] = q0[n];
                else if constexpr (cls<SIDE>(q) == 0) g[n][q] = arrive(qc, n, me + ((nz - 1) & 1) * ALONG * PL);
                else if constexpr (cls<SIDE>(q) == 1) g[n][q] = wo[n][slot(q)];
                else {
                    const bool bb = own && core && wcl[(r - EY[q]) * CW + c - EX[q]] == -1;
                    const T vbb = me[plane(OPP[q]) * PL + n];
                    g[n][q] = bb ? vbb : wn[n][slot(MIR[q])];
                }
            });
        });
        collide_all(g);
        push(nz - 1, g);
        if (!DS && rec) {
            const double a = wave_sum64(srho), b = wave_sum64(smom);
            if (lane == 0) {
                rec[0] = a;
                rec[1] = b;
            }
        }
        if (DS && L.dsum) {
            const double a = wave_sum64(sdm), b = wave_sum64(sdd);
            if (lane == 0) {
                double *o = L.dsum + 2 * ((size_t)y * tilesx + tx);
                o[0] = a;
                o[1] = b;
            }
        }
    }
}

// waves per SIMD that the registers must allow: FP32 in small tiles four, two workgroups a CU
template <class S, int TILE>
constexpr int min_waves() { return TILE == B2_SMALL && sizeof(S) == 4 ? 4 : 1; }

template <class S, int TILE, bool DS>
__global__ __launch_bounds__(64 * b2_rows(TILE), (min_waves<S, TILE>())) void k_band2(Batch<LatArgs> P) {
    using T = typename ComputeOf<S>::T;
    constexpr int NR = b2_rows(TILE), CW = 64 * npl<S, TILE>(), PAD = 2;  // PAD: ring lanes read one value beside the array and ignore it
    __shared__ T lds[NPLANES * NR * CW + 2 * PAD];
    __shared__ int8_t wcl[NR * CW + 2 * PAD];  // the tile's wall codes, ring included
    if (halted(P.halt)) return;
    const int bg = xcd_remap(blockIdx.x, gridDim.x);
    const int it = batch_find(P.first, P.n, bg);
    const LatArgs &L = P.it[it];
    const int tile = bg - P.first[it];
    if (L.lo_kind == BOUND_WALL) band2_tile<S, TILE, 0, DS>(L, tile, lds + PAD, wcl + PAD);
    else band2_tile<S, TILE, 1, DS>(L, tile, lds + PAD, wcl + PAD);
}

}  // namespace

template <class S, int TILE>
static void band2_launch(hipStream_t s, const Batch<LatArgs> &P, bool ds) {
    const dim3 g(P.first[BATCH_MAX]), b(64 * b2_rows(TILE));
    if (ds) hipLaunchKernelGGL((k_band2<S, TILE, true>), g, b, 0, s, P);
    else hipLaunchKernelGGL((k_band2<S, TILE, false>), g, b, 0, s, P);
}

template <class S>
static void band2_launch(hipStream_t s, const Batch<LatArgs> &P, bool ds, int tile) {
    if (tile == B2_HUGE) band2_launch<S, B2_HUGE>(s, P, ds);
    else if (sizeof(S) == 2 || tile == B2_LARGE) band2_launch<S, B2_LARGE>(s, P, ds);
    else if constexpr (sizeof(S) != 2) band2_launch<S, B2_SMALL>(s, P, ds);
}

hipError_t launch_band2(hipStream_t s, const LatArgs *bands, int prec, int tile, const int *halt) {
    const int elem = prec == DNSG_PREC_FP64 ? 8 : (prec == DNSG_PREC_FP32 ? 4 : 2);
    if (tile == B2_OFF || (tile == B2_SMALL && elem == 2) || (tile != B2_HUGE && !buf_fits(bands[0].nx, bands[0].ny, elem)))
        return hipErrorInvalidValue;
    Batch<LatArgs> P;
    P.halt = halt;
    P.n = 2;
    int blocks = 0;
    for (int i = 0; i < BATCH_MAX; i++) {
        P.it[i] = bands[i < 2 ? i : 0];
        P.first[i] = blocks;
        if (i < 2) blocks += band2_tiles(bands[i].nx, bands[i].ny, elem, tile);
    }
    P.first[BATCH_MAX] = blocks;
    const bool ds = bands[0].dsum != nullptr || bands[1].dsum != nullptr;
    if (prec == DNSG_PREC_FP64) band2_launch<double>(s, P, ds, tile);
    else if (prec == DNSG_PREC_FP32) band2_launch<float>(s, P, ds, tile);
    else band2_launch<__half>(s, P, ds, tile);
    return hipGetLastError();
}

}  // namespace dnsg
