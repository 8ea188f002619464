// Discrete adjoint of System::timeStep (detail.h:1539-1570) for Cuspy +
// Laplace1d replicas (no reference counterpart). With the well index of every
// particle taken as a constant at every step (the indices the trajectory
// visited), one step is the map (u, v, a) -> (u1, v3, a3):
//   u1 = u + dt v + dt^2/2 a
//   g  = k_frame (u_frame - u1) + mu (ym - u1) + k L u1     ym = (y_l + y_r) / 2
//   v1 = v + dt a,               a1 = (g - eta v1) / m
//   v2 = v + dt/2 (a + a1),      a2 = (g - eta v2) / m
//   v3 = v + dt/2 (a + a2),      a3 = (g - eta v3) / m
// (L: periodic second difference). The adjoint runs the step backwards for the
// cotangents of (u1, v3, a3) and accumulates the derivatives with respect to
// mu, k, k_frame, eta and the yield positions y_l, y_r of the visited wells.
//
// A run of n steps is split into windows of K steps. For each window, last
// to first: k_adj_record re-runs the window from its checkpoint (the same
// expressions in the same order as the resident kernel, so the same
// trajectory and the same wells) and writes a tape of u1 and v of every step;
// k_adj_reverse then walks the tape backwards. What else a step used follows
// from these and is not written: its acceleration is that of the preceding
// step's last stage, (g - eta v) / m with the g of the preceding u1, and its
// well is the one that holds u1 (a window's wells are walked to from those of
// its checkpoint). Where a walk of the window passed yield positions that do not
// ascend (a user may set any), two wells can hold a slip: the record kernel
// reports it (ADJ_ERR_ROWS) and the host repeats the pass with the wells on
// the tape (tj). Both kernels are bound by the tape's bytes: 64 chains of
// 4096, 2000 steps, record / reverse with u1, v, a and the well (28 bytes per
// particle-step): 3.0 / 4.6 ms, with u1 and v (16 bytes): 1.9 / 3.3
// ms (4.5 / 2.6 TB/s; in the reverse kernel the instructions of a step come
// next).
// The tape is particle-major per step ([step][replica][particle]) and both
// kernels give a thread the particles t, t + T, t + 2T, ... of its segment,
// so that every tape load and store of a wavefront is contiguous; neighbours
// are exchanged through LDS.
//
// k_adj_reverse spreads each replica over tiles (many workgroups per
// replica): a tile walks its particles together with a halo of K + 1
// particles on each side, whose cotangents start from the adjoint state of
// their owners (the cotangents of the forces do not depend on the tape, so a
// halo reads none of it, but for the slip next to the tile's own particles). The cotangent of a particle at the open end of the extended
// segment lacks one neighbour, and the error this makes moves inwards by one
// particle per reversed step (through the second difference of the
// cotangents of the forces), so after the K steps of a window the tile's own
// particles are exact. The adjoint state is double-buffered across windows
// (tiles read their halo from the buffer that no tile writes in the same
// launch); the parameter derivatives are summed per tile and then over the
// tiles in a fixed order (k_adj_params).
#pragma once

#include "fq_physics.hpp"
#include "fq_resident.hpp"

#include <type_traits>

namespace fq {


// Record windows w0 + blockIdx.y (each of min(K, n - w K) steps) from their
// start states, one workgroup per replica, tile and window (blockIdx.x =
// replica * rnt + tile): every window is independent given its checkpoint,
// so all of a group run at once. With one tile per replica the workgroup
// holds the whole periodic chain; with several, a tile steps its particles
// together with a halo of rhalo >= K particles on each side (recomputed from
// their owners' checkpoint with the same expressions: the open ends' error
// moves inwards by one particle per step and never reaches the tile's own
// particles within a window) and writes the tape of its own particles only.
// Thread t holds local particles t + T k (k < SLOTS) of the segment; the
// slips of a step are exchanged through LDS, double-buffered by step parity
// (one barrier per step). RING: one tile per replica (local = global index,
// every particle its own: compile-time offsets of the tape entries).
template <int SLOTS, int MAXT, bool RING>
__global__ void __launch_bounds__(MAXT) k_adj_record(const SysView* __restrict__ views, AdjBuffers ab, int flow,
                                                     double v_frame)
{
    extern __shared__ double sx[]; // [2][E]
    const int r = blockIdx.x / ab.rnt, tile = blockIdx.x % ab.rnt;
    const int64_t w = ab.w0 + blockIdx.y;
    const int steps = (int)(ab.n - w * ab.K < ab.K ? ab.n - w * ab.K : ab.K);
    // this window's start state and tape
    ab.wu += blockIdx.y * ab.ws;
    ab.wv += blockIdx.y * ab.ws;
    ab.wa += blockIdx.y * ab.ws;
    ab.wj += blockIdx.y * ab.ws;
    ab.wuf += blockIdx.y * ab.R;
    ab.tu += blockIdx.y * ab.ts;
    ab.tv += blockIdx.y * ab.ts;
    ab.tuf += blockIdx.y * ab.K * ab.R;
    ab.tj = ab.tj ? ab.tj + blockIdx.y * ab.ts : nullptr;
    const SysView& S = views[r];
    constexpr int T = MAXT; // launched with exactly MAXT threads
    const int t = threadIdx.x;
    const int N = (int)ab.N;
    const int64_t off = (int64_t)r * N;
    constexpr bool ring = RING;
    const int p0 = tile * (int)ab.rtp;
    const int p1 = p0 + (int)ab.rtp < N ? p0 + (int)ab.rtp : N;
    const int H = ring ? 0 : (int)ab.rhalo;
    const int E = ring ? N : (p1 - p0) + 2 * H; // particles of the segment
    const Landscape& L = S.ls;
    const double* const Y = L.y;
    const int64_t nch = L.nchunk;
    const int32_t jmin = (int32_t)L.buffer;
    const int32_t jmax = (int32_t)(L.nchunk - 2 - L.buffer);
    const int64_t Rnp = ab.R * ab.np;

    double u[SLOTS], v[SLOTS], a[SLOTS], yl[SLOTS], yr[SLOTS];
    int32_t jl[SLOTS], pp[SLOTS];
    bool own[SLOTS];
#pragma unroll
    for (int k = 0; k < SLOTS; ++k) {
        u[k] = v[k] = a[k] = yl[k] = yr[k] = 0.0;
        jl[k] = 0;
        const int e = t + T * k;
        int p = e;
        if constexpr (!RING) {
            p = p0 - H + e;
            p = p < 0 ? p + N : (p >= N ? p - N : p);
        }
        pp[k] = p;
        own[k] = e < E && (RING || (e >= H && e < H + (p1 - p0)));
        if (e < E) {
            u[k] = ab.wu[off + p];
            v[k] = ab.wv[off + p];
            a[k] = ab.wa[off + p];
            jl[k] = ab.wj[off + p];
            yl[k] = Y[p * nch + jl[k]];
            yr[k] = Y[p * nch + jl[k] + 1];
        }
    }
    const double dt = S.dt, c2 = 0.5 * dt * dt, hdt = 0.5 * dt, meta = -S.eta, inv_m = S.inv_m, kf = S.k_frame;
    const double dv = v_frame * dt;
    double uf = ab.wuf[r];
    int bad = 0;

    for (int n = 0; n < steps; ++n) {
        double* const xb = sx + (n & 1) * E;
        if (flow) {
            uf = uf + dv;
        }
        const int64_t tn = (int64_t)n * Rnp + (int64_t)r * ab.np;
        if (t == 0 && tile == 0) {
            ab.tuf[(int64_t)n * ab.R + r] = uf;
        }
#pragma unroll
        for (int k = 0; k < SLOTS; ++k) {
            const int e = t + T * k;
            if (e < E) {
                const int64_t q = tn + (RING ? t + T * k : pp[k]);
                u[k] = u[k] + dt * v[k] + c2 * a[k];
                const double x = u[k];
                if (own[k]) {
                    ab.tv[q] = v[k];
                    ab.tu[q] = x;
                }
                if (!(yl[k] <= x && x < yr[k])) {
                    const double* row = Y + (int64_t)pp[k] * nch;
                    int32_t j = jl[k];
                    double lo = yl[k], hi = yr[k];
                    while (x >= hi && j < jmax) {
                        ++j;
                        lo = hi;
                        hi = row[j + 1];
                        bad |= own[k] && hi < lo ? ADJ_ERR_ROWS : 0;
                    }
                    while (x < lo && j > jmin) {
                        --j;
                        hi = lo;
                        lo = row[j];
                        bad |= own[k] && hi < lo ? ADJ_ERR_ROWS : 0;
                    }
                    bad |= own[k] && !(lo <= x && x < hi) ? ADJ_ERR_WALK : 0;
                    jl[k] = j;
                    yl[k] = lo;
                    yr[k] = hi;
                }
                if (ab.tj && own[k]) {
                    ab.tj[q] = jl[k];
                }
                xb[e] = x;
            }
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < SLOTS; ++k) {
            const int e = t + T * k;
            if (e < E) {
                // neighbours: periodic on the ring; at the open ends of a
                // tile's segment, any finite value (the particle's own slip)
                double um, up;
                if (ring) {
                    um = xb[e == 0 ? N - 1 : e - 1];
                    up = xb[e == N - 1 ? 0 : e + 1];
                }
                else {
                    um = e == 0 ? u[k] : xb[e - 1];
                    up = e == E - 1 ? u[k] : xb[e + 1];
                }
                const double fi = chain_force<INT_LAPLACE1D>(S, um, u[k], up);
                const double fp = potential_force<POT_CUSPY>(S, u[k], yl[k], yr[k]);
                const double ff = kf * (uf - u[k]);
                const double sum3 = ff + fp + fi;
                const double vn = v[k], an = a[k];
                double vv = vn + dt * an;
                double f = sum3 + meta * vv;
                double aa = f * inv_m;
                vv = vn + hdt * (an + aa);
                f = sum3 + meta * vv;
                aa = f * inv_m;
                vv = vn + hdt * (an + aa);
                f = sum3 + meta * vv;
                aa = f * inv_m;
                v[k] = vv;
                a[k] = aa;
            }
        }
    }
    if (bad) {
        atomicOr(ab.err, bad);
    }
}

// Walk the tape of one window backwards on one tile of one replica
// (blockIdx.x = replica * nt + tile), updating the adjoint state of the
// tile's particles and its partial parameter derivatives. Since dg/dy_l =
// dg/dy_r = mu/2, one accumulator per particle collects the derivative for
// both yield positions of its current well; it is added to the output when
// the well changes.
//
// One barrier per step: the cotangent G of the force is linear in the
// cotangents after the step alone, so it is exchanged together with the slips
// of the step before, whose force gives this step's acceleration. The tape is
// loaded two steps ahead.
// WELLS: with the wells on the tape.
template <int SLOTS, bool WELLS>
__global__ void __launch_bounds__(ADJ_REV_THREADS) k_adj_reverse(const SysView* __restrict__ views, AdjBuffers ab,
                                                                   int steps)
{
    // neighbour exchange: cotangents of g and slips u1, double-buffered by
    // the parity of their step (a buffer is rewritten two barriers after the
    // one that precedes its reads)
    extern __shared__ double s_x[]; // [2][B] cotangents, [2][B] slips
    __shared__ double s_red[4][ADJ_REV_THREADS / 64];
    const int r = blockIdx.x / ab.nt, tile = blockIdx.x % ab.nt;
    const SysView& S = views[r];
    constexpr int T = ADJ_REV_THREADS;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    constexpr int nw = T / 64;
    const int N = (int)ab.N;
    const int64_t off = (int64_t)r * N;
    const bool ring = ab.nt == 1; // one tile: the whole periodic chain, no halo
    const int p0 = tile * (int)ab.tp;
    const int p1 = p0 + (int)ab.tp < N ? p0 + (int)ab.tp : N;
    const int H = ring ? 0 : (int)ab.halo;
    const int E = ring ? N : (p1 - p0) + 2 * H; // particles of the extended segment
    constexpr int B = adj_rev_stride(SLOTS); // local index e at 1 + e: a neighbour's place on each side
    const double* const Y = S.ls.y;
    const int64_t nch = S.ls.nchunk;
    const int32_t jmin = (int32_t)S.ls.buffer;
    const int32_t jmax = (int32_t)(nch - 2 - S.ls.buffer);
    const int64_t Rnp = ab.R * ab.np;

    const double dt = S.dt, c2 = 0.5 * dt * dt, h = 0.5 * dt, meta = -S.eta, w = S.inv_m, kf = S.k_frame;
    const double mu = S.mu, k = S.k;
    const double e1 = meta * w; // -eta / m
    // The stages' cotangents, a3 = w (g - eta v3), v3 = v + h a + h a2 and so
    // on down to v1 = v + dt a, are multiples of V3 = V + e1 A: of a2 h V3, of
    // v2 e1 h V3, of a1 e1 h^2 V3, of v1 (e1 h)^2 V3
    const double eh = e1 * h, ehh = eh * eh, dehh = dt * ehh, kfm = -(kf + mu);

    // slot i: local index e = t + T i of the extended segment, particle p;
    // own: this tile's; slip: its u1 is read (its own particles and the one
    // next to them on each side)
    int pp[SLOTS];
    bool own[SLOTS], slip[SLOTS], live[SLOTS];
#pragma unroll
    for (int i = 0; i < SLOTS; ++i) {
        const int e = t + T * i;
        live[i] = e < E;
        own[i] = live[i] && (ring || (e >= H && e < H + (p1 - p0)));
        slip[i] = live[i] && (ring || (e >= H - 1 && e < H + (p1 - p0) + 1));
        int q = ring ? e : p0 - H + e;
        q = q < 0 ? q + N : (q >= N ? q - N : q);
        pp[i] = q;
    }
    // U, V, A: cotangents of u, v, a after the step being reversed
    // x, v, lu, d, g, lo, hi: slip, velocity, second difference of the slips,
    // distance to the well's middle, force without damping and the well
    // (index jc) of that step; acc: sum of G over the steps in that well
    double U[SLOTS], V[SLOTS], A[SLOTS], acc[SLOTS];
    double x[SLOTS], v[SLOTS], lu[SLOTS], d[SLOTS], g[SLOTS], lo[SLOTS], hi[SLOTS];
    int32_t jc[SLOTS];
#pragma unroll
    for (int i = 0; i < SLOTS; ++i) {
        U[i] = V[i] = A[i] = acc[i] = 0.0;
        x[i] = v[i] = lu[i] = d[i] = g[i] = lo[i] = hi[i] = 0.0;
        jc[i] = 0;
        if (live[i]) {
            U[i] = ab.au[off + pp[i]];
            V[i] = ab.av[off + pp[i]];
            A[i] = ab.aa[off + pp[i]];
        }
        if (own[i]) {
            jc[i] = ab.wj[off + pp[i]];
            lo[i] = Y[(int64_t)pp[i] * nch + jc[i]];
            hi[i] = Y[(int64_t)pp[i] * nch + jc[i] + 1];
        }
    }
    double gmu = 0.0, gk = 0.0, gkf = 0.0, geta = 0.0;

    auto flush = [&](int i) {
        if (ab.gy && own[i]) {
            double* row = ab.gy + (off + pp[i]) * nch;
            const double dy = 0.5 * mu * acc[i];
            row[jc[i]] += dy;
            row[jc[i] + 1] += dy;
        }
        acc[i] = 0.0;
    };
    // the well of slip y of an own particle at step n, from the current one
    auto walk = [&](int i, double y, int n) {
        if constexpr (WELLS) {
            const int32_t j = ab.tj[(int64_t)n * Rnp + (int64_t)r * ab.np + pp[i]];
            if (j != jc[i]) {
                flush(i);
                jc[i] = j;
                lo[i] = Y[(int64_t)pp[i] * nch + j];
                hi[i] = Y[(int64_t)pp[i] * nch + j + 1];
            }
        }
        else if (!(lo[i] <= y && y < hi[i])) {
            if (acc[i] != 0.0) {
                flush(i);
            }
            const double* row = Y + (int64_t)pp[i] * nch;
            int32_t j = jc[i];
            double a = lo[i], b = hi[i];
            while (y >= b && j < jmax) {
                ++j;
                a = b;
                b = row[j + 1];
            }
            while (y < a && j > jmin) {
                --j;
                b = a;
                a = row[j];
            }
            jc[i] = j;
            lo[i] = a;
            hi[i] = b;
        }
    };
    // the ends' neighbours: on the ring copies of the other end's values; at
    // the open ends of a tile's segment 0, any finite value would do (the
    // error zone that never reaches the tile's own particles)
    if (!ring && t < 8) {
        s_x[(t >> 1) * B + ((t & 1) ? E + 1 : 0)] = 0.0;
    }
    double* const sx = s_x + 1 + t;
    auto put = [&](int buf, int i, double y) {
        sx[buf * B + T * i] = y;
        if (ring && t + T * i == 0) {
            s_x[buf * B + E + 1] = y;
        }
        if (ring && t + T * i == E - 1) {
            s_x[buf * B] = y;
        }
    };
    auto neighbours = [&](int buf, int i) { return sx[buf * B + T * i - 1] + sx[buf * B + T * i + 1]; };

    // force of an own particle from its slip and the neighbours'
    auto force = [&](int buf, int i, double f, int n) {
        lu[i] = __builtin_fma(-2.0, x[i], neighbours(buf, i));
        walk(i, x[i], n);
        d[i] = __builtin_fma(0.5, lo[i] + hi[i], -x[i]);
        g[i] = __builtin_fma(k, lu[i], __builtin_fma(mu, d[i], kf * (f - x[i])));
    };

    // the tape of step n (n = -1: the checkpoint's acceleration in qu), loaded
    // two steps before its use
    struct Tape {
        double u[SLOTS], v[SLOTS], uf;
    };
    auto load = [&](Tape& q, int n) {
        const int64_t tn = (n >= 0 ? n * Rnp : 0) + (int64_t)r * ab.np;
        const double* const tu = (n >= 0 ? ab.tu : ab.wa) + tn;
        const double* const tv = ab.tv + tn;
#pragma unroll
        for (int i = 0; i < SLOTS; ++i) {
            if (slip[i]) {
                q.u[i] = tu[(uint32_t)pp[i]];
            }
            if (own[i] && n >= 0) {
                q.v[i] = tv[(uint32_t)pp[i]];
            }
        }
        if (n >= 0) {
            q.uf = ab.tuf[(int64_t)n * ab.R + r];
        }
    };
    double uf = 0.0;
    // reverse step n; q: the tape of step n - 1
    auto step = [&](int n, Tape& q, auto odd) {
        constexpr int gb = decltype(odd)::value, xb = 2 + (1 - decltype(odd)::value);
        double G[SLOTS], V3[SLOTS], px[SLOTS], pv[SLOTS];
        const double puf = q.uf;
#pragma unroll
        for (int i = 0; i < SLOTS; ++i) {
            px[i] = q.u[i];
            pv[i] = q.v[i];
            if (live[i]) {
                V3[i] = __builtin_fma(e1, A[i], V[i]);
                G[i] = w * __builtin_fma(h, __builtin_fma(eh, V3[i], V3[i]), A[i]);
                put(gb, i, G[i]);
            }
            if (n > 0 && slip[i]) {
                put(xb, i, px[i]);
            }
        }
        __syncthreads();
        if (n > 1) {
            load(q, n - 3);
        }
#pragma unroll
        for (int i = 0; i < SLOTS; ++i) {
            if (own[i]) {
                // the force of the step before gives the acceleration at the
                // start of this one, and from it the velocities of its stages
                const double gn = g[i];
                gkf = __builtin_fma(uf - x[i], G[i], gkf);
                gmu = __builtin_fma(d[i], G[i], gmu);
                gk = __builtin_fma(lu[i], G[i], gk);
                acc[i] += G[i];
                double a = px[i];
                if (n > 0) {
                    x[i] = px[i];
                    force(xb, i, puf, n - 1);
                    a = w * __builtin_fma(meta, v[i], g[i]);
                }
                const double v1 = __builtin_fma(dt, a, v[i]);
                const double a1 = w * __builtin_fma(meta, v1, gn);
                const double v2 = __builtin_fma(h, a + a1, v[i]);
                const double a2 = w * __builtin_fma(meta, v2, gn);
                const double v3 = __builtin_fma(h, a + a2, v[i]);
                geta = __builtin_fma(h * V3[i], __builtin_fma(eh, v1, v2), __builtin_fma(v3, A[i], geta));
                v[i] = pv[i];
            }
            if (live[i]) {
                // g depends on u1 through -(k_frame + mu) u1 + k L u1 (L
                // symmetric); u1 = u + dt v + c2 a
                const double s2 = __builtin_fma(eh, V3[i], V3[i]);
                U[i] = __builtin_fma(k, __builtin_fma(-2.0, G[i], neighbours(gb, i)),
                                     __builtin_fma(kfm, G[i], U[i]));
                V[i] = __builtin_fma(dt, U[i], __builtin_fma(ehh, V3[i], s2));
                A[i] = __builtin_fma(c2, U[i], __builtin_fma(dehh, V3[i], h * s2));
            }
        }
        uf = puf;
    };
    if (steps > 0) { // the last step's slips, wells and velocities
        Tape q0 = {}, q1 = {};
        load(q0, steps - 1);
        uf = q0.uf;
#pragma unroll
        for (int i = 0; i < SLOTS; ++i) {
            x[i] = q0.u[i];
            v[i] = q0.v[i];
            if (slip[i]) {
                put(2, i, x[i]);
            }
        }
        load(q0, steps - 2);
        if (steps > 1) {
            load(q1, steps - 3);
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < SLOTS; ++i) {
            if (own[i]) {
                force(2, i, uf, steps - 1);
            }
        }
        // (the first step's slips go to the other buffer)
        int n = steps - 1;
        for (; n > 0; n -= 2) {
            step(n, q0, std::integral_constant<int, 0>());
            step(n - 1, q1, std::integral_constant<int, 1>());
        }
        if (n == 0) {
            step(0, q0, std::integral_constant<int, 0>());
        }
    }
#pragma unroll
    for (int i = 0; i < SLOTS; ++i) {
        if (own[i]) {
            ab.bu[off + pp[i]] = U[i];
            ab.bv[off + pp[i]] = V[i];
            ab.ba[off + pp[i]] = A[i];
            flush(i);
        }
    }
    // parameter derivatives of the tile: block sums in a fixed order
    gmu = wave_sum(gmu);
    gk = wave_sum(gk);
    gkf = wave_sum(gkf);
    geta = wave_sum(-w * geta);
    if (lane == 0) {
        s_red[0][wave] = gmu;
        s_red[1][wave] = gk;
        s_red[2][wave] = gkf;
        s_red[3][wave] = geta;
    }
    __syncthreads();
    if (t < 4) {
        double s = 0.0;
        for (int q = 0; q < nw; ++q) {
            s += s_red[t][q];
        }
        ab.gpart[(int64_t)blockIdx.x * 4 + t] = s;
    }
}

// The state of all replicas at the start of a window.
__global__ void __launch_bounds__(256) k_adj_checkpoint(const double* __restrict__ u, const double* __restrict__ v,
                                                        const double* __restrict__ a, const int32_t* __restrict__ j,
                                                        double* __restrict__ cu, double* __restrict__ cv,
                                                        double* __restrict__ ca, int32_t* __restrict__ cj, int64_t n)
{
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        cu[i] = u[i];
        cv[i] = v[i];
        ca[i] = a[i];
        cj[i] = j[i];
    }
}

// The parameter derivatives of a window: the tiles' partial sums of each
// replica, in tile order, added to the totals (one thread per replica and
// parameter).
__global__ void __launch_bounds__(256) k_adj_params(AdjBuffers ab)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= ab.R * 4) {
        return;
    }
    const int64_t r = i / 4, c = i % 4;
    double s = 0.0;
    for (int tile = 0; tile < ab.nt; ++tile) {
        s += ab.gpart[(r * ab.nt + tile) * 4 + c];
    }
    ab.gpar[i] += s;
}

} // namespace fq
