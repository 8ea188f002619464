// Resident kernel for timeSteps / flowSteps of chains (MODE_STEPS only):
//   timeStep            detail.h:1539-1570
//   timeSteps/flowSteps detail.h:1577-1583, 1637-1645
//   RandomNormalForcing::force detail.h:930-943         (EXT = 1)
// Same ownership, expressions and results as k_resident (fq_resident.hpp),
// bit for bit, with less work per particle-step:
//  * software-pipelined: the slips of step it+1, u + dt v + dt^2/2 a, are
//    computed once at the end of step it (into separate registers, so a stop
//    before step it+1 discards them), checked for reachability and published
//    to the LDS exchange buffer (it+1)&1 for the neighbours; step it+1 then
//    commits them. One __syncthreads per step, at the top of the step.
//  * the constants of the current well (well_consts: Cuspy its mid-point) are
//    kept in registers, recomputed when the well changes;
//  * with m = 1 the multiplication by 1/m (exact) is skipped;
//  * no event / residual bookkeeping;
//  * FULL (every system of the launch has N divisible by PPT, so a thread
//    holds PPT particles or none): the thread's last particle is register
//    PPT - 1 at compile time, which removes a select per register and step
//    from the interaction and makes the publication of the last slip one
//    store.
#pragma once

#include "fq_resident.hpp"

#include <type_traits>

namespace fq {

// One entry of k_flow: from the state in memory to the state in memory, until
// the launch's step budget (of which earlier entries took `launch_done`) or a
// NaN; but for REFILL_INLINE also up to a step that has to move a window
// (ST_REFILL; REFILL_ENTRY: `refill_mask`, this thread's particles). Returns
// why it stopped. WC: the well's constants are kept.
enum FlowRefill { REFILL_HOST, REFILL_ENTRY, REFILL_INLINE };

template <int POT, int INT, int EXT, int PPT, bool UNIT, bool FULL, FlowRefill REFILL, bool WC>
__device__ __forceinline__ int32_t flow_entry(const SysView* __restrict__ views, const RunArgs& ra,
                                              int64_t& launch_done, uint32_t& refill_mask)
{
    const SysView& S = views[blockIdx.x];
    // the system's parameters as a local copy: registers for the whole launch
    // instead of a reload of the ones the forces use after every barrier
    const SysView P = S;
    RunState* const rs = S.rs;
    const int64_t room = rs->target - rs->steps, budget = ra.max_steps - launch_done;
    const int limit = uniform_i((int)(room < budget ? (room > 0 ? room : 0) : budget));

    __shared__ int s_nan[2];
    // (unused with REFILL_INLINE, but the exchange buffers begin 16 bytes into
    // LDS with it: 8 bytes in, 1000 steps of 1024 chains of 4096 take 5.37 ms
    // instead of 5.32)
    __shared__ int s_refill[2];
    __shared__ int s_scan_w[RES_MAX_WAVES];
    __shared__ long long s_min_w[RES_MAX_WAVES];
    extern __shared__ double s_dyn[];

    const int t = threadIdx.x, T = blockDim.x;
    const int64_t N = S.N;
    const int64_t base = (int64_t)t * PPT;
    const int cnt = (int)(N - base >= PPT ? PPT : (N - base > 0 ? N - base : 0));
    const int Tact = (int)((N + PPT - 1) / PPT);
    // register of the thread's last particle (FULL: cnt is PPT or 0, and a
    // thread without particles neither publishes nor stores)
    const int last = FULL ? PPT - 1 : cnt - 1;
    const Landscape& L = S.ls;
    double* const Y = L.y;
    const int64_t nch = L.nchunk;
    const int32_t jmin = (int32_t)L.buffer;
    const int32_t jmax = (int32_t)(L.nchunk - 2 - L.buffer);
    double* h_first = s_dyn;        // [2][T] first slip of each thread
    double* h_last = s_dyn + 2 * T; // [2][T] last slip of each thread

    // Slips live in two register arrays used in turn: one holds the state of
    // the current step, the other the slips prepared for the next step (and,
    // before they are committed, the state of the previous one). The step
    // loop is unrolled by two so that the arrays swap roles without copies.
    // Registers i >= cnt are padding: zero state (reset after every step) in
    // an unbounded well, so they never walk, never request a refill, never
    // set the NaN flag and never publish; the hot loops run over all PPT
    // registers without per-particle branches and only the stores are
    // guarded. The reset runs only in wavefronts that hold padding (a scalar
    // branch: a full wavefront skips it).
    double sa[PPT], sb[PPT], v[PPT], a[PPT], yl[PPT], yr[PPT], fth[PPT];
    // constants of the current well (well_consts)
    constexpr bool WC1 = POT != POT_CUSPY && WC;
    double c0[WC ? PPT : 1], c1[WC1 ? PPT : 1];
    auto set_well = [&](int i, double lo, double hi) {
        yl[i] = lo;
        yr[i] = hi;
        if constexpr (WC) {
            double k1;
            well_consts<POT>(P, lo, hi, c0[i], k1);
            if constexpr (WC1) {
                c1[i] = k1;
            }
        }
    };
    auto well_force = [&](int i, double x) -> double {
        if constexpr (!WC) {
            return potential_force<POT>(P, x, yl[i], yr[i]);
        }
        return potential_force_wc<POT>(P, x, yl[i], yr[i], c0[WC ? i : 0], c1[WC1 ? i : 0]);
    };
    int32_t jl[PPT];
#pragma unroll
    for (int i = 0; i < PPT; ++i) {
        sa[i] = sb[i] = v[i] = a[i] = c0[WC ? i : 0] = fth[i] = 0.0;
        if constexpr (WC1) {
            c1[i] = 0.0;
        }
        yl[i] = -__builtin_inf();
        yr[i] = __builtin_inf();
        jl[i] = 0;
        if (i < cnt) {
            const int64_t p = base + i;
            sa[i] = S.u[p];
            v[i] = S.v[p];
            a[i] = S.a[p];
            jl[i] = L.jloc[p];
            set_well(i, Y[p * nch + jl[i]], Y[p * nch + jl[i] + 1]);
            if constexpr (EXT) {
                fth[i] = S.f_th[p];
            }
        }
    }

    const double dt = S.dt;
    const double c2 = 0.5 * dt * dt;
    const double hdt = 0.5 * dt;
    const double meta = -S.eta;
    const double inv_m = S.inv_m;
    const double kf = S.k_frame;
    const double dv = ra.v_frame * dt;

    if (t == 0) {
        s_nan[0] = 0;
        s_nan[1] = 0;
        s_refill[0] = 0;
        s_refill[1] = 0;
    }
    int64_t inc = uniform_ll(rs->inc); // scalar: its increment is a scalar add
    double uf = rs->u_frame;
    const bool pad_wave = uniform_i(__any(cnt < PPT)) != 0;
    uint64_t rng = rs->rng_state;
    const uint64_t rng_inc = rs->rng_inc;
    int64_t min_next = rs->min_next;
    if constexpr (EXT) {
        long long mn = 0x7fffffffffffffffLL;
#pragma unroll
        for (int i = 0; i < PPT; ++i) {
            if (i < cnt) {
                long long nx = S.next[base + i];
                mn = nx < mn ? nx : mn;
            }
        }
        min_next = uniform_ll(block_min_i(mn, s_min_w));
    }
    __syncthreads(); // flags cleared before any thread sets them

    // publish the first and last value of x (registers) into exchange buffer
    // b; the last one is stored under a predicate per register (an indexed
    // read x[cnt - 1] would move the array to scratch memory)
    auto publish = [&](const double(&x)[PPT], int b) {
        if (cnt > 0) {
            h_first[b * T + t] = x[0];
#pragma unroll
            for (int i = 0; i < PPT; ++i) {
                if (i == last) {
                    h_last[b * T + t] = x[i];
                }
            }
        }
    };

    // slips of step `it` from the state x into y, and publication into
    // exchange buffer it&1; pend: some slip of this thread leaves its well (or
    // is NaN), so that the commit of the step walks only then. But for
    // REFILL_INLINE their reachability as well (rmask, s_refill).
    int pend = 0;
    uint32_t rmask = 0;
    auto prepare = [&](int it, const double(&x)[PPT], double(&y)[PPT]) {
        const int b = it & 1;
        int out = 0;
#pragma unroll
        for (int i = 0; i < PPT; ++i) {
            y[i] = x[i] + dt * v[i] + c2 * a[i];
            out |= !(yl[i] <= y[i] && y[i] < yr[i]);
        }
        pend = out;
        if constexpr (REFILL != REFILL_INLINE) {
            uint32_t mask = 0;
            if (out) { // rare: some slip leaves its well
                // opaque copies: the addresses and comparisons of this rare
                // path stay in it instead of being evaluated for every step
                int64_t bq = base;
                __asm__ volatile("" : "+v"(bq));
#pragma unroll
                for (int i = 0; i < PPT; ++i) {
                    double z = y[i];
                    __asm__ volatile("" : "+v"(z));
                    if (!(yl[i] <= z && z < yr[i]) && __builtin_isfinite(z) &&
                        !reachable(Y + (bq + i) * nch, jl[i], yl[i], yr[i], z, jmin, jmax)) {
                        mask |= 1u << i;
                    }
                }
                if (mask) {
                    s_refill[b] = it;
                }
            }
            if constexpr (REFILL == REFILL_ENTRY) {
                rmask = mask;
            }
        }
        publish(y, b);
    };

    auto left_of = [&](int b) -> double { return h_last[b * T + (t == 0 ? Tact - 1 : t - 1)]; };
    auto right_of = [&](int b) -> double { return h_first[b * T + (t == Tact - 1 ? 0 : t + 1)]; };
    auto interaction = [&](int i, int b, const double(&x)[PPT]) -> double {
        if constexpr (INT == INT_NONE) {
            return 0.0;
        }
        else {
            double um = 0.0, up = 0.0;
#pragma unroll
            for (int q = 0; q < PPT; ++q) {
                if (q == i) {
                    um = (q == 0) ? left_of(b) : x[q > 0 ? q - 1 : 0];
                    up = (q == last) ? right_of(b) : x[q + 1 < PPT ? q + 1 : q];
                }
            }
            return chain_force<INT>(P, um, x[i], up);
        }
    };

    int32_t status = ST_RUNNING;
    int refilled = 0;

    // step `it` with the prepared slips in x (the previous state in y, which
    // receives the slips of step it+1); false if the run stops before it
    auto step = [&](int it, double(&x)[PPT], double(&y)[PPT]) -> bool {
        const int b = it & 1;
        __syncthreads(); // slips of step `it` published, flags of step it-1 set

        if (it > 1 && uniform_i(s_nan[(it - 1) & 1]) == it - 1) {
            status = ST_NAN;
            return false;
        }
        if (it > limit) {
            return false;
        }
        if constexpr (REFILL != REFILL_INLINE) {
            if (uniform_i(s_refill[b]) == it) {
                status = ST_REFILL;
                return false;
            }
        }

        inc += 1;
        if (ra.flow) {
            uf = uf + dv;
        }
        if constexpr (EXT) {
            if (inc >= min_next) {
                int due = 0;
#pragma unroll
                for (int i = 0; i < PPT; ++i) {
                    if (i < cnt && inc >= S.next[base + i]) {
                        ++due;
                    }
                }
                int total = 0;
                int rank = block_excl_scan(due, s_scan_w, total);
                if (due > 0) {
                    uint64_t st = pcg_advance(rng, rng_inc, 2 * (int64_t)rank);
#pragma unroll
                    for (int i = 0; i < PPT; ++i) {
                        if (i < cnt) {
                            const int64_t p = base + i;
                            int64_t nx = S.next[p];
                            if (inc >= nx) {
                                fth[i] = draw_normal(st, rng_inc, S.mean, S.stddev);
                                S.next[p] = nx + S.dinc[p];
                            }
                        }
                    }
                }
                long long mn = 0x7fffffffffffffffLL;
#pragma unroll
                for (int i = 0; i < PPT; ++i) {
                    if (i < cnt) {
                        long long nx = S.next[base + i];
                        mn = nx < mn ? nx : mn;
                    }
                }
                rng = pcg_advance(rng, rng_inc, 2 * (int64_t)uniform_i(total));
                min_next = uniform_ll(block_min_i(mn, s_min_w));
            }
        }

        // commit: the slips in x are the state now; walk to their wells
        uint32_t need = 0;
        if (pend) { // rare
            int nanf = 0;
            // opaque copy of the first index: the window addresses of this
            // rare path are computed in it, not kept live through the loop
            int64_t bq = base;
            __asm__ volatile("" : "+v"(bq));
#pragma unroll
            for (int i = 0; i < PPT; ++i) {
                const double z = x[i];
                nanf |= __builtin_isnan(z);
                if (!(yl[i] <= z && z < yr[i])) {
                    const double* row = Y + (bq + i) * nch;
                    int32_t j = jl[i];
                    double lo = yl[i], hi = yr[i];
                    while (z >= hi && j < jmax) {
                        ++j;
                        lo = hi;
                        hi = row[j + 1];
                    }
                    while (z < lo && j > jmin) {
                        --j;
                        hi = lo;
                        lo = row[j];
                    }
                    if (lo <= z && z < hi) {
                        jl[i] = j;
                        set_well(i, lo, hi);
                    }
                    else if (REFILL == REFILL_INLINE && __builtin_isfinite(z)) {
                        need |= 1u << i;
                    }
                }
            }
            if (nanf) {
                s_nan[b] = it;
            }
        }
        // windows that have to move (rare): one particle at a time by the
        // whole wavefront, the other wavefronts do not wait for it
        if (REFILL == REFILL_INLINE && __builtin_expect(__any(need != 0), 0)) {
#pragma unroll
            for (int i = 0; i < PPT; ++i) {
                uint64_t lanes = __ballot((need >> i) & 1u);
                while (lanes) {
                    const int src = __builtin_ctzll(lanes);
                    lanes &= lanes - 1;
                    const double z = lane_d(x[i], src);
                    const int64_t p = ((int64_t)(t & ~63) + src) * PPT + i;
                    const WellAt w = refill_one(&S, p, z, __builtin_amdgcn_readlane(jl[i], src));
                    if ((t & 63) == src) {
                        jl[i] = w.j;
                        set_well(i, w.lo, w.hi);
                    }
                }
            }
            refilled = 1;
        }

        // the reference's three velocity / acceleration passes (detail.h:1552-1565)
#pragma unroll
        for (int i = 0; i < PPT; ++i) {
            const double fi = interaction(i, b, x);
            const double fp = well_force(i, x[i]);
            const double ff = kf * (uf - x[i]);
            const double sum3 = ff + fp + fi;
            const double vn = v[i], an = a[i];
            double vv = vn + dt * an;
            double f = EXT ? sum3 + meta * vv + fth[i] : sum3 + meta * vv;
            double aa = UNIT ? f : f * inv_m;
            vv = vn + hdt * (an + aa);
            f = EXT ? sum3 + meta * vv + fth[i] : sum3 + meta * vv;
            aa = UNIT ? f : f * inv_m;
            vv = vn + hdt * (an + aa);
            f = EXT ? sum3 + meta * vv + fth[i] : sum3 + meta * vv;
            aa = UNIT ? f : f * inv_m;
            v[i] = vv;
            a[i] = aa;
        }
        if (pad_wave) { // padding registers stay at rest (FULL: all of them)
            // (the empty asm keeps this branch apart from the per-lane one
            // below, so that it stays a scalar branch)
            __asm__ volatile("");
            if (cnt < PPT) {
#pragma unroll
                for (int i = 0; i < PPT; ++i) {
                    if (FULL || i >= cnt) {
                        v[i] = 0.0;
                        a[i] = 0.0;
                    }
                }
            }
        }
        prepare(it + 1, x, y);
        return true;
    };

    // state and forces of the final configuration (slips in x, `done` steps
    // taken); its slips are in exchange buffer done&1 (published before step
    // `done`, or initially)
    auto finish = [&](const double(&x)[PPT], int done) -> int32_t {
        if (status == ST_RUNNING) {
            status = ST_BUDGET;
        }
        const int fb = done & 1;
#pragma unroll
        for (int i = 0; i < PPT; ++i) {
            if (i < cnt) {
                const int64_t p = base + i;
                S.u[p] = x[i];
                S.v[p] = v[i];
                S.a[p] = a[i];
                L.jloc[p] = jl[i];
                if (status != ST_NAN && status != ST_REFILL) {
                    const double fi = interaction(i, fb, x);
                    const double fp = well_force(i, x[i]);
                    const double ff = kf * (uf - x[i]);
                    const double fd = meta * v[i];
                    S.f_int[p] = fi;
                    S.f_pot[p] = fp;
                    S.f_frame[p] = ff;
                    S.f_damp[p] = fd;
                    S.f[p] = EXT ? ff + fp + fi + fd + fth[i] : ff + fp + fi + fd;
                }
                if constexpr (EXT) {
                    S.f_th[p] = fth[i];
                }
            }
        }
        if (refilled) {
            rs->refilled = 1;
        }
        if (t == 0) {
            rs->inc = inc;
            rs->u_frame = uf;
            rs->steps += done;
            rs->status = status;
            rs->rng_state = rng;
            rs->min_next = min_next;
        }
        launch_done += done;
        refill_mask = rmask;
        return status;
    };

    // the current slips into buffer 0 (forces of the final state when no step
    // is taken), the slips of step 1 into buffer 1
    publish(sa, 0);
    prepare(1, sa, sb);
    for (int it = 1;; it += 2) {
        if (!step(it, sb, sa)) {
            return finish(sa, it - 1);
        }
        if (!step(it + 1, sa, sb)) {
            return finish(sb, it);
        }
    }
}

// Windows that have to move are handled inside the launch (MOVES): variants of up to
// 512 threads (256 registers) call the refill from the commit of the step, by
// the wavefronts that need it; in variants of 1024 threads (128 registers)
// that call would spill the step loop's registers (4 x 1024 on 1024 chains of
// 4096: 34 ms instead of 5.1 ms per 1000 steps), so with up to 2 particles per
// thread the entry ends, refills from memory and starts again. With 4 the
// loop around the entry alone costs 14% (5.8 ms), so there the launch ends and
// the host relaunches it after k_refill. Sliding chains (256 x 1999, windows
// of 100, 4 x 512; a window moves somewhere in nearly every step): 13 ms per
// 1000 steps, against 273 ms with a relaunch each time.
// One particle per thread: the step alone takes 64 registers, with the refill's
// call 124, half as many wavefronts per SIMD. Batches whose workgroups do not
// all fit that way start with the form that leaves refills to the host (MOVES
// false) and go on with the other one once a window has to move (800 chains of
// 300, 300 steps, us, with / without the call: SemiSmooth-Laplace 576 / 346,
// Cuspy-Quartic 500 / 297).
template <int POT, int INT, int EXT, int PPT, int MAXT, bool UNIT, bool FULL = false, bool MOVES = true>
__global__ void __launch_bounds__(MAXT) k_flow(const SysView* __restrict__ views, RunArgs ra)
{
    static_assert(is_chain<INT>(), "k_flow handles chains");
    const RunState* const rs = views[blockIdx.x].rs;
    if (rs->status != ST_RUNNING && rs->status != ST_BUDGET) {
        return;
    }
    int64_t launch_done = 0;
    uint32_t rmask = 0;
    if constexpr (MAXT <= 512) {
        flow_entry<POT, INT, EXT, PPT, UNIT, FULL, REFILL_INLINE, true>(views, ra, launch_done, rmask);
    }
    else if constexpr (PPT > 2 || !MOVES) {
        // (more than two per thread: the well's constants would spill;
        // SemiSmooth, 100 chains of 4096, 300 steps 1.04 ms, with them 1.36;
        // a forced Cuspy chain of 4096, 400 steps 1.88 ms, with them 2.40)
        flow_entry<POT, INT, EXT, PPT, UNIT, FULL, REFILL_HOST, PPT <= 2 || (POT == POT_CUSPY && EXT == 0)>(
            views, ra, launch_done, rmask);
    }
    else {
        bool refilled = false;
        while (flow_entry<POT, INT, EXT, PPT, UNIT, FULL, REFILL_ENTRY, true>(views, ra, launch_done, rmask) ==
               ST_REFILL) {
            __syncthreads(); // the state of every lane's particles is in memory
            refilled = true;
            refill_wave(views, (int64_t)threadIdx.x * PPT, 0, rmask);
            __syncthreads();
        }
        if (refilled && threadIdx.x == 0) {
            views[blockIdx.x].rs->refilled = 1;
        }
    }
}

} // namespace fq
