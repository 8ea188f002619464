// Host-side launchers of the kernels. The resident kernels are instantiated in
// fq_res_<unit>.hip (generated by gen_instances.py); the service kernels in
// fq_service.hip.
#pragma once

#include "fq_common.hpp"
#include "fq_res_units.hpp"

namespace fq {

// per-unit launchers (generated, fq_res_<unit>.hip)
#define FQ_TRY_POT(P, CALL)                                                                                    \
    if (pot == P) {                                                                                            \
        FQ_UNITS_##P                                                                                           \
    }

// k_resident (all modes) for a potential / interaction / forcing / shape
inline bool launch_resident(int pot, int inter, int ext, int ppt, int maxt, int threads, size_t lds,
                            const SysView* views, int nsys, const RunArgs& ra, hipStream_t stream)
{
#define X(u)                                                                                                   \
    if (launch_resident_##u(inter, ext, ppt, maxt, threads, lds, views, nsys, ra, stream)) {                 \
        return true;                                                                                           \
    }
    FQ_TRY_POT(POT_CUSPY, )
    FQ_TRY_POT(POT_SEMISMOOTH, )
    FQ_TRY_POT(POT_SMOOTH, )
#undef X
    return false;
}

// k_flow (timeSteps / flowSteps of chains); false if not instantiated.
// unit_mass: every system has m = 1 (the multiplication by 1/m is left out);
// full: every system has N divisible by ppt
inline bool launch_flow(int pot, int inter, int ext, int ppt, int maxt, int threads, size_t lds,
                        const SysView* views, int nsys, const RunArgs& ra, hipStream_t stream, bool unit_mass,
                        bool full, bool moves)
{
#define X(u)                                                                                                   \
    if (launch_flow_##u(inter, ext, ppt, maxt, threads, lds, views, nsys, ra, stream, unit_mass, full, moves)) { \
        return true;                                                                                           \
    }
    FQ_TRY_POT(POT_CUSPY, )
    FQ_TRY_POT(POT_SEMISMOOTH, )
    FQ_TRY_POT(POT_SMOOTH, )
#undef X
    return false;
}

// The quasistatic driver (no external forcing): k_quasi_chain for the variants
// of chains and lattices whose registers hold it (gen_instances.py:
// pipelined), k_quasi otherwise; false if not instantiated for this potential /
// interaction / shape (unit_mass: every system has m = 1; full: every system
// has N divisible by ppt)
inline bool launch_quasi(int pot, int inter, int ppt, int maxt, int threads, size_t lds, const SysView* views,
                         int nsys, const RunArgs& ra, const QsArgs& qa, hipStream_t stream, bool unit_mass, bool full)
{
#define X(u)                                                                                                   \
    if (launch_quasi_##u(inter, ppt, maxt, threads, lds, views, nsys, ra, qa, stream, unit_mass, full)) {    \
        return true;                                                                                           \
    }
    FQ_TRY_POT(POT_CUSPY, )
    FQ_TRY_POT(POT_SEMISMOOTH, )
    FQ_TRY_POT(POT_SMOOTH, )
#undef X
    return false;
}

// the (particles per thread, max threads) variants compiled for a class
inline int resident_variants(int pot, int inter, int ext, int* ppt, int* maxt, int cap)
{
#define X(u)                                                                                                   \
    {                                                                                                          \
        const int n = resident_variants_##u(inter, ext, ppt, maxt, cap);                                      \
        if (n > 0) {                                                                                           \
            return n;                                                                                          \
        }                                                                                                      \
    }
    FQ_TRY_POT(POT_CUSPY, )
    FQ_TRY_POT(POT_SEMISMOOTH, )
    FQ_TRY_POT(POT_SMOOTH, )
#undef X
    return 0;
}
#undef FQ_TRY_POT

// LDS bytes of a resident launch (must agree with k_resident's layout).
inline size_t resident_lds(int inter, int64_t N, int threads)
{
    if (inter == INT_NONE || inter == INT_LAPLACE1D || inter == INT_QUARTIC1D || inter == INT_QUARTICGRADIENT1D) {
        return sizeof(double) * 4 * (size_t)threads;
    }
    if (inter == INT_LONGRANGE1D) {
        return sizeof(double) * (N <= LR_LDS_PREF_MAX ? 4 : 2) * (size_t)N;
    }
    return sizeof(double) * 2 * (size_t)N;
}

// LDS bytes of a launch of the quasistatic driver (must agree with the
// layouts of k_quasi_chain and k_quasi)
inline size_t quasi_lds(int inter, int64_t N, int ppt, int maxt, int threads)
{
    return resident_lds(inter, N, threads) +
           (inter != INT_LONGRANGE1D && quasi_inplace(ppt, maxt) ? sizeof(double) * (size_t)ppt * threads : 0);
}

// batched long range (fq_longrange.hip)
int lr_split_blocks(); // summation ranges are multiples of this many indices
hipError_t launch_lr_gemm(const double* pref, const LrBuffers& lb, int64_t lr_m, hipStream_t stream);
int lr_fft_log2(int64_t N); // log2 of the transform's complex points (0: use launch_lr_gemm)
hipError_t launch_lr_fft(int log2_points, const double* tw, const double* sd, const LrBuffers& lb, hipStream_t stream);
hipError_t launch_lr_elem(int ext, const SysView* views, const LrBuffers& lb, const RunArgs& ra, hipStream_t stream);
hipError_t launch_lr_prologue(const SysView* views, const LrBuffers& lb, hipStream_t stream);

// adjoint (fq_adjoint.hip)
int adj_variants(int* ppt, int* maxt, int cap);
bool launch_adj_record(int ppt, int threads, const SysView* views, const AdjBuffers& ab, int windows, int flow,
                       double v_frame, hipStream_t stream);
// extended-segment particles per thread of the reverse kernel for a segment
// of `extended` particles (0: too long)
hipError_t launch_adj_checkpoint(const double* u, const double* v, const double* a, const int32_t* j, double* cu,
                                 double* cv, double* ca, int32_t* cj, int64_t n, hipStream_t stream);
int adj_reverse_slots(int64_t extended);
bool launch_adj_reverse(const SysView* views, const AdjBuffers& ab, int slots, int steps, hipStream_t stream);

// tiled per-step path (fq_tile.hip): large systems over many workgroups
bool tile_supported(int pot, int inter, int ext);
hipError_t launch_tile_prologue(const SysView* views, const TileDesc* tiles, int ntiles, hipStream_t stream);
bool launch_tile_step(int pot, int inter, const SysView* views, const TileDesc* tiles, int ntiles, size_t lds,
                      double* part, int32_t* tflag, const RunArgs& ra, hipStream_t stream);
hipError_t launch_tile_decide(const SysView* views, int nsys, const int32_t* tile_first, const double* part,
                              int32_t* tflag, const RunArgs& ra, hipStream_t stream);
// blocks of K steps per launch (chains: k_tile_block; lattices:
// k_tile_block2d with `lds` bytes of dynamic LDS, 2 x 8 x the extended sites
// of the largest tile; lone: no more tiles than compute units; false for other
// interactions)
bool tile_block_supported(int pot, int inter);
bool launch_tile_block(int pot, int inter, const SysView* views, const TileDesc* tiles, int ntiles, double* part,
                       int32_t* tfail, const RunArgs& ra, int K, size_t lds, bool unit_mass, bool lone,
                       hipStream_t stream);
hipError_t launch_tile_block_decide(const SysView* views, int nsys, const int32_t* tile_first, const double* part,
                                    const int32_t* tfail, const RunArgs& ra, int K, hipStream_t stream);
bool launch_tile_finish(int pot, int inter, const SysView* views, const TileDesc* tiles, int ntiles,
                        hipStream_t stream);

// streaming kernel (fq_stream.hip): systems of any size, one workgroup each
bool launch_stream(int pot, int inter, int ext, const SysView* views, int nsys, const RunArgs& ra,
                   hipStream_t stream);

// service kernels (fq_service.hip); views are device pointers, nsys systems
hipError_t launch_landscape_init(const SysView* views, int nsys, int64_t maxN, hipStream_t stream);
hipError_t launch_restore(const SysView* views, int64_t N, const uint64_t* state, const double* value,
                          const int64_t* index, hipStream_t stream);
// (maxN: particles of the largest system)
bool launch_forces(int pot, int inter, int ext, const SysView* views, int nsys, int64_t maxN, int32_t flags,
                   hipStream_t stream);
bool launch_max_uniform(int pot, const SysView* views, int nsys, int64_t maxN, int32_t direction, hipStream_t stream);
hipError_t launch_trigger(const SysView* views, int64_t p, double eps, int32_t direction, int32_t do_align,
                          hipStream_t stream);
hipError_t launch_set_iref(const SysView* views, int nsys, int64_t maxN, hipStream_t stream);
hipError_t launch_refill(const SysView* views, int nsys, int64_t maxN, hipStream_t stream);
hipError_t launch_trigger_each(const SysView* views, int nsys, const int64_t* ps, double eps, int32_t direction,
                               int32_t do_align, hipStream_t stream);
hipError_t launch_qs_record(const SysView* views, int nsys, int64_t maxN, const QsArgs& qa, int64_t e, int begin,
                            hipStream_t stream);
// no-passing sweeps over tiles (fq_tile.hip): chains of any length; one call
// enqueues one sweep (sweep, residual sums, StopList and buffer flip)
hipError_t launch_np_sweep(const SysView* views, const TileDesc* tiles, int ntiles, int nsys,
                           const int32_t* tile_first, double* part, const RunArgs& ra, hipStream_t stream);
hipError_t launch_np_finish(const SysView* views, const TileDesc* tiles, int ntiles, hipStream_t stream);
bool launch_nopassing(int ppt, int threads, size_t lds, const SysView* views, int nsys, const RunArgs& ra,
                      hipStream_t stream);

} // namespace fq
