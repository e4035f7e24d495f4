// kernels.hpp — host-side launch entry points of the gfx950 kernels.
#pragma once

#include "amps_internal.hpp"

namespace amps {

// Which type group each field belongs to (-1: always FP64).
struct GroupMap {
    int nfields;
    int ngroups;
    signed char fg[AMPS_MAX_FIELDS];
};

enum { CONVERT_CHANGED = 0, CONVERT_ENCODE_LOW = 1 };

// Config validation, the descriptor of one instance (tile base and cell
// base 0) and error recording, shared with host code outside api.cpp.
int validate_config(const amps_config& c);
void config_desc(InstDesc& d, const amps_config& c);
int fail_with(int code, const char* msg);

int launch_init(const InstDesc* inst_dev, int inst, long long ncells, int model, int init, int q, const Buf& b,
                long long total_cells, hipStream_t s);
int launch_convert(const InstDesc* inst, const int* tile_inst, const Buf& b, long long total_cells, int total_tiles,
                   const int* type_old, const int* type, const GroupMap& gm, int mode, int tile, hipStream_t s);
// reset: the counters of the classification that follows (CLASSIFY_SLOTS, at
// a stride of STATS_STRIDE), set to 0 by the monitor kernel.
int launch_monitor(const StepArgs& a, int kind, int tile, int ngroups_eval, int field0, int field_stride,
                   int type_groups, double* md, double* last, unsigned long long* reset, hipStream_t s);
int launch_monitor_last_init(const StepArgs& a, int tile, int ngroups_eval, int field0, int field_stride,
                             double* last, hipStream_t s);
// Classification and conversion of a monitor pass.  single: one instance
// (descriptor 0 for every tile).  same_flags (may be null): one per (group,
// tile), cleared where the type changes.  stats: the FP64 counts of all passes
// and of the last one, CLASSIFY_SLOTS each at a stride of STATS_STRIDE.
int launch_classify_convert(const InstDesc* inst, const int* tile_inst, const Buf& b, long long total_cells,
                            int total_tiles, int broadcast, int single, const double* md, double thr, int dilate,
                            int* type_old, int* type, const GroupMap& gm, int* same_flags, unsigned long long* stats,
                            int tile, hipStream_t s);
int launch_gather(const InstDesc* inst, const Buf& b, long long total_cells, int total_tiles, const int* type,
                  int group, int instid, int ntiles_inst, int field, double* dst, int* bad, int tile, hipStream_t s);
int launch_nonfinite(const double* v, long long n, int* bad, hipStream_t s);
// out (host memory): the classification's and the sweeps' counters, kind by
// kind (see StepArgs::spread; cls: all of them), each summed over its slots
// and, from kind 2 on, added to stats[kind].
int launch_counters(const unsigned long long* cls, const unsigned long long* stats, unsigned long long* out,
                    hipStream_t s);
int launch_fill_u64(unsigned long long* p, int n, unsigned long long v, hipStream_t s);
int launch_advance_step(long long* step_ctr, int n, hipStream_t s);

// ev (may be null): timing events bound to the step's sweep kernels: the
// start and end of the first (snowflake adaptive: the bulk-hold sweep) and,
// for the snowflake's adaptive step only, of the second (the mixed sweep).
int launch_sf_step(const StepArgs& a, int tile, bool adaptive, hipStream_t s, const hipEvent_t* ev = nullptr);
// The snowflake's low-precision step in one launch (grids with few tiles; not
// HALF2); counts its tiles in a.spread.
int launch_sf_one(const StepArgs& a, int tile, hipStream_t s);
// PURE_FP64 step `step` of one grid from a.in to a.out, its descriptor passed
// by value (a.inst and a.step_ctr unused).
int launch_sf_step_arg(const StepArgs& a, const InstDesc& d, long long step, int tile, hipStream_t s);
// PURE_FP64: bm.k steps in one launch on the blocks of bm (a.in to a.out).
int launch_sf_multi(const StepArgs& a, const BlockMap& bm, hipStream_t s);
int launch_gg_multi(const StepArgs& a, const BlockMap& bm, hipStream_t s);
int launch_sn_multi(const StepArgs& a, const BlockMap& bm, hipStream_t s);
int launch_worklist(const int* type, const int* type_old, int total_tiles, int* wl_hi, int* wl_lo, int* counts,
                    int* same_flags, hipStream_t s);
int launch_gg_step(const StepArgs& a, int tile, bool adaptive, int grid, hipStream_t s, const hipEvent_t* ev = nullptr);
// type_old (may be null): refresh only tiles where some field's type differs from a.type.
int launch_gg_aux(const StepArgs& a, int tile, const int* type_old, hipStream_t s);
int launch_sn_step(const StepArgs& a, int tile, bool adaptive, int grid, hipStream_t s, const hipEvent_t* ev = nullptr);

// Reverse-time adjoint of one FP64 step (snowflake, sintering).  Arrays are
// [field][total_cells] like the FP64 state.
struct AdjArgs {
    const InstDesc* inst;
    const int* tile_inst;
    int total_tiles;
    long long total_cells;
    const double* u;       // state before the step
    const double* un;      // state after the step
    const double* lam_n;   // dJ/d(state after)
    double* lam;           // dJ/d(state before), written
    double* gacc;          // [gradient slot][total_tiles] accumulators
    const long long* step_ctr;  // step index of the forward step = *step_ctr + step_add
    int step_add;
    int t_halo;            // snowflake: reach of the widest Laplacian among the instances
};
int launch_adjoint_step(const AdjArgs& a, int model, int tile, hipStream_t s);

}  // namespace amps
