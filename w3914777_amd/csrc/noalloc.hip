// noalloc.hip — the FP64 snowflake step on caller-owned device buffers with
// no device memory of the library's own: amps_sf_step_fp64_noalloc.
//
// The instance descriptor and the step index travel as kernel arguments, so a
// call is one launch: nothing to write to the device first (256^2: 4.7 us of
// GPU time, 7.1 with a setup kernel before the sweep), nothing shared between
// calls, and the call can be captured into a HIP graph.
#include "kernels.hpp"

using namespace amps;

extern "C" int amps_sf_step_fp64_noalloc(const amps_config* cfg, const double* d_in, double* d_out, int64_t step,
                                         void* stream) {
    if (!cfg || !d_in || !d_out) return fail_with(AMPS_E_ARG, "NULL argument");
    if (cfg->model != AMPS_SNOWFLAKE) return fail_with(AMPS_E_UNSUPPORTED, "the no-allocation step covers the snowflake model");
    if (cfg->mode != AMPS_PURE_FP64) return fail_with(AMPS_E_UNSUPPORTED, "the no-allocation step is the PURE_FP64 step");
    const int rc = validate_config(*cfg);
    if (rc != AMPS_OK) return rc;
    if (step < 0) return fail_with(AMPS_E_ARG, "step must be >= 0");
    const size_t n = 2 * (size_t)cfg->nx * cfg->ny;
    const char* a0 = reinterpret_cast<const char*>(d_in);
    const char* b0 = reinterpret_cast<const char*>(d_out);
    if (a0 < b0 + n * sizeof(double) && b0 < a0 + n * sizeof(double))
        return fail_with(AMPS_E_ARG, "d_in and d_out overlap");
    InstDesc d;
    config_desc(d, *cfg);
    StepArgs a{};
    a.total_cells = (long long)cfg->nx * cfg->ny;
    a.total_tiles = d.tx * d.ty;
    a.nwork = a.total_tiles;
    a.nfields = 2;
    a.ninst = 1;
    a.in.f64 = const_cast<double*>(d_in);
    a.out.f64 = d_out;
    const int lr = launch_sf_step_arg(a, d, (long long)step, cfg->tile, static_cast<hipStream_t>(stream));
    return lr == AMPS_OK ? AMPS_OK : fail_with(lr, "FP64 sweep launch failed");
}
