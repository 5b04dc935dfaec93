// The short-K kernel (gemm_short_k.h): 16-bit and int8 inputs, the four operand layouts.
#include "gemm_short_k.h"
#include "variants.h"

namespace acc950 {

template <int IN>
static hipError_t launch_in(const GemmArgs& a, hipStream_t stream, LaunchGeom* geom, bool dry_run)
{
    // (K contiguous where the element stride along K is one; a single row or column of an operand is taken either way)
    if (a.a_cs == 1) return a.b_rs == 1 ? launch_short_k_layout<IN, true, true>(a, stream, geom, dry_run) : launch_short_k_layout<IN, true, false>(a, stream, geom, dry_run);
    return a.b_rs == 1 ? launch_short_k_layout<IN, false, true>(a, stream, geom, dry_run) : launch_short_k_layout<IN, false, false>(a, stream, geom, dry_run);
}

hipError_t launch_short_k(const GemmArgs& a, hipStream_t stream, LaunchGeom* geom, bool dry_run)
{
    switch (a.in_type) {
    case T_F16: return launch_in<IN_F16>(a, stream, geom, dry_run);
    case T_BF16: return launch_in<IN_BF16>(a, stream, geom, dry_run);
    case T_I8: return launch_in<IN_I8>(a, stream, geom, dry_run);
    default: return hipErrorInvalidValue;
    }
}

} // namespace acc950
