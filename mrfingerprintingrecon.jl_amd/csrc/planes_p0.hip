// Fused line passes for the lengths of part 0 (MSR_FFT_LINE_LENGTHS_P0).
#include "planes_impl.hpp"

namespace msr {

bool plane_part0(int which, const PlanePass& p, const void* tw, hipStream_t st) {
    MSR_PLANE_PART_BODY(MSR_FFT_LINE_LENGTHS_P0)
}

}  // namespace msr
