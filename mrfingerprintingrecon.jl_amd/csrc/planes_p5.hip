// Fused line passes for the lengths of part 5 (MSR_FFT_LINE_LENGTHS_P5).
#include "planes_impl.hpp"

namespace msr {

bool plane_part5(int which, const PlanePass& p, const void* tw, hipStream_t st) {
    MSR_PLANE_PART_BODY(MSR_FFT_LINE_LENGTHS_P5)
}

}  // namespace msr
