// Fused line passes for the lengths of part 2 (MSR_FFT_LINE_LENGTHS_P2).
#include "planes_impl.hpp"

namespace msr {

bool plane_part2(int which, const PlanePass& p, const void* tw, hipStream_t st) {
    MSR_PLANE_PART_BODY(MSR_FFT_LINE_LENGTHS_P2)
}

}  // namespace msr
