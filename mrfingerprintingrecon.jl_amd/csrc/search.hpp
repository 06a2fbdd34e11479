// Binary search over sorted keys, kept free of HIP so that its index range can
// be tested on the host.
#pragma once

#ifdef __HIPCC__
#define MSR_HOST_DEVICE __host__ __device__ __forceinline__
#else
#define MSR_HOST_DEVICE inline
#endif

namespace msr {

// First position i <= n with at(i) >= v, of n ascending keys at(0) .. at(n - 1).
// Reads positions in [0, n) only, for every n that an int holds: the middle is
// lo + (hi - lo) / 2, since lo + hi exceeds an int from 2^30 keys on.
template <class At>
MSR_HOST_DEVICE int lower_bound_at(int n, int v, At&& at) {
    int lo = 0, hi = n;
    while (lo < hi) {
        const int mid = lo + (hi - lo) / 2;
        if (at(mid) < v) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}

}  // namespace msr
