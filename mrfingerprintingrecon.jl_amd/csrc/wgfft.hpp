// Line FFTs by a whole workgroup: a stage's butterflies, over all the lines in
// LDS, are dealt out to the threads, at most 8 values (10 in radix 5, 9 in
// radix 3) per thread whatever the length's factors, and stages are separated
// by workgroup barriers.  The transforms of fft.hpp keep a line in one wavefront
// and need no barrier, but a plan with few threads per line (T = 1 to 16 where
// the factors 3 and 5 leave no common power of two) holds up to 40 values per
// thread.  The first stage can take its inputs from global memory and the last
// one hand its outputs over in registers, a line's LDS round trip less at
// either end.  Plans, twiddles and butterflies are those of fft.hpp: the results
// differ at most by the fused multiply-adds that the compiler chooses.
#pragma once

#include "fft.hpp"

namespace msr {

constexpr int WG_VALUES = 8;  // values per thread: blockDim.x * WG_VALUES >= lines * NF

// Lengths whose lines the fused 2D passes transform this way: plans that would
// hold more than 8 values per thread, the passes' threads mostly idle besides
// (at 128 x 96, 6 coils, K = 4, pass B of length 192 runs 64 of its 384 threads
// in the transforms, 24 values each, and spilled: 57 us, 16 this way).
template <int NF>
constexpr bool wg_preferred() { return NF / FFTPlan<NF>::T > 8; }

// butterflies per thread of a radix-R stage
constexpr int wg_per(int R) { return (WG_VALUES + R - 1) / R; }

// One stage of nl lines of NF by the whole workgroup (blockDim.x * 8 >= nl NF):
// in(m, p, v) fetches the R inputs of butterfly m, the thread's p-th, and
// out(m, p, v) transforms and hands them over.  SYNC: a barrier between the two
// (both in the same LDS lines).
template <int NF, int R, int NS, int DIR, bool SYNC, class CT, class IN, class OUT>
__device__ __forceinline__ void wg_stage(int nl, const CT* tw, IN&& in, OUT&& out) {
    constexpr int NB = NF / R, PER = wg_per(R);
    CT v[PER][R];
#pragma unroll
    for (int p = 0; p < PER; ++p) {
        const int m = threadIdx.x + p * blockDim.x;
        if (m < nl * NB) in(m, p, v[p]);
    }
    if constexpr (SYNC) __syncthreads();
#pragma unroll
    for (int p = 0; p < PER; ++p) {
        const int m = threadIdx.x + p * blockDim.x;
        if (m < nl * NB) out(m, p, v[p]);
    }
}

// LDS place of element i of a line, and the pitch of the lines: the swizzled
// layout of fft.hpp for ComplexF64 from 64 points on, its padding otherwise
template <int NF, class CT> constexpr bool wg_swizzled() { return sizeof(CT) == 16 && NF >= 64; }
template <int NF, class CT>
__device__ __forceinline__ int wg_at(int i) { return lds_pad<NF, CT, wg_swizzled<NF, CT>()>(i); }
template <int NF, class CT>
constexpr int wg_pitch() { return lds_line<NF, CT, wg_swizzled<NF, CT>()>() + 1; }

// Where butterfly m of a stage works: line l, butterfly j of the line.  Lines
// that are neighbours in memory (2^sh of them per plane k, line k 2^sh + w) may
// be dealt out line first, so that consecutive threads touch neighbours.
struct WgSpot {
    int l, j;
};
template <int NB>
__device__ __forceinline__ WgSpot wg_spot(int m, bool line_first, int sh) {
    if (!line_first) {
        const int l = m / NB;
        return {l, m - l * NB};
    }
    const int w = m & ((1 << sh) - 1), r = m >> sh, k = r / NB;
    return {(k << sh) + w, r - k * NB};
}

// Transform of nl lines, element i of line l at s[l * LP + wg_at(i)]:
// FIRST: get(l, i) supplies the first stage's inputs (dealt out line first if
// lf_in), else they are in LDS; LAST: put(p, r, l, i, value) takes the last
// stage's outputs (line first if lf_out), value p R + r of the thread, else
// they go to LDS.  Ends with a barrier (LDS free, or the result visible) unless
// LAST, where the caller places it before the LDS lines are written again.
// HALF: the upper half of the line is zero padding at that end: with an even
// radix there it is neither fetched nor handed over (with an odd one, get and
// put see all elements).
template <int NF, int DIR, int S, int NS, bool FIRST, bool LAST, class CT, bool HALF = false, class GET, class PUT>
__device__ __forceinline__ void wg_fft(CT* s, int nl, const CT* tw, bool lf_in, bool lf_out, int sh,
                                       GET&& get, PUT&& put) {
    using Pl = FFTPlan<NF>;
    if constexpr (S < Pl::NST) {
        constexpr int R = Pl::R[S], NB = NF / R, LP = wg_pitch<NF, CT>();
        constexpr bool GIN = FIRST && S == 0, POUT = LAST && S == Pl::NST - 1;
        constexpr int RIO = HALF && R % 2 == 0 ? R / 2 : R;  // values met at an outer end
        wg_stage<NF, R, NS, DIR, !GIN && !POUT, CT>(
            nl, tw,
            [&](int m, int, CT* v) {
                const WgSpot q = wg_spot<NB>(m, (GIN && lf_in) || (POUT && lf_out), sh);
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    if constexpr (GIN) v[r] = r < RIO ? get(q.l, q.j + r * NB) : cz<CT>();
                    else v[r] = s[q.l * LP + wg_at<NF, CT>(q.j + r * NB)];
                }
            },
            [&](int m, int p, CT* v) {
                const WgSpot q = wg_spot<NB>(m, (GIN && lf_in) || (POUT && lf_out), sh);
                const int k = q.j % NS;
                stage_twiddle<NF, R, NS, DIR>(v, tw, k);
                Butterfly<R, DIR>::run(v);
                const int base = (q.j - k) * R + k;
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    if constexpr (POUT) {
                        if (r < RIO) put(p, r, q.l, base + r * NS, v[r]);
                    } else {
                        s[q.l * LP + wg_at<NF, CT>(base + r * NS)] = v[r];
                    }
                }
            });
        if constexpr (!POUT) __syncthreads();
        wg_fft<NF, DIR, S + 1, NS * R, FIRST, LAST, CT, HALF>(s, nl, tw, lf_in, lf_out, sh, get, put);
    }
}

}  // namespace msr
