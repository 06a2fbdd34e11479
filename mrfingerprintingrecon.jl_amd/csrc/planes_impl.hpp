// Kernels of the fused line passes (see planes.hpp), instantiated per length
// by the planes_p*.hip translation units.  The lines of a workgroup are
// transformed by all its threads together (wgfft.hpp): with a few threads per
// line (fft_lds) the multiply took 148-256 VGPRs, one workgroup per CU, and
// 443 us at 240 x 300 / 12 coils / K = 6 in ComplexF64 instead of 228.
#pragma once

#include "planes.hpp"
#include "wgfft.hpp"

namespace msr {

constexpr int PLANE_KMAX = 8;        // coefficients held in registers by the multiply
constexpr int PLANE_MAX_ROW = 1024;  // longest row FFT (threads of a row tile)

// Workgroup i runs on XCD i mod 8: consecutive logical blocks on one XCD when
// the count divides by 8, so neighbours share their L2's lines.
__device__ __forceinline__ int64_t plane_xcd(int64_t b, int64_t n) {
    return n % 8 ? b : (b % 8) * (n / 8) + b / 8;
}

// rows per tile: 64-byte pieces of neighbouring rows, more for short lines
// (at least 128 threads)
template <int NF, class CT>
constexpr int plane_rows() {
    int f = sizeof(CT) == 16 ? 4 : 8;
    while (f < 32 && f * NF < 128 * WG_VALUES) f *= 2;
    while (f > 1 && f * NF > 1024 * WG_VALUES) f /= 2;
    return f;
}
constexpr int plane_shift(int f) { return f <= 1 ? 0 : 1 + plane_shift(f / 2); }
template <int NF, class CT>
constexpr int plane_row_block() {
    return ((plane_rows<NF, CT>() * NF + WG_VALUES - 1) / WG_VALUES + 63) / 64 * 64;
}

// ---------------------------------------------------------------- expand
// Block = (row tile, k, c), the coil fastest: a tile of b is read from HBM
// once for all coils.
template <int NF, class CT>
__global__ void __launch_bounds__((plane_row_block<NF, CT>()))
plane_expand_kernel(PlanePass p, const CT* __restrict__ tw) {
    if (p.skip && *p.skip) return;
    constexpr int F = plane_rows<NF, CT>(), SH = plane_shift(F), BLK = plane_row_block<NF, CT>();
    constexpr int LP = wg_pitch<NF, CT>();
    __shared__ CT s[F * LP];
    const int64_t tiles = (p.nrows + F - 1) / F;
    const int64_t lb = plane_xcd(blockIdx.x, tiles * p.K * p.nc);
    const int c = (int)(lb % p.nc), k = (int)((lb / p.nc) % p.K);
    const int64_t r0 = lb / ((int64_t)p.nc * p.K) * F;
    const int nr = (int)(p.nrows - r0 < F ? p.nrows - r0 : F), len = p.len;
    const CT* b = static_cast<const CT*>(p.b) + ((int64_t)k * p.nrows + r0) * len;
    const float2* cm = p.cmaps ? p.cmaps + ((int64_t)c * p.nrows + r0) * len : nullptr;
    CT* T = static_cast<CT*>(p.T) + ((int64_t)c * p.K + k) * p.plane + r0 * p.rs;
    auto get = [&](int l, int i) {
        if (i >= len || l >= nr) return cz<CT>();
        const CT v = b[l * len + i];
        return cm ? cmul(cto<CT>(cm[l * len + i]), v) : v;
    };
    if (p.qs == 1) {  // rows stay rows: straight from the last stage
        wg_fft<NF, -1, 0, 1, true, true, CT>(s, F, tw, false, false, SH, get,
            [&](int, int, int l, int q, CT v) { if (l < nr) T[l * p.rs + q] = v; });
        return;
    }
    wg_fft<NF, -1, 0, 1, true, false, CT>(s, F, tw, false, false, SH, get, [](int, int, int, int, CT) {});
    for (int e = threadIdx.x; e < F * NF; e += BLK) {
        const int q = e >> SH, l = e & (F - 1);
        if (l < nr) T[l * p.rs + q * p.qs] = s[l * LP + wg_at<NF, CT>(q)];
    }
}

// --------------------------------------------------------------- combine
// Block = (row tile, coil group, k), the coefficient fastest (a group's coil
// map tiles are read once for all coefficients).
template <int NF, class CT>
__global__ void __launch_bounds__((plane_row_block<NF, CT>()))
plane_combine_kernel(PlanePass p, const CT* __restrict__ tw) {
    if (p.skip && *p.skip) return;
    constexpr int F = plane_rows<NF, CT>(), SH = plane_shift(F);
    constexpr int LP = wg_pitch<NF, CT>();
    constexpr int RL = FFTPlan<NF>::R[FFTPlan<NF>::NST - 1], PER = wg_per(RL), NBL = NF / RL;
    __shared__ CT s[F * LP];
    const int64_t tiles = (p.nrows + F - 1) / F;
    const int64_t lb = plane_xcd(blockIdx.x, tiles * p.K * p.G);
    const int k = (int)(lb % p.K), grp = (int)((lb / p.K) % p.G);
    const int64_t r0 = lb / ((int64_t)p.K * p.G) * F;
    const int c0 = (int)((int64_t)p.nc * grp / p.G), c1 = (int)((int64_t)p.nc * (grp + 1) / p.G);
    const int nr = (int)(p.nrows - r0 < F ? p.nrows - r0 : F), len = p.len;
    CT* part = static_cast<CT*>(p.partial) + (((int64_t)grp * p.K + k) * p.nrows + r0) * len;
    CT acc[PER * RL];
    // the thread's outputs of the last stage: visit(value index, row, element)
    auto mine = [&](auto&& visit) {
#pragma unroll
        for (int q = 0; q < PER; ++q) {
            const int m = threadIdx.x + q * blockDim.x;
            if (m >= F * NBL) continue;
            // (one stage alone is dealt out as its inputs are)
            const WgSpot w = wg_spot<NBL>(m, FFTPlan<NF>::NST == 1 && p.qs != 1, SH);
#pragma unroll
            for (int r = 0; r < RL; ++r)
                if (w.j + r * NBL < len && w.l < nr) visit(q * RL + r, w.l * len + w.j + r * NBL);
        }
    };
#pragma unroll
    for (int q = 0; q < PER * RL; ++q) acc[q] = cz<CT>();
    if (p.accumulate) mine([&](int a, int o) { acc[a] = part[o]; });
    for (int c = c0; c < c1; ++c) {
        const CT* T = static_cast<const CT*>(p.T) + ((int64_t)c * p.K + k) * p.plane + r0 * p.rs;
        const float2* cm = p.cmaps ? p.cmaps + ((int64_t)c * p.nrows + r0) * len : nullptr;
        wg_fft<NF, +1, 0, 1, true, true, CT>(s, F, tw, p.qs != 1, false, SH,
            [&](int l, int q) { return l < nr ? T[l * p.rs + q * p.qs] : cz<CT>(); },
            [&](int q, int r, int l, int i, CT v) {
                if (i < len && l < nr) {
                    if (cm) cfmac(acc[q * RL + r], cto<CT>(cm[l * len + i]), v);
                    else acc[q * RL + r] = cadd(acc[q * RL + r], v);
                }
            });
        if constexpr (FFTPlan<NF>::NST > 1) __syncthreads();
    }
    mine([&](int a, int o) { part[o] = acc[a]; });
}

// -------------------------------------------------------------- multiply
// In-place product of one cell's K values (col[k step]) with its kernel, entry e
// at lam[e NF]: the full K x K block (FULL) or the packed Hermitian (real
// symmetric) upper triangle.  A column's entries are loaded together, past the
// end the last one again, while the column before is multiplied: guarded by
// j < K one by one they were waited for one by one (127 us per multiply at
// 256 x 256 / 20 coils / K = 5, full complex blocks, instead of 72).
template <int NF, bool FULL, class CT, class LT>
__device__ __forceinline__ void plane_cell(const LT* __restrict__ lam, int K, CT* col, int step) {
    using RT = real_t<CT>;
    constexpr int KM = PLANE_KMAX;
    auto column = [&](int k, LT (&l)[KM]) {  // k: compile-time after unrolling
        const int kk = k < K ? k : K - 1;
        const LT* src = lam + (FULL ? K * kk : kk * (kk + 1) / 2) * NF;
        const int last = FULL ? K - 1 : kk;
#pragma unroll
        for (int j = 0; j < KM; ++j)
            if (FULL || j <= k) l[j] = src[(j < last ? j : last) * NF];
    };
    auto term = [](CT& a, LT l, CT x, bool conj) {
        if constexpr (sizeof(LT) == sizeof(float)) {
            a.x = fma((RT)l, x.x, a.x);
            a.y = fma((RT)l, x.y, a.y);
        } else if (conj) {
            cfmac(a, cto<CT>(l), x);
        } else {
            cfma(a, cto<CT>(l), x);
        }
    };
    CT in[KM], acc[KM];
    LT l[KM], next[KM];
    column(0, l);
#pragma unroll
    for (int k = 0; k < KM; ++k) {
        acc[k] = cz<CT>();
        in[k] = col[(k < K ? k : K - 1) * step];
    }
#pragma unroll
    for (int k = 0; k < KM; ++k)
        if (k < K) {
            if (k + 1 < KM) column(k + 1, next);
#pragma unroll
            for (int j = 0; j < KM; ++j) {
                if (FULL || j <= k) term(acc[j], l[j], in[k], false);
                if (!FULL && j < k) term(acc[k], l[j], in[j], true);
            }
#pragma unroll
            for (int j = 0; j < KM; ++j)
                if (FULL || j <= k + 1) l[j] = next[j];
        }
#pragma unroll
    for (int k = 0; k < KM; ++k)
        if (k < K) col[k * step] = acc[k];
}

// Block = (column tile of 2^wcs columns, coil), the coil fastest (the blocks of
// one tile run on one XCD and share its kernel entries in L2); the K lines of
// every column in LDS: forward FFT, K x K multiply per cell (one thread per
// cell, entries read coalesced along the line), inverse FFT, the stored
// elements written back in place.
template <int NF, class CT>
__global__ void __launch_bounds__(1024)
plane_multiply_kernel(PlanePass p, const CT* __restrict__ tw, int wcs) {
    if (p.skip && *p.skip) return;
    constexpr int LP = wg_pitch<NF, CT>();
    extern __shared__ double2 plane_lds[];
    CT* s = reinterpret_cast<CT*>(plane_lds);
    const int K = p.K, NL = K << wcs, len = p.len;
    const int64_t tiles = (p.ncols + (1 << wcs) - 1) >> wcs;
    const int64_t lb = plane_xcd(blockIdx.x, tiles * p.nc);
    const int c = (int)(lb % p.nc);
    const int64_t col0 = (lb / p.nc) << wcs;
    const int ncol = (int)(p.ncols - col0 < (1 << wcs) ? p.ncols - col0 : (int64_t)1 << wcs);
    const int P = p.lam_full ? K * K : K * (K + 1) / 2;
    CT* T = static_cast<CT*>(p.T) + (int64_t)c * K * p.plane + col0 * p.cs;
    const bool lf = p.es != 1;
    const int wm = (1 << wcs) - 1;
    // line l = k 2^wcs + w; a thread stores what its own block alone has read
    wg_fft<NF, -1, 0, 1, true, false, CT>(s, NL, tw, lf, false, wcs,
        [&](int l, int i) {
            const int w = l & wm;
            return i < len && w < ncol ? T[(l >> wcs) * p.plane + w * p.cs + i * p.es] : cz<CT>();
        },
        [](int, int, int, int, CT) {});
    auto multiply = [&]<bool FULL, class LT>(const LT* lam) {
        for (int v = threadIdx.x; v < (NF << wcs); v += blockDim.x) {
            const int w = v / NF, i = v - w * NF;
            if (w < ncol)
                plane_cell<NF, FULL>(lam + (col0 + w) * P * NF + i, K, s + w * LP + wg_at<NF, CT>(i), LP << wcs);
        }
    };
    if (p.lam_full) {
        if (p.lam_real) multiply.template operator()<true>(static_cast<const float*>(p.lam));
        else multiply.template operator()<true>(static_cast<const float2*>(p.lam));
    } else {
        if (p.lam_real) multiply.template operator()<false>(static_cast<const float*>(p.lam));
        else multiply.template operator()<false>(static_cast<const float2*>(p.lam));
    }
    __syncthreads();
    wg_fft<NF, +1, 0, 1, false, true, CT>(s, NL, tw, false, lf, wcs,
        [](int, int) { return cz<CT>(); },
        [&](int, int, int l, int i, CT v) {
            const int w = l & wm;
            if (i < len && w < ncol) T[(l >> wcs) * p.plane + w * p.cs + i * p.es] = v;
        });
}

// ---------------------------------------------------------- forward model
// Stored element of FFT bin q when the len elements are centred on frequency
// zero (element len/2 in bin 0), or >= len in the padding.
template <int NF>
__device__ __forceinline__ int plane_centred(int q, int len) {
    const int i = q + len / 2;
    return i >= NF ? i - NF : i;
}

// Block = (row tile, k, c): rows of S_c x_k, placed, deapodised and transformed
// along x, written transposed.
template <int NF>
__global__ void __launch_bounds__((plane_row_block<NF, float2>()))
plane_place_kernel(PlanePass p, const float2* __restrict__ tw) {
    constexpr int F = plane_rows<NF, float2>(), SH = plane_shift(F), BLK = plane_row_block<NF, float2>();
    constexpr int LP = wg_pitch<NF, float2>();
    __shared__ float2 s[F * LP];
    const int64_t tiles = (p.nrows + F - 1) / F;
    const int64_t lb = plane_xcd(blockIdx.x, tiles * p.K * p.nc);
    const int c = (int)(lb % p.nc), k = (int)((lb / p.nc) % p.K);
    const int64_t r0 = lb / ((int64_t)p.nc * p.K) * F;
    const int nr = (int)(p.nrows - r0 < F ? p.nrows - r0 : F), len = p.len;
    const float2* b = static_cast<const float2*>(p.b) + ((int64_t)k * p.nrows + r0) * len;
    const float2* cm = p.cmaps ? p.cmaps + ((int64_t)c * p.nrows + r0) * len : nullptr;
    float2* T = static_cast<float2*>(p.T) + ((int64_t)k * p.nc + c) * p.plane + r0;
    wg_fft<NF, -1, 0, 1, true, false, float2>(s, F, tw, false, false, SH,
        [&](int l, int q) {
            const int i = plane_centred<NF>(q, len);
            if (i >= len || l >= nr) return make_float2(0.f, 0.f);
            const float2 v = b[l * len + i];
            return cscale(cm ? cmul(cm[l * len + i], v) : v, p.win[i]);
        },
        [](int, int, int, int, float2) {});
    for (int e = threadIdx.x; e < F * NF; e += BLK) {
        const int q = e >> SH, l = e & (F - 1);
        if (l < nr) T[l + (int64_t)q * p.nrows] = s[l * LP + wg_at<NF, float2>(q)];
    }
}

// Block = (k, coil group, column): the group's lines along y, placed and
// transformed, written with the coils side by side.
template <int NF>
__global__ void __launch_bounds__(1024) plane_coils_kernel(PlanePass p, const float2* __restrict__ tw) {
    constexpr int F = PLANE_COIL_GROUP, LP = wg_pitch<NF, float2>();
    __shared__ float2 s[F * LP];
    const int CB = (p.nc + F - 1) / F, len = p.len;
    const int64_t lb = plane_xcd(blockIdx.x, p.ncols * CB * p.K);
    const int64_t col = lb % p.ncols, g = lb / p.ncols;  // g = k CB + coil group
    const int k = (int)(g / CB), c0 = (int)(g % CB) * F;
    const float2* T = static_cast<const float2*>(p.T) + ((int64_t)k * p.nc + c0) * p.plane + col * len;
    wg_fft<NF, -1, 0, 1, true, false, float2>(s, F, tw, false, false, 3,
        [&](int l, int q) {
            const int i = plane_centred<NF>(q, len);
            if (i >= len || c0 + l >= p.nc) return make_float2(0.f, 0.f);
            return cscale(T[l * p.plane + i], p.win[i]);
        },
        [](int, int, int, int, float2) {});
    float2* out = p.out + (g * p.ncols + col) * NF * F;
    for (int e = threadIdx.x; e < F * NF; e += blockDim.x)
        out[e] = s[(e & (F - 1)) * LP + wg_at<NF, float2>(e / F)];
}

// ---------------------------------------------------------------- launch
inline unsigned plane_grid(int64_t n) {
    MSR_REQUIRE(n >= 1 && n < (int64_t)1 << 31, MSR_ERR_ARGUMENT, "launch of %lld blocks", (long long)n);
    return (unsigned)n;
}

template <int NF, class CT>
void launch_plane_n(int which, const PlanePass& p, const CT* tw, hipStream_t st) {
    if (which == PLANE_PLACE || which == PLANE_COILS) {
        if constexpr (sizeof(CT) == 8 && NF <= PLANE_MAX_ROW) {
            if (which == PLANE_PLACE) {
                const int64_t tiles = ceil_div(p.nrows, plane_rows<NF, CT>());
                constexpr int BLK = plane_row_block<NF, CT>();
                hipLaunchKernelGGL((plane_place_kernel<NF>), dim3(plane_grid(tiles * p.K * p.nc)), dim3(BLK),
                                   0, st, p, tw);
            } else {
                constexpr int BLK = (PLANE_COIL_GROUP * NF + WG_VALUES - 1) / WG_VALUES;
                hipLaunchKernelGGL((plane_coils_kernel<NF>),
                                   dim3(plane_grid(p.ncols * ceil_div(p.nc, PLANE_COIL_GROUP) * p.K)),
                                   dim3((BLK + 63) / 64 * 64), 0, st, p, tw);
            }
        } else {
            fail(MSR_ERR_ERROR, "forward-model pass of length %d", NF);
        }
        return;
    }
    if (which == PLANE_MULTIPLY) {
        // columns per block: strided ones 64 bytes of neighbours, contiguous
        // ones up to 256 threads; fewer while the block would leave room for
        // one block per CU only, or exceed 1024 threads
        auto bytes = [&](int w) { return sizeof(CT) * ((size_t)p.K << w) * wg_pitch<NF, CT>(); };
        auto threads = [&](int w) { return ((p.K << w) * NF + WG_VALUES - 1) / WG_VALUES; };
        int wcs = sizeof(CT) == 16 ? 2 : 3;
        if (p.es == 1)
            for (wcs = 0; threads(wcs + 1) <= 256 && (int64_t)1 << wcs < p.ncols; ++wcs) {}
        while (wcs > 0 && (bytes(wcs) > (size_t)80 * 1024 || threads(wcs) > 1024)) --wcs;
        MSR_REQUIRE(threads(wcs) <= 1024 && bytes(wcs) <= (size_t)160 * 1024, MSR_ERR_ERROR,
                    "%d lines of %d values exceed the workgroup", p.K, NF);
        const int64_t tiles = (p.ncols + (1 << wcs) - 1) >> wcs;
        const size_t lds = bytes(wcs);
        const int blk = (threads(wcs) + 63) / 64 * 64;
        hipLaunchKernelGGL((plane_multiply_kernel<NF, CT>), dim3(plane_grid(tiles * p.nc)), dim3(blk), lds,
                           st, p, tw, wcs);
        return;
    }
    if constexpr (NF <= PLANE_MAX_ROW) {
        const int64_t tiles = ceil_div(p.nrows, plane_rows<NF, CT>());
        constexpr int BLK = plane_row_block<NF, CT>();
        if (which == PLANE_EXPAND)
            hipLaunchKernelGGL((plane_expand_kernel<NF, CT>), dim3(plane_grid(tiles * p.K * p.nc)),
                               dim3(BLK), 0, st, p, tw);
        else
            hipLaunchKernelGGL((plane_combine_kernel<NF, CT>), dim3(plane_grid(tiles * p.K * p.G)),
                               dim3(BLK), 0, st, p, tw);
    } else {
        fail(MSR_ERR_ERROR, "row pass of length %d", NF);
    }
}

#define MSR_PLANE_PART_BODY(LIST) \
    switch (p.nf) {               \
        LIST(MSR_PLANE_CASE)      \
        default: return false;    \
    }
#define MSR_PLANE_CASE(NN)                                                               \
    case NN:                                                                             \
        if (p.f64) launch_plane_n<NN, double2>(which, p, static_cast<const double2*>(tw), st); \
        else launch_plane_n<NN, float2>(which, p, static_cast<const float2*>(tw), st);   \
        return true;

}  // namespace msr
