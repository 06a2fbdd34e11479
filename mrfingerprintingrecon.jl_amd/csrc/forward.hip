// Forward subspace model (type-2 NUFFT side), the data simulation of the
// reference tests (test/reconstruct_radial.jl:62-74: for every coil and frame,
// NonuniformFFTs exec_type2! of S_c * sum_k U[t, k] x_k):
//   y_{j,c} = sum_k U[t_j, k] sum_n S_c[n] x_k[n] exp(-2 pi i k_j . (n - N/2))
// On the device: S_c x_k, centred placement on the sigma = 2 grid with
// deapodisation 1/phihat, forward FFTs, then ES interpolation (W = 8) at the
// samples.  Two forms of the interpolation:
//  - 2D, on the matrix cores (interp_mfma_kernel): samples sorted by region of
//    4 x 5 cells, 16 samples of one region at a time;
//  - one wavefront per sample (interp_kernel: 3D, and the shapes the rule in
//    fwd_batches_pay leaves): each lane owns one kernel cell, folds the K
//    channels with U[t_j, k] in registers, and the wavefront reduces the 64
//    (8x8, z looped in 3D) cell contributions.
#include <algorithm>

#include <hipcub/hipcub.hpp>

#include "fft.hpp"
#include "fftlines.hpp"
#include "planes.hpp"
#include "search.hpp"
#include "spread.hpp"

namespace msr {

void fill_floats(void* p, int64_t n, float v, hipStream_t st);  // normalop.hip

// Z[(c*K + k)][v] = S_c[v] x_k[v]
__global__ void expand_kernel(const float2* __restrict__ x, const float2* __restrict__ cmaps, int C,
                              int K, int64_t V, float2* __restrict__ Z) {
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < (int64_t)C * K * V;
         e += (int64_t)gridDim.x * blockDim.x) {
        const int64_t v = e % V;
        const int64_t ck = e / V;
        const int k = (int)(ck % K), c = (int)(ck / K);
        const float2 xv = x[(int64_t)k * V + v];
        Z[e] = cmaps ? cmul(cmaps[(int64_t)c * V + v], xv) : xv;
    }
}

__device__ __forceinline__ float es_phi_fw(float t) {
    const float z = t * (2.0f / SPREAD_W);
    const float a = 1.0f - z * z;
    return a > 0.0f ? expf(SPREAD_BETA * (sqrtf(a) - 1.0f)) : 0.0f;
}

__device__ __forceinline__ void cell_frac(float k, int64_t n, int64_t& cell, float& frac) {
    const double s = (double)k * (double)n;
    const double fl = floor(s);
    frac = (float)(s - fl);
    int64_t c = (int64_t)fl % n;
    if (c < 0) c += n;
    cell = c;
}

struct FwdGeom {
    int64_t n[3];
};

// one wavefront per sample; lane = kernel cell (ox, oy), z looped.  The
// sample's position, weights and frame are read once; its coils run in
// groups of FW_CB whose grid loads are independent of each other (several
// loads in flight per wavefront); a group is reduced over the 64 cells by one
// reduce-scatter (10 lane exchanges for 4 coils instead of 48).  Each
// (sample, coil) sums its K channels in channel order and its cells in a
// fixed tree.
constexpr int FW_CB = 4;  // the reduce-scatter below splits lane bits 5..3 over 4 coils x 2 parts
static_assert(FW_CB == 4, "the interpolation reduce-scatter is written for 4 coils");
template <int D>
__global__ void __launch_bounds__(256)
interp_kernel(const float* __restrict__ kc, const int* __restrict__ frame,
              const int64_t* __restrict__ sel, int64_t M, int64_t nsel, const float2* __restrict__ G,
              FwdGeom g, int K, int C, const void* __restrict__ U, int u_real, int64_t nt,
              float2* __restrict__ out) {
    const int lane = threadIdx.x & 63;
    const int ox = (lane & 7) - 3, oy = (lane >> 3) - 3;
    const int64_t wave0 = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const int64_t nwaves = ((int64_t)gridDim.x * blockDim.x) >> 6;
    const int64_t Gc = g.n[0] * g.n[1] * g.n[2];
    for (int64_t j = wave0; j < M; j += nwaves) {
        int64_t cx, cy, cz = 0;
        float fx, fy, fz = 0.f;
        cell_frac(kc[j * D + 0], g.n[0], cx, fx);
        cell_frac(kc[j * D + 1], g.n[1], cy, fy);
        if (D == 3) cell_frac(kc[j * D + 2], g.n[2], cz, fz);
        const float wxy = es_phi_fw((float)ox - fx) * es_phi_fw((float)oy - fy);
        int64_t gx = (cx + ox) % g.n[0];
        if (gx < 0) gx += g.n[0];
        int64_t gy = (cy + oy) % g.n[1];
        if (gy < 0) gy += g.n[1];
        const int64_t off = gy * g.n[0] + gx;
        const int t = frame[j];
        const int64_t idx = sel ? sel[j] : j;
        for (int c0 = 0; c0 < C; c0 += FW_CB) {
            float2 acc[FW_CB];
#pragma unroll
            for (int cc = 0; cc < FW_CB; ++cc) acc[cc] = make_float2(0.f, 0.f);
            for (int k = 0; k < K; ++k) {
                float2 u;
                if (!U) u = make_float2(t == k ? 1.f : 0.f, 0.f);
                else if (u_real) u = make_float2(reinterpret_cast<const float*>(U)[t + (int64_t)k * nt], 0.f);
                else u = reinterpret_cast<const float2*>(U)[t + (int64_t)k * nt];
#pragma unroll
                for (int cc = 0; cc < FW_CB; ++cc) {
                    const int c = c0 + cc < C ? c0 + cc : C - 1;  // a spare slot repeats the last coil
                    const float2* Gk = G + ((int64_t)c * K + k) * Gc;
                    float2 s = make_float2(0.f, 0.f);
                    if (D == 2) {
                        const float2 v = Gk[off];
                        s = make_float2(wxy * v.x, wxy * v.y);
                    } else {
#pragma unroll
                        for (int oz = -3; oz <= 4; ++oz) {
                            int64_t gz = (cz + oz) % g.n[2];
                            if (gz < 0) gz += g.n[2];
                            const float wz = wxy * es_phi_fw((float)oz - fz);
                            const float2 v = Gk[gz * g.n[1] * g.n[0] + off];
                            s.x += wz * v.x;
                            s.y += wz * v.y;
                        }
                    }
                    cfma(acc[cc], u, s);
                }
            }
            // reduce-scatter over the 64 lanes: lane bits 5, 4 pick the coil
            // of the group, bit 3 the component, then bits 2..0 sum it
            float a[2 * FW_CB];
#pragma unroll
            for (int cc = 0; cc < FW_CB; ++cc) {
                a[2 * cc] = acc[cc].x;
                a[2 * cc + 1] = acc[cc].y;
            }
#pragma unroll
            for (int h = 2 * FW_CB / 2, bit = 32; h >= 1; h >>= 1, bit >>= 1) {
                const bool up = (lane & bit) != 0;
#pragma unroll
                for (int i = 0; i < h; ++i) {
                    const float send = up ? a[i] : a[h + i];
                    const float keep = up ? a[h + i] : a[i];
                    a[i] = keep + __shfl_xor(send, bit, 64);
                }
            }
#pragma unroll
            for (int o = 4; o > 0; o >>= 1) a[0] += __shfl_xor(a[0], o, 64);
            const int cc = lane >> 4, comp = (lane >> 3) & 1;
            if ((lane & 7) == 0 && c0 + cc < C)
                reinterpret_cast<float*>(out)[2 * (idx + (int64_t)(c0 + cc) * nsel) + comp] = a[0];
        }
    }
}

// --------------------------------------------- 2D on the matrix cores
// A region is 4 x 5 cells; the kernels of the samples whose floor cell lies in
// it reach 11 x 12 cells (rows qx, columns qy).  One wavefront takes 16 samples
// of a region (the MFMA's columns) and, group by group of 8 coils, the product
//   Z (16 floats: 8 coils re/im x 16 samples) = G (16 x 132 cells) W (132 x 16)
// as 33 v_mfma_f32_16x16x4f32, four neighbouring cells along qy per step: lane
// (r = lane mod 16, s = lane div 16) supplies float r of cell s (the grid is
// stored [k][coil group][qx][qy][8 coils], so a step's 64 lanes read 256
// consecutive bytes) and the weight w_x w_y of cell s for sample r.  The rows
// of cells go to four accumulators in turn, each of which holds two coils of one
// sample, the middle columns (the largest weights) last; their sum is folded
// with U[t_j, k], in Float64, before the next coefficient.  A step's grid values
// are loaded one (coil group, coefficient) ahead.
//
// Error: one accumulator for all 132 products and a fold in Float32 gave 1.03 to
// 1.08 times the error against 64 bits of the lane tree below (interp_kernel);
// this form 0.997 to 1.002 times (32 x 32 to 500 x 500, K = 1 to 8).
//
// Bound: matrix-core issue (33 x 32 cycles per 16 samples, coefficient and 8
// coils; the 64 cells of a kernel are 48 % of the region's 132, and a region
// away from the centre fills about 12 of the 16 columns).  At 256 x 256, 20
// coils, K = 5, 512 000 samples on MI355X: interpolation
// 3.43 -> 0.55 ms, a call with its FFTs 4.11 -> 0.68 ms.  Three waves per SIMD:
// with four the accumulators lie in AGPRs and the call takes 0.72 ms (320 x 240, 32
// coils, 2.02 ms for 1.88; 384 x 384, 16 coils, the other way, 0.54 for 0.55).
constexpr int FW_TX = 4, FW_TY = 5;                      // region (floor cells)
constexpr int FW_RX = FW_TX + 7, FW_RY = (FW_TY + 7) / 4;  // rows, column quads it reaches
constexpr int FW_STEPS = FW_RX * FW_RY;
static_assert(FW_RY * 4 == FW_TY + 7, "the columns of a region come in quads");
constexpr int FW_ACC = 4;                                // accumulators
constexpr int FW_PTS = 16;                               // samples per batch

__global__ void fwd_region_kernel(const float* __restrict__ kc, int64_t M, FwdGeom g, int nry,
                                  int* __restrict__ key, int* __restrict__ idx) {
    for (int64_t j = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; j < M;
         j += (int64_t)gridDim.x * blockDim.x) {
        int64_t cx, cy;
        float f;
        cell_frac(kc[2 * j], g.n[0], cx, f);
        cell_frac(kc[2 * j + 1], g.n[1], cy, f);
        key[j] = (int)(cx / FW_TX) * nry + (int)(cy / FW_TY);
        idx[j] = (int)j;
    }
}

// first position of a sorted key >= v
__device__ __forceinline__ int lower_bound(const int* __restrict__ sorted, int n, int v) {
    return lower_bound_at(n, v, [&](int i) { return sorted[i]; });
}

// first[r] = first sample of region r (r <= nr), nb[r] = its batches
__global__ void fwd_count_kernel(const int* __restrict__ sorted, int M, int nr, int* __restrict__ first,
                                 int* __restrict__ nb) {
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r > nr) return;
    const int a = lower_bound(sorted, M, r);
    first[r] = a;
    nb[r] = r < nr ? (lower_bound(sorted, M, r + 1) - a + FW_PTS - 1) / FW_PTS : 0;
}

// batch b -> {region, first sample, samples}
__global__ void fwd_batch_kernel(const int* __restrict__ first, const int* __restrict__ pos, int nr, int nbatch,
                                 int4* __restrict__ batches) {
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= nbatch) return;
    const int r = lower_bound(pos, nr + 1, b + 1) - 1;  // pos[r] <= b < pos[r + 1]
    const int s = first[r] + (b - pos[r]) * FW_PTS;
    const int left = first[r + 1] - s;
    batches[b] = make_int4(r, s, left < FW_PTS ? left : FW_PTS, 0);
}

// Samples sorted by region (stable) and cut into batches, once per trajectory
// and grid; only the building holds the handle.
static const FwdPlan& fwd_plan(const msr_traj* traj, const FwdGeom& g, hipStream_t st) {
    std::lock_guard<std::recursive_mutex> lock(traj->mu);
    std::array<int64_t, 2> key{g.n[0], g.n[1]};
    auto it = traj->fwd_plans.find(key);
    if (it != traj->fwd_plans.end()) return *it->second;
    auto p = std::make_unique<FwdPlan>();
    const int M = (int)traj->M;
    p->nry = (int)ceil_div(g.n[1], FW_TY);
    const int nr = (int)ceil_div(g.n[0], FW_TX) * p->nry;
    TempBuf keys{st}, sorted{st}, idx{st}, temp{st}, first{st}, nb{st}, pos{st};
    keys.alloc(sizeof(int) * M);
    sorted.alloc(sizeof(int) * M);
    idx.alloc(sizeof(int) * M);
    p->perm.alloc(sizeof(int) * M);
    first.alloc(sizeof(int) * (nr + 1));
    nb.alloc(sizeof(int) * (nr + 1));
    pos.alloc(sizeof(int) * (nr + 1));
    const int grid = (int)std::min<int64_t>((traj->M + 255) / 256, 8192);
    hipLaunchKernelGGL(fwd_region_kernel, dim3(grid), dim3(256), 0, st, traj->kc.as<float>(), traj->M, g,
                       p->nry, keys.as<int>(), idx.as<int>());
    MSR_CHECK_LAUNCH();
    int bits = 1;
    while ((int64_t(1) << bits) < nr) ++bits;
    size_t tb = 0, ts = 0;
    MSR_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, tb, keys.as<int>(), sorted.as<int>(), idx.as<int>(),
                                               p->perm.as<int>(), M, 0, bits, st));
    MSR_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, ts, nb.as<int>(), pos.as<int>(), nr + 1, st));
    temp.alloc(std::max<size_t>(std::max(tb, ts), 16));
    MSR_HIP(hipcub::DeviceRadixSort::SortPairs(temp.p, tb, keys.as<int>(), sorted.as<int>(), idx.as<int>(),
                                               p->perm.as<int>(), M, 0, bits, st));
    hipLaunchKernelGGL(fwd_count_kernel, dim3((nr + 256) / 256), dim3(256), 0, st, sorted.as<int>(), M, nr,
                       first.as<int>(), nb.as<int>());
    MSR_CHECK_LAUNCH();
    MSR_HIP(hipcub::DeviceScan::ExclusiveSum(temp.p, ts, nb.as<int>(), pos.as<int>(), nr + 1, st));
    MSR_HIP(hipMemcpyAsync(&p->nbatch, pos.as<int>() + nr, sizeof(int), hipMemcpyDeviceToHost, st));
    MSR_HIP(hipStreamSynchronize(st));
    p->batches.alloc(sizeof(int4) * std::max(p->nbatch, 1));
    hipLaunchKernelGGL(fwd_batch_kernel, dim3((p->nbatch + 255) / 256), dim3(256), 0, st, first.as<int>(),
                       pos.as<int>(), nr, p->nbatch, p->batches.as<int4>());
    MSR_CHECK_LAUNCH();
    MSR_HIP(hipStreamSynchronize(st));  // temporaries are freed on return
    auto& ref = *p;
    traj->fwd_plans[key] = std::move(p);
    return ref;
}

using f32x4 = __attribute__((__vector_size__(4 * sizeof(float)))) float;

__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3, 3)))
interp_mfma_kernel(const float* __restrict__ kc, const int* __restrict__ frame, const int64_t* __restrict__ sel,
                   const int* __restrict__ perm, const int4* __restrict__ batches, int nbatch, int nry,
                   int64_t nsel, const float* __restrict__ G, FwdGeom g, int K, int C,
                   const void* __restrict__ U, int u_real, int64_t nt, float2* __restrict__ out) {
    // consecutive batches (neighbouring regions) on one XCD
    const int nblk = gridDim.x;
    const int lb = nblk % 8 ? (int)blockIdx.x : (int)(blockIdx.x % 8) * (nblk / 8) + (int)blockIdx.x / 8;
    const int wv = __builtin_amdgcn_readfirstlane(lb * 4 + (threadIdx.x >> 6));
    if (wv >= nbatch) return;
    const int lane = threadIdx.x & 63, r = lane & 15, s = lane >> 4;
    const int4 bt = batches[wv];
    const int X0 = bt.x / nry * FW_TX - 3, Y0 = bt.x % nry * FW_TY - 3;  // first cell reached
    const bool on = r < bt.z;
    const int64_t j = perm[bt.y + (on ? r : 0)];
    int64_t cx, cy;
    float fx, fy;
    cell_frac(kc[2 * j], g.n[0], cx, fx);
    cell_frac(kc[2 * j + 1], g.n[1], cy, fy);
    const int t = frame[j];
    const int64_t idx = sel ? sel[j] : j;
    const int n0 = (int)g.n[0], n1 = (int)g.n[1];
    float wx[FW_RX], wy[FW_RY];
    int oy[FW_RY];
#pragma unroll
    for (int i = 0; i < FW_RX; ++i) wx[i] = on ? es_phi_fw((float)(X0 + i - (int)cx) - fx) : 0.f;
#pragma unroll
    for (int q = 0; q < FW_RY; ++q) {
        const int y = Y0 + 4 * q + s;
        wy[q] = es_phi_fw((float)(y - (int)cy) - fy);
        oy[q] = ((y % n1 + n1) % n1) * (2 * PLANE_COIL_GROUP) + r;  // float of the cell
    }
    const int CB = (C + PLANE_COIL_GROUP - 1) / PLANE_COIL_GROUP, ng = CB * K;
    const int64_t plane = (int64_t)n0 * n1 * (2 * PLANE_COIL_GROUP);
    const int row = n1 * 2 * PLANE_COIL_GROUP;
    float a[FW_STEPS];
    // group q = cb K + k
    auto base = [&](int q) { return G + ((int64_t)(q % K) * CB + q / K) * plane; };
    auto load = [&](const float* b, int st) {
        const int x = X0 + st / FW_RY;
        return b[(int64_t)((x % n0 + n0) % n0) * row + oy[st % FW_RY]];
    };
    const float* b0 = base(0);
#pragma unroll
    for (int st = 0; st < FW_STEPS; ++st) a[st] = load(b0, st);
    double2 y[2] = {make_double2(0.0, 0.0), make_double2(0.0, 0.0)};
    int k = 0, cb = 0;
    for (int q = 0; q < ng; ++q) {
        const float* nb = base(q + 1 < ng ? q + 1 : q);
        float2 u;
        if (u_real) u = make_float2(reinterpret_cast<const float*>(U)[t + (int64_t)k * nt], 0.f);
        else u = reinterpret_cast<const float2*>(U)[t + (int64_t)k * nt];
        f32x4 z[FW_ACC];
#pragma unroll
        for (int i = 0; i < FW_ACC; ++i) z[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int o = 0; o < FW_STEPS; ++o) {
            constexpr int quad[FW_RY] = {0, 2, 1};  // the middle columns, the largest weights, last
            const int st = o % FW_RX * FW_RY + quad[o / FW_RX];
            f32x4& zi = z[st / FW_RY % FW_ACC];
            zi = __builtin_amdgcn_mfma_f32_16x16x4f32(a[st], wx[st / FW_RY] * wy[st % FW_RY], zi, 0, 0, 0);
            a[st] = load(nb, st);
        }
        const f32x4 zs = (z[0] + z[1]) + (z[2] + z[3]);
        cfma(y[0], cto<double2>(u), make_double2(zs[0], zs[1]));
        cfma(y[1], cto<double2>(u), make_double2(zs[2], zs[3]));
        if (++k == K) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int c = cb * PLANE_COIL_GROUP + 2 * s + h;
                if (on && c < C) out[idx + (int64_t)c * nsel] = cto<float2>(y[h]);
                y[h] = make_double2(0.0, 0.0);
            }
            k = 0;
            ++cb;
        }
    }
}

// Whether the batches can pay, which decides if they are made at all: from 4
// coils on (the grid is stored for whole groups of 8), for grids that the fused
// placement takes, and for sample counts whose batches, 64 threads each, stay
// below the 2^32 threads of a launch.
static bool fwd_batches_possible(const msr_traj* traj, const int64_t* nos, int C) {
    return C >= 4 && nos[0] <= 1024 && nos[1] <= 1024 && traj->M > 0 && traj->M <= (int64_t)1 << 29;
}

// Whether they do pay: a batch costs the same however many samples it
// holds, 0.43 ns per coefficient and 8 coils at full rate against 0.27 ns per
// sample, coefficient and 4 coils of the one-wavefront-per-sample kernel
// (measured 3.43 ms at 512 000 samples, 20 coils, K = 5).
static bool fwd_batches_pay(int64_t nbatch, int64_t M, int C) {
    return 8 * nbatch * ceil_div(C, 8) <= 5 * M * ceil_div(C, 4);
}

constexpr size_t FW_WORK = (size_t)6 << 30;  // grids of a chunk of coils (interp_kernel)

// Device copy of the coil maps, packed (C, V): one launch per 32 coils.
constexpr int FW_MAPS = 32;
struct FwdMaps {
    const float2* p[FW_MAPS];
};
__global__ void pack_maps_kernel(FwdMaps m, int64_t V, float2* __restrict__ out) {
    const float2* src = m.p[blockIdx.y];
    for (int64_t v = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; v < V; v += (int64_t)gridDim.x * blockDim.x)
        out[(int64_t)blockIdx.y * V + v] = src[v];
}

void forward_model(msr_ctx* ctx, const msr_traj* traj, int d, const int64_t* N, const void* x,
                   int K, const void* U, int u_real, int ncoils, const void* const* cmaps, void* out,
                   hipStream_t st) {
    MSR_REQUIRE(!traj->integer, MSR_ERR_ARGUMENT, "the forward model takes a non-Cartesian trajectory");
    MSR_REQUIRE(traj->d == d, MSR_ERR_ARGUMENT, "trajectory has %d dimensions, image %d", traj->d, d);
    MSR_REQUIRE(K >= 1, MSR_ERR_ARGUMENT, "K = %d", K);
    MSR_REQUIRE(U != nullptr || K == traj->nt, MSR_ERR_ARGUMENT,
                "U = I(Nt) needs K = Nt (%lld), got %d", (long long)traj->nt, K);
    const int C = ncoils >= 1 ? ncoils : 1;
    int64_t nos[3] = {1, 1, 1}, NN[3] = {1, 1, 1}, V = 1, Gos = 1;
    for (int a = 0; a < d; ++a) {
        NN[a] = N[a];
        nos[a] = 2 * N[a];
        MSR_REQUIRE(N[a] >= 1 && fft_len_supported(nos[a]), MSR_ERR_UNSUPPORTED,
                    "forward-model grid 2N[%d] = %lld has no FFT kernel in this build", a,
                    (long long)nos[a]);
        V *= N[a];
        Gos *= nos[a];
    }
    const FwdGeom g{{nos[0], nos[1], nos[2]}};
    const FwdPlan* plan = nullptr;
    if (d == 2 && U && fwd_batches_possible(traj, nos, C)) {
        plan = &fwd_plan(traj, g, st);
        if (!fwd_batches_pay(plan->nbatch, traj->M, C)) plan = nullptr;
    }
    const int CB = (int)ceil_div(C, PLANE_COIL_GROUP);
    const bool maps = ncoils >= 1 && cmaps;
    const size_t mb = maps ? (sizeof(float2) * (size_t)C * V + 255) / 256 * 256 : 0;
    // workspace: coil maps, then S_c x_k and two grid buffers, or (matrix
    // cores) the row transforms and the grid in groups of 8 coils.  The call's
    // own, from the idle blocks: calls on one trajectory run side by side, and
    // nothing stays with the handle.  One wavefront per sample takes a multiple of
    // its groups' coils at a time, within FW_WORK bytes of grids, which the idle
    // blocks can hold (128 x 128 x 128, 16 coils, K = 4: 18 GB at once, mapped for
    // every call, took 20.3 ms, 4.6 GB in four chunks 19.6)
    const size_t coil = sizeof(float2) * (size_t)K * (V + 2 * Gos);
    const int Cw = plan ? C : (int)std::min<int64_t>(C, std::max<int64_t>(1, FW_WORK / coil / FW_CB) * FW_CB);
    const size_t zb = plan ? 0 : sizeof(float2) * (size_t)Cw * K * V;
    const size_t ab = plan ? (sizeof(float2) * (size_t)C * K * nos[0] * NN[1] + 255) / 256 * 256
                           : sizeof(float2) * (size_t)Cw * K * Gos;
    const size_t bb = plan ? sizeof(float2) * (size_t)K * CB * PLANE_COIL_GROUP * Gos : ab;
    TempBuf work{st};
    work.alloc(mb + zb + ab + bb);
    float2* mp = maps ? work.as<float2>() : nullptr;
    float2* Z = reinterpret_cast<float2*>(work.as<char>() + mb);
    float2* A = reinterpret_cast<float2*>(work.as<char>() + mb + zb);
    float2* B = reinterpret_cast<float2*>(work.as<char>() + mb + zb + ab);
    if (maps)
        for (int c0 = 0; c0 < C; c0 += FW_MAPS) {
            FwdMaps m{};
            const int nc = std::min(FW_MAPS, C - c0);
            for (int c = 0; c < nc; ++c) {
                MSR_REQUIRE(cmaps[c0 + c] != nullptr, MSR_ERR_ARGUMENT, "cmaps[%d] is NULL", c0 + c);
                m.p[c] = (const float2*)cmaps[c0 + c];
            }
            hipLaunchKernelGGL(pack_maps_kernel, dim3((unsigned)std::min<int64_t>((V + 255) / 256, 1024), nc),
                               dim3(256), 0, st, m, V, mp + (int64_t)c0 * V);
            MSR_CHECK_LAUNCH();
        }
    const int64_t nsel = traj->nsamp * traj->nt;
    if (traj->sel.p) fill_floats(out, 2 * nsel * C, 0.f, st);  // masked-out samples are 0
    if (plan) {
        PlanePass px;
        px.nf = (int)nos[0];
        px.len = (int)NN[0];
        px.K = K;
        px.nc = C;
        px.T = A;
        px.plane = nos[0] * NN[1];
        px.nrows = NN[1];
        px.b = x;
        px.cmaps = mp;
        px.win = deapod_table(ctx, (int)nos[0], (int)NN[0], SEL_CENTER);
        run_plane(PLANE_PLACE, px, ctx, st);
        PlanePass py = px;
        py.nf = (int)nos[1];
        py.len = (int)NN[1];
        py.ncols = nos[0];
        py.out = B;
        py.win = deapod_table(ctx, (int)nos[1], (int)NN[1], SEL_CENTER);
        run_plane(PLANE_COILS, py, ctx, st);
        hipLaunchKernelGGL(interp_mfma_kernel, dim3((plan->nbatch + 3) / 4), dim3(256), 0, st,
                           traj->kc.as<float>(), traj->frame.as<int>(),
                           traj->sel.p ? traj->sel.as<int64_t>() : nullptr, plan->perm.as<int>(),
                           plan->batches.as<int4>(), plan->nbatch, plan->nry, nsel,
                           reinterpret_cast<const float*>(B), g, K, C, U, u_real, traj->nt, (float2*)out);
        MSR_CHECK_LAUNCH();
        MSR_HIP(hipStreamSynchronize(st));  // the workspace is freed on return
        return;
    }
    for (int c0 = 0; c0 < C; c0 += Cw) {
        const int nc = std::min(Cw, C - c0), nch = nc * K;
        float2* o = (float2*)out + (int64_t)c0 * nsel;
        int grid = (int)std::min<int64_t>(((int64_t)nch * V + 255) / 256, 16384);
        hipLaunchKernelGGL(expand_kernel, dim3(grid), dim3(256), 0, st, (const float2*)x,
                           mp ? mp + (int64_t)c0 * V : nullptr, nc, K, V, Z);
        MSR_CHECK_LAUNCH();
        // x: centred placement + deapodisation, forward FFT over 2Nx  -> A [ch][z][y][qx]
        LinePass px;
        px.in = Z;
        px.out = A;
        px.nf = (int)nos[0];
        px.dir = -1;
        px.lin = (int)NN[0];
        px.isel = SEL_CENTER;
        px.win = deapod_table(ctx, (int)nos[0], (int)NN[0], SEL_CENTER);
        px.lout = (int)nos[0];
        px.sel = SEL_FIRST;
        px.nlines = (int64_t)nch * NN[1] * NN[2];
        px.in_pitch = NN[0];
        px.out_pitch = nos[0];
        run_rows(px, ctx, st);
        // y: A [ch][z][y][qx] -> B [ch][z][qy][qx]
        LinePass py;
        py.in = A;
        py.out = B;
        py.nf = (int)nos[1];
        py.dir = -1;
        py.lin = (int)NN[1];
        py.isel = SEL_CENTER;
        py.win = deapod_table(ctx, (int)nos[1], (int)NN[1], SEL_CENTER);
        py.lout = (int)nos[1];
        py.sel = SEL_FIRST;
        py.nb = (int64_t)nch * NN[2];
        py.ncols = nos[0];
        py.in_bstride = NN[1] * nos[0];
        py.in_stride = nos[0];
        py.out_bstride = nos[1] * nos[0];
        py.out_stride = nos[0];
        run_cols(py, ctx, st);
        const float2* Gfin = B;
        if (d == 3) {
            // z: B [ch][z][qy][qx] -> A [ch][qz][qy][qx]
            LinePass pz;
            pz.in = B;
            pz.out = A;
            pz.nf = (int)nos[2];
            pz.dir = -1;
            pz.lin = (int)NN[2];
            pz.isel = SEL_CENTER;
            pz.win = deapod_table(ctx, (int)nos[2], (int)NN[2], SEL_CENTER);
            pz.lout = (int)nos[2];
            pz.sel = SEL_FIRST;
            pz.nb = nch;
            pz.ncols = nos[1] * nos[0];
            pz.in_bstride = NN[2] * nos[1] * nos[0];
            pz.in_stride = nos[1] * nos[0];
            pz.out_bstride = Gos;
            pz.out_stride = nos[1] * nos[0];
            run_cols(pz, ctx, st);
            Gfin = A;
        }
        const int64_t waves = traj->M;
        const int blocks = (int)std::min<int64_t>((waves * 64 + 255) / 256, 65536);
        if (d == 2)
            hipLaunchKernelGGL(interp_kernel<2>, dim3(blocks), dim3(256), 0, st, traj->kc.as<float>(),
                               traj->frame.as<int>(), traj->sel.p ? traj->sel.as<int64_t>() : nullptr,
                               traj->M, nsel, Gfin, g, K, nc, U, u_real, traj->nt, o);
        else
            hipLaunchKernelGGL(interp_kernel<3>, dim3(blocks), dim3(256), 0, st, traj->kc.as<float>(),
                               traj->frame.as<int>(), traj->sel.p ? traj->sel.as<int64_t>() : nullptr,
                               traj->M, nsel, Gfin, g, K, nc, U, u_real, traj->nt, o);
        MSR_CHECK_LAUNCH();
    }
    MSR_HIP(hipStreamSynchronize(st));  // the workspace is freed on return
}

}  // namespace msr
