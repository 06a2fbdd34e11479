// FP64 spreading of the kernel construction, output-owned.  Each wavefront owns
// 16 cells (4 x 4, a plane of 4 x 4 x 4 in 3D) and sums the samples whose W = 8
// support can reach them: those of the 3 x 3 (x 3) bins of 4 cells around,
// which are 3 (9) runs of the sorted samples, or twice as many at the grid's
// edge.  The sums are the product of the samples' values (rows: real and
// imaginary parts of the pair products, 16 per tile) and weights (columns: the
// 16 cells), four samples per v_mfma_f64_16x16x4f64:
//   lane (r = lane mod 16, g = lane div 16): A = value row r, B = weight of cell
//   r, both of sample 4 step + g; D element e = row g + 4 e of cell r.
// Rows are ordered so that a lane's four are the two parts of two channels.  The
// values depend on the frame alone and come from a table (cache-resident);
// weights were evaluated once per sample.  Every cell sums its samples in
// sorted order, so the result is bit-reproducible, and every cell is written,
// so the grid needs no clearing and no second pass.
//
// Bound: matrix-core issue (64 cycles per 4 samples, tile of rows and cells;
// 9 (27) visits per sample) and the latency of the chain from sample to weight.
// On MI355X, before (tiles of 32 x 32 or 16 x 8 x 8 cells in LDS, then a gather over
// the padded tiles) and after: 256 x 256, K = 5 (15 pairs), 512 000 samples
// 4.60 -> 0.60 ms; 80 x 72 x 64, K = 4 real, 320 000 samples 17.7 -> 3.0 ms (all 10
// pairs in one row tile); taking only the samples that reach the wave's plane gave 2.54
// ms per launch after 3.47 (2D: 0.60 after 0.64).
#include "kernel_spread.hpp"

#include "blockgrid.hpp"

#include <hipcub/hipcub.hpp>

#include <algorithm>

namespace msr {

using f64x4 = __attribute__((__vector_size__(4 * sizeof(double)))) double;

struct KernelGeom {
    int n[3], nb[3];
};

__device__ __forceinline__ int floor_cell(float k, int n, double& frac) {
    const double s = (double)k * (double)n;
    const double fl = floor(s);
    frac = s - fl;
    int64_t c = (int64_t)fl % n;
    return (int)(c < 0 ? c + n : c);
}

__global__ void kspread_key_kernel(const float* __restrict__ kc, int d, int64_t M, KernelGeom g,
                                   int* __restrict__ key, int* __restrict__ idx) {
    for (int64_t j = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; j < M;
         j += (int64_t)gridDim.x * blockDim.x) {
        int b = 0;
        for (int a = d - 1; a >= 0; --a) {
            double f;
            b = b * g.nb[a] + floor_cell(kc[j * d + a], g.n[a], f) / 4;
        }
        key[j] = b;
        idx[j] = (int)j;
    }
}

// one thread per (sorted sample, dimension, weight)
template <int D>
__global__ void kspread_points_kernel(const float* __restrict__ kc, const int* __restrict__ frame,
                                      const int* __restrict__ perm, int64_t M, KernelGeom g,
                                      int4* __restrict__ cells, double* __restrict__ wts) {
    const int64_t total = M * D * 8;
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total;
         e += (int64_t)gridDim.x * blockDim.x) {
        const int64_t s = e / (D * 8);
        const int r = (int)(e - s * (D * 8)), a = r >> 3, o = r & 7;
        const int64_t j = perm[s];
        double f;
        const int c = floor_cell(kc[j * D + a], g.n[a], f);
        const double z = ((double)(o - 3) - f) * (2.0 / SPREAD_W);
        const double q = 1.0 - z * z;
        wts[e] = q > 0.0 ? exp((double)SPREAD_BETA * (sqrt(q) - 1.0)) : 0.0;
        int* out = reinterpret_cast<int*>(cells + s);
        if (o == 0) out[a] = c;
        if (r == 0) {
            if (D == 2) out[2] = 0;
            out[3] = frame[j];
        }
    }
}

// vals[(t T + tile) 16 + i]: row i of a tile of 8 complex (16 real) channels:
// channel (i / 8) 4 + i mod 4, part (i / 4) mod 2; a real basis: channel i
__global__ void kspread_values_kernel(ValueSrc src, int np, int tiles, double* __restrict__ vals) {
    const int64_t total = src.nt * tiles * 16;
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total;
         e += (int64_t)gridDim.x * blockDim.x) {
        const int i = (int)(e & 15), tile = (int)((e >> 4) % tiles);
        const int64_t t = (e >> 4) / tiles;
        const int ch = src.u_real ? tile * 16 + i : tile * 8 + (i / 8) * 4 + i % 4;
        double v = 0.0;
        if (ch < np) {
            const int64_t a = t + src.pair_j[ch] * src.nt, b = t + src.pair_k[ch] * src.nt;
            if (src.u_real) {
                const float* U = reinterpret_cast<const float*>(src.U);
                v = (double)U[a] * (double)U[b];
            } else {
                const float2* U = reinterpret_cast<const float2*>(src.U);
                const double2 p = cmulc(cto<double2>(U[a]), cto<double2>(U[b]));  // conj(U_j) U_k
                v = (i / 4) % 2 ? p.y : p.x;
            }
        }
        vals[e] = v;
    }
}

// blockIdx.z: group of MT row tiles; blocks are counted over x and y (split_blocks)
template <int D, int MT, bool REAL>
__global__ void __launch_bounds__(256)
kspread_gather_kernel(const int4* __restrict__ cells, const double* __restrict__ wts,
                      const int* __restrict__ first, const double* __restrict__ vals, int tiles, KernelGeom g,
                      int np, double2* __restrict__ grid) {
    constexpr int NR = D == 2 ? 6 : 18;  // runs of sorted samples, two per bin row
    __shared__ int4 s_pt[4][72];         // {sample, offsets dx, dy dz, frame}: up to 7 left over and a chunk
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int r = lane & 15, q4 = lane >> 4, lx = r & 3, ly = r >> 2;
    // neighbouring tiles on one XCD
    const int64_t nblk = (int64_t)gridDim.x * gridDim.y, b = (int64_t)blockIdx.y * gridDim.x + blockIdx.x;
    int64_t lb = nblk % 8 ? b : (b % 8) * (nblk / 8) + b / 8;
    if (D == 2) lb = lb * 4 + wave;
    const int nbx = g.nb[0], nby = g.nb[1], nbz = D == 3 ? g.nb[2] : 1;
    if (lb >= (int64_t)nbx * nby * nbz) return;  // (a wave without a tile; waves never synchronise)
    const int tx = (int)(lb % nbx), ty = (int)(lb / nbx % nby), tz = (int)(lb / ((int64_t)nbx * nby));
    const int X = 4 * tx, Y = 4 * ty, Z = D == 3 ? 4 * tz + wave : 0;
    // the runs: bins tx - 1 .. tx + 1 of each bin row, cut where x wraps
    const int a0 = tx == 0 ? nbx - 1 : tx - 1, a1 = tx == 0 ? nbx - 1 : (tx == nbx - 1 ? tx : tx + 1);
    const int b0 = tx == nbx - 1 ? 0 : (tx == 0 ? 0 : 1), b1 = tx == nbx - 1 ? 0 : (tx == 0 ? 1 : 0);
    int start[NR], pre[NR], total = 0;
#pragma unroll
    for (int i = 0; i < NR / 2; ++i) {
        const int y = (ty + i % 3 - 1 + nby) % nby, z = D == 3 ? (tz + i / 3 - 1 + nbz) % nbz : 0;
        const int row = (z * nby + y) * nbx;
        start[2 * i] = first[row + a0];
        pre[2 * i] = total;
        total += first[row + a1 + 1] - start[2 * i];
        start[2 * i + 1] = first[row + b0];
        pre[2 * i + 1] = total;
        if (b1 >= b0) total += first[row + b1 + 1] - start[2 * i + 1];
    }
    const int mt0 = blockIdx.z * MT;
    f64x4 acc[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[m] = f64x4{0.0, 0.0, 0.0, 0.0};
    // samples left over from the chunk before, at the front of s_pt
    int left = 0;
    for (int p0 = 0; p0 < total; p0 += 64) {
        const int p = min(p0 + lane, total - 1);
        int s = 0;
#pragma unroll
        for (int i = 0; i < NR; ++i)
            if (p >= pre[i]) s = start[i] + p - pre[i];
        const int4 c = cells[s];
        // first cell of the tile relative to the sample's first, in -4 .. 7
        int dx = X - c.x + 3, dy = Y - c.y + 3, dz = D == 3 ? Z - c.z + 3 : 0;
        dx += dx < -4 ? g.n[0] : 0;
        dx -= dx > 7 ? g.n[0] : 0;
        dy += dy < -4 ? g.n[1] : 0;
        dy -= dy > 7 ? g.n[1] : 0;
        if (D == 3) {
            dz += dz < -4 ? g.n[2] : 0;
            dz -= dz > 7 ? g.n[2] : 0;
        }
        // keep the samples whose support meets the tile, 121 of 144 cells of
        // the bins around (3D: the plane, 968 of 1728), in their order
        const bool reach = p0 + lane < total && dx > -4 && dy > -4 && (D == 2 || (unsigned)dz <= 7u);
        const uint64_t kept = __ballot(reach);
        const int at = left + __builtin_amdgcn_mbcnt_hi((unsigned)(kept >> 32),
                                                        __builtin_amdgcn_mbcnt_lo((unsigned)kept, 0u));
        if (reach) s_pt[wave][at] = make_int4(s, dx, (dy & 0xFFFF) | (dz << 16), c.w);
        left += __popcll(kept);
        int use = left & ~7;
        if (p0 + 64 >= total) {  // the last chunk: fill up with samples of no weight (offset 8)
            use = (left + 7) & ~7;
            if (lane < use - left) s_pt[wave][left + lane] = make_int4(s, 8, 0, c.w);
            left = use;
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        for (int q = 0; q < use; q += 8) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int4 e = s_pt[wave][q + 4 * h + q4];
                const int ox = e.y + lx, oy = (int)(short)(e.z & 0xFFFF) + ly, oz = e.z >> 16;
                const double* w = wts + (int64_t)e.x * (D * 8);
                double b = w[ox & 7] * w[8 + (oy & 7)];
                if (D == 3) b *= w[D * 8 - 8 + (oz & 7)];
                if ((unsigned)ox > 7u || (unsigned)oy > 7u) b = 0.0;
                const double* v = vals + ((int64_t)e.w * tiles + mt0) * 16 + r;
#pragma unroll
                for (int m = 0; m < MT; ++m)
                    acc[m] = __builtin_amdgcn_mfma_f64_16x16x4f64(v[m * 16], b, acc[m], 0, 0, 0);
            }
        }
        left -= use;
        int4 e = make_int4(0, 8, 0, 0);
        if (lane < left) e = s_pt[wave][use + lane];
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        if (lane < left) s_pt[wave][lane] = e;
    }
    const int64_t G = (int64_t)g.n[0] * g.n[1] * (D == 3 ? g.n[2] : 1);
    double2* dst = grid + ((int64_t)Z * g.n[1] + Y + ly) * g.n[0] + X + lx;
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        if constexpr (REAL) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int ch = (mt0 + m) * 16 + q4 + 4 * e;
                if (ch < np) dst[ch * G] = make_double2(acc[m][e], 0.0);
            }
        } else {
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const int ch = (mt0 + m) * 8 + 4 * e + q4;
                if (ch < np) dst[ch * G] = make_double2(acc[m][2 * e], acc[m][2 * e + 1]);
            }
        }
    }
}

bool kernel_spread_supported(int d, const int64_t* n) {
    for (int a = 0; a < d; ++a)
        if (n[a] < 12 || n[a] % 4) return false;
    return true;
}

static KernelGeom geom_of(const KernelSpread& k) {
    KernelGeom g;
    for (int a = 0; a < 3; ++a) {
        g.n[a] = k.n[a];
        g.nb[a] = k.nb[a];
    }
    return g;
}

void KernelSpread::build(const msr_traj* traj, const int64_t* grid_n, hipStream_t st) {
    if (built) return;
    d = traj->d;
    M = traj->M;
    MSR_REQUIRE(M < (int64_t)INT32_MAX, MSR_ERR_UNSUPPORTED, "more than 2^31 samples");
    int64_t nbins = 1;
    for (int a = 0; a < d; ++a) {
        n[a] = (int)grid_n[a];
        nb[a] = n[a] / 4;
        nbins *= nb[a];
    }
    MSR_REQUIRE(nbins < (int64_t)INT32_MAX, MSR_ERR_UNSUPPORTED, "grid too large");
    const KernelGeom g = geom_of(*this);
    TempBuf keys{st}, sorted{st}, idx{st}, perm{st}, temp{st};
    keys.alloc(sizeof(int) * M);
    sorted.alloc(sizeof(int) * M);
    idx.alloc(sizeof(int) * M);
    perm.alloc(sizeof(int) * M);
    cells.alloc(sizeof(int4) * M);
    wts.alloc(sizeof(double) * 8 * d * M);
    first.alloc(sizeof(int) * (nbins + 1));
    const int gr = (int)std::min<int64_t>((M + 255) / 256, 8192);
    hipLaunchKernelGGL(kspread_key_kernel, dim3(gr), dim3(256), 0, st, traj->kc.as<float>(), d, M, g,
                       keys.as<int>(), idx.as<int>());
    MSR_CHECK_LAUNCH();
    int bits = 1;
    while ((int64_t(1) << bits) < nbins) ++bits;
    size_t tb = 0;
    MSR_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, tb, keys.as<int>(), sorted.as<int>(), idx.as<int>(),
                                               perm.as<int>(), (int)M, 0, bits, st));
    temp.alloc(std::max<size_t>(tb, 16));
    MSR_HIP(hipcub::DeviceRadixSort::SortPairs(temp.p, tb, keys.as<int>(), sorted.as<int>(), idx.as<int>(),
                                               perm.as<int>(), (int)M, 0, bits, st));
    sorted_first(sorted.as<int>(), M, nbins, first.as<int>(), st);
    const int gw = (int)std::min<int64_t>((M * d * 8 + 255) / 256, 32768);
    if (d == 2)
        hipLaunchKernelGGL(kspread_points_kernel<2>, dim3(gw), dim3(256), 0, st, traj->kc.as<float>(),
                           traj->frame.as<int>(), perm.as<int>(), M, g, cells.as<int4>(), wts.as<double>());
    else
        hipLaunchKernelGGL(kspread_points_kernel<3>, dim3(gw), dim3(256), 0, st, traj->kc.as<float>(),
                           traj->frame.as<int>(), perm.as<int>(), M, g, cells.as<int4>(), wts.as<double>());
    MSR_CHECK_LAUNCH();
    MSR_HIP(hipStreamSynchronize(st));  // temporaries are freed on return
    built = true;
}

void KernelSpread::release() {
    for (DevBuf* b : {&cells, &wts, &first, &vals}) b->release();
    built = false;
}

// Row tiles of np channels: MT per wave, in groups.
struct KernelTiles {
    int mt, groups;
};
static KernelTiles tiles_of(const ValueSrc& src, int np) {
    const int tiles = (int)ceil_div(np, src.u_real ? 16 : 8);
    const int mt = tiles == 1 ? 1 : (tiles == 2 ? 2 : 4);
    return {mt, (int)ceil_div(tiles, mt)};
}

void KernelSpread::reserve(const ValueSrc& src, int np) {
    const KernelTiles t = tiles_of(src, np);
    const size_t vb = sizeof(double) * 16 * (size_t)src.nt * t.groups * t.mt;
    if (vals.bytes < vb) vals.alloc(vb);
}

void KernelSpread::run(const ValueSrc& src, int np, double2* grid, hipStream_t st) {
    MSR_REQUIRE(src.kind == 1 && src.U, MSR_ERR_ERROR, "the kernel's spreading takes basis pair products");
    const KernelGeom g = geom_of(*this);
    const auto [mt, groups] = tiles_of(src, np);
    const int tiles = groups * mt;
    reserve(src, np);
    const int gv = (int)std::min<int64_t>((src.nt * tiles * 16 + 255) / 256, 4096);
    hipLaunchKernelGGL(kspread_values_kernel, dim3(gv), dim3(256), 0, st, src, np, tiles, vals.as<double>());
    MSR_CHECK_LAUNCH();
    const int64_t nblk = d == 2 ? ceil_div((int64_t)nb[0] * nb[1], 4) : (int64_t)nb[0] * nb[1] * nb[2];
    const BlockGrid xy = split_blocks(nblk, 256);
    const dim3 gr(xy.x, xy.y, (unsigned)groups);
#define MSR_KGATHER(DD, MM, RR)                                                                           \
    hipLaunchKernelGGL((kspread_gather_kernel<DD, MM, RR>), gr, dim3(256), 0, st, cells.as<int4>(),       \
                       wts.as<double>(), first.as<int>(), vals.as<double>(), tiles, g, np, grid)
#define MSR_KGATHER_M(DD, RR)              \
    if (mt == 1) MSR_KGATHER(DD, 1, RR);   \
    else if (mt == 2) MSR_KGATHER(DD, 2, RR); \
    else MSR_KGATHER(DD, 4, RR)
    if (d == 2) {
        if (src.u_real) { MSR_KGATHER_M(2, true); }
        else { MSR_KGATHER_M(2, false); }
    } else {
        if (src.u_real) { MSR_KGATHER_M(3, true); }
        else { MSR_KGATHER_M(3, false); }
    }
#undef MSR_KGATHER_M
#undef MSR_KGATHER
    MSR_CHECK_LAUNCH();
}

}  // namespace msr
