// Dispatch of the fused line passes (see planes.hpp) to the translation units
// that instantiate each length (planes_p*.hip).
#include "planes.hpp"

#include <algorithm>

#include "fft.hpp"
#include "fftlines.hpp"
#include "normalop.hpp"

namespace msr {

using PlanePartFn = bool (*)(int, const PlanePass&, const void*, hipStream_t);
static const PlanePartFn kPlaneParts[MSR_FFT_LINE_PARTS] = {
    plane_part0, plane_part1, plane_part2, plane_part3, plane_part4, plane_part5};

void run_plane(int which, const PlanePass& p, msr_ctx* ctx, hipStream_t st) {
    const void* tw = p.f64 ? (const void*)twiddle_table64(ctx, p.nf) : (const void*)twiddle_table(ctx, p.nf);
    for (PlanePartFn f : kPlaneParts)
        if (f(which, p, tw, st)) {
            MSR_CHECK_LAUNCH();
            return;
        }
    fail(MSR_ERR_UNSUPPORTED, "no FFT kernel for length %d", p.nf);
}

bool planes_supported(int d, const int64_t* N, int pad, int K) {
    const int64_t last = pad * N[d - 1];
    // one column's K lines in ComplexF64 (padded by an eighth, or rounded up to
    // a multiple of 16) within the 160 KiB of LDS and, at 8 values per thread,
    // 1024 threads; rows up to 1024 points; K in the multiply's registers
    return K <= 8 && pad * N[0] <= 1024 && K * last <= 8192 &&
           (size_t)K * ((size_t)last + last / 8 + 16) * sizeof(double2) <= (size_t)160 * 1024;
}

void launch_planes_passes(msr_normalop* op, const void* b, bool f64, hipStream_t st, const int* skip,
                          int c_begin, int c_end, int G) {
    MSR_REQUIRE(0 <= c_begin && c_begin < c_end && c_end <= op->C && 1 <= G && G <= op->G, MSR_ERR_ERROR,
                "coils [%d, %d) of %d in %d groups", c_begin, c_end, op->C, G);
    const int d = op->d, K = op->K, pad = op->cart ? 1 : 2;
    const int64_t nx = op->N[0], ny = op->N[1], nz = d == 3 ? op->N[2] : 1;
    const int64_t fx = pad * nx, fy = pad * ny;
    const size_t es = f64 ? sizeof(double2) : sizeof(float2);
    MSR_REQUIRE(op->T.bytes >= es * general_scratch(op, 0) && op->T2.bytes >= es * general_scratch(op, 1),
                MSR_ERR_ERROR, "apply scratch not allocated for this precision");
    PlanePass row;
    row.f64 = f64 ? 1 : 0;
    row.nf = (int)fx;
    row.len = (int)nx;
    row.K = K;
    row.T = op->T.p;
    row.plane = fx * ny * nz;
    row.nrows = ny * nz;
    row.rs = d == 2 ? 1 : fx;
    row.qs = d == 2 ? ny : 1;
    row.skip = skip;
    PlanePass mul = row;
    mul.nf = (int)(pad * op->N[d - 1]);
    mul.len = (int)op->N[d - 1];
    mul.ncols = d == 2 ? fx : fx * fy;
    mul.cs = d == 2 ? ny : 1;
    mul.es = d == 2 ? 1 : fx * fy;
    mul.lam = op->lam->p;
    mul.lam_real = op->lam_real;
    mul.lam_full = op->cart;
    if (d == 3) {
        mul.T = op->T2.p;
        mul.plane = fx * fy * nz;
    }
    for (int c0 = c_begin; c0 < c_end; c0 += op->Cb) {
        const int nc = std::min(op->Cb, c_end - c0);
        row.nc = mul.nc = nc;
        row.cmaps = op->identity_cmaps ? nullptr : op->cmaps.as<float2>() + (size_t)c0 * op->V;
        PlanePass ex = row;
        ex.b = b;
        run_plane(PLANE_EXPAND, ex, op->ctx, st);
        LinePass y;  // 3D: T [ck][z][y][qx] -> T2 [ck][z][qy][qx] and back
        y.f64 = row.f64;
        y.nf = (int)fy;
        y.nb = (int64_t)nc * K * nz;
        y.ncols = fx;
        y.in_stride = y.out_stride = fx;
        y.skip = skip;
        if (d == 3) {
            y.in = op->T.p;
            y.out = op->T2.p;
            y.dir = -1;
            y.lin = (int)ny;
            y.lout = (int)fy;
            y.in_bstride = ny * fx;
            y.out_bstride = fy * fx;
            run_cols(y, op->ctx, st);
        }
        run_plane(PLANE_MULTIPLY, mul, op->ctx, st);
        if (d == 3) {
            y.in = op->T2.p;
            y.out = op->T.p;
            y.dir = +1;
            y.lin = (int)fy;
            y.lout = (int)ny;
            y.in_bstride = fy * fx;
            y.out_bstride = ny * fx;
            run_cols(y, op->ctx, st);
        }
        PlanePass co = row;
        co.G = G;
        co.partial = op->partial.p;
        co.accumulate = c0 > c_begin ? 1 : 0;
        run_plane(PLANE_COMBINE, co, op->ctx, st);
    }
}

}  // namespace msr
