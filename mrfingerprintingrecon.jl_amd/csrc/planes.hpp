// Normal-operator apply in fused line passes for every line-FFT length and
// K <= 8 (the shapes outside the fused Toeplitz passes, and the Cartesian
// operator), in 2D and 3D, with or without zero padding:
//   expand    rows x of S_c b_k, FFT along x                          -> T
//   (3D: y columns forward, LinePass)
//   multiply  the last axis: FFT, per-cell K x K kernel, inverse FFT, crop
//   (3D: y columns inverse, LinePass)
//   combine   inverse FFT along x, crop, sum over coils of conj(S_c) img
// so that no zero-padded last axis and no separate multiply, expansion or
// coil sum passes through memory.  T is addressed by strides: 2D
// T[c][k][qx][y] (y fastest, so that the multiply's lines are contiguous), 3D
// T[c][k][z][y][qx].
//
// Bound: the expand and combine passes stream T once; the multiply reads and
// writes it once and works in LDS.  On MI355X, ComplexF64, before (separate
// expand, line, multiply and combine passes) and after:
//   240 x 300, 12 coils, K = 6, real kernel: 1.96 -> 0.40 ms (expand 51, multiply 228, combine 91 us)
//   Cartesian 256 x 256, 20 coils, K = 5:    0.252 -> 0.143 ms (expand 30, multiply 72, combine 40 us)
#pragma once

#include "internal.hpp"

namespace msr {

enum { PLANE_EXPAND = 0, PLANE_MULTIPLY = 1, PLANE_COMBINE = 2, PLANE_PLACE = 3, PLANE_COILS = 4 };

struct PlanePass {
    int f64 = 0;
    int nf = 0;                    // FFT length of the pass
    int len = 0;                   // stored elements of the line: inputs (expand), kept
                                   // outputs (combine), both (multiply); the rest is padding
    int K = 1;
    int nc = 1, G = 1;             // coils of this launch; groups the combine sums them in
    void* T = nullptr;
    int64_t plane = 0;             // elements of T per (coil, coefficient)
    // rows (expand, combine): row r, bin q of a plane at r * rs + q * qs
    int64_t nrows = 0, rs = 0, qs = 0;
    const void* b = nullptr;       // (K, nrows, len)
    void* partial = nullptr;       // (G, K, nrows, len)
    int accumulate = 0;            // add to partial instead of overwriting it
    const float2* cmaps = nullptr; // of the launch's first coil, (nc, nrows, len), or none
    // columns (multiply): column col, element i of a plane at col * cs + i * es
    int64_t ncols = 0, cs = 0, es = 0;
    const void* lam = nullptr;     // lam[(col * P + p) * nf + i]
    int lam_real = 0, lam_full = 0;// Float32; P = K * K entries j + K k (else packed Hermitian)
    // forward model (ComplexF32): rows placed around frequency zero and scaled
    // (place), then lines along y of PLANE_COIL_GROUP coils at a time (coils):
    // T[(k nc + c) plane + q nrows + row] -> out[((k CB + c / 8) ncols + col) nf + q][c % 8]
    const float* win = nullptr;    // deapodisation of the stored elements
    float2* out = nullptr;
    const int* skip = nullptr;
};

constexpr int PLANE_COIL_GROUP = 8;  // coils side by side: 64 bytes of a cell

// Place and coils passes cover nf <= 1024 on both axes.
// Launches one pass (twiddles from the context's tables).
void run_plane(int which, const PlanePass& p, msr_ctx* ctx, hipStream_t st);

// True when the three passes take the shape: image size N, nf = pad * N per
// axis, K coefficients.
bool planes_supported(int d, const int64_t* N, int pad, int K);

// The passes of an operator with op->planes over its coils [c_begin, c_end):
// partial[g] gets the unscaled sums of G coil groups.
void launch_planes_passes(msr_normalop* op, const void* b, bool f64, hipStream_t st, const int* skip,
                          int c_begin, int c_end, int G);

bool plane_part0(int which, const PlanePass& p, const void* tw, hipStream_t st);
bool plane_part1(int which, const PlanePass& p, const void* tw, hipStream_t st);
bool plane_part2(int which, const PlanePass& p, const void* tw, hipStream_t st);
bool plane_part3(int which, const PlanePass& p, const void* tw, hipStream_t st);
bool plane_part4(int which, const PlanePass& p, const void* tw, hipStream_t st);
bool plane_part5(int which, const PlanePass& p, const void* tw, hipStream_t st);

}  // namespace msr
