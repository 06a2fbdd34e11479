// Spreading half of the kernel construction: the basis pair products of every
// sample gathered onto the sigma = 2 grid in FP64 on the matrix cores (see
// kernel_spread.hip).
#pragma once

#include "spread.hpp"

namespace msr {

// Samples of a trajectory sorted by bins of 4 cells per dimension of the grid
// n, with their kernel weights; lives for one kernel construction.
struct KernelSpread {
    int d = 2;
    int n[3] = {1, 1, 1}, nb[3] = {1, 1, 1};
    int64_t M = 0;
    TempBuf cells;  // (M) int4: floor cell per dimension, frame
    TempBuf wts;    // (M, d, 8) double: ES weights of the cells c - 3 .. c + 4
    TempBuf first;  // (bins + 1) int32: first sorted sample of a bin
    TempBuf vals;   // pair products per frame (basis values only)
    bool built = false;
    explicit KernelSpread(hipStream_t st) : cells(st), wts(st), first(st), vals(st) {}
    // Once; again does nothing, unless an allocation failed.
    void build(const msr_traj* traj, const int64_t* grid, hipStream_t st);
    void release();  // the tables
    // Room for the values of up to np channels of src.
    void reserve(const ValueSrc& src, int np);
    // grid (np, prod n) ComplexF64, overwritten: channel p = sum over samples of
    // conj(U[t, pair_j]) U[t, pair_k] times the weights (src.kind 1); real
    // values for a real basis
    void run(const ValueSrc& src, int np, double2* grid, hipStream_t st);
};

// Grids of at least 12 cells (three bins) per dimension, in multiples of 4.
bool kernel_spread_supported(int d, const int64_t* n);

}  // namespace msr
