// pair.hpp -- the reference's per-element arithmetic of every pair primitive,
// shared by the one-primitive sweeps (sweep.hip) and the resident-row program
// (rows.hip).  Compiled without FMA contraction, so results match the
// reference CPU path exactly.
#pragma once
#pragma clang fp contract(off)

#include <hip/hip_runtime.h>

#include "prim.hpp"

namespace dmx {

constexpr double kS2I = 0.70710678118654752440;  // src/config.hpp:57

// Output for the pos0 (SEL = 0) or pos1 (SEL = 1) entry of a pair
// (a0 + i b0, a1 + i b1); expressions as in src/dmsim_amdgpu_omp.hpp:1019-1480.
template <int K>
__host__ __device__ __forceinline__ void out0(const double* c, double a0, double b0, double a1, double b1,
                                     double& yr, double& yi)
{
    if constexpr (K == PK_C1) {
        yr = (c[0] * a0) - (c[1] * b0) + (c[2] * a1) - (c[3] * b1);
        yi = (c[0] * b0) + (c[1] * a0) + (c[2] * b1) + (c[3] * a1);
    } else if constexpr (K == PK_X) {
        yr = a1; yi = b1;
    } else if constexpr (K == PK_Y) {
        yr = b1; yi = -a1;
    } else if constexpr (K == PK_H) {
        yr = kS2I * (a0 + a1); yi = kS2I * (b0 + b1);
    } else if constexpr (K == PK_SRN) {
        yr = 0.5 * (a0 + a1); yi = 0.5 * (b0 - b1);
    } else if constexpr (K == PK_RX) {
        yr = (c[0] * a0) - (c[1] * b1); yi = (c[0] * b0) + (c[1] * a1);
    } else if constexpr (K == PK_RY) {
        yr = (c[0] * a0) + (c[1] * a1); yi = (c[0] * b0) + (c[1] * b1);
    } else if constexpr (K == PK_W) {
        yr = kS2I * (a0 + b1); yi = kS2I * (b0 - a1);
    } else {  // pos1-only kinds keep pos0
        yr = a0; yi = b0;
    }
}

template <int K>
__host__ __device__ __forceinline__ void out1(const double* c, double a0, double b0, double a1, double b1,
                                     double& yr, double& yi)
{
    if constexpr (K == PK_C1) {
        yr = (c[4] * a0) - (c[5] * b0) + (c[6] * a1) - (c[7] * b1);
        yi = (c[4] * b0) + (c[5] * a0) + (c[6] * b1) + (c[7] * a1);
    } else if constexpr (K == PK_X) {
        yr = a0; yi = b0;
    } else if constexpr (K == PK_Y) {
        yr = -b0; yi = a0;
    } else if constexpr (K == PK_H) {
        yr = kS2I * (a0 - a1); yi = kS2I * (b0 - b1);
    } else if constexpr (K == PK_SRN) {
        yr = 0.5 * (a0 + a1); yi = 0.5 * (-b0 + b1);
    } else if constexpr (K == PK_RX) {
        yr = -(c[1] * b0) + (c[0] * a1); yi = (c[1] * a0) + (c[0] * b1);
    } else if constexpr (K == PK_RY) {
        yr = (c[2] * a0) + (c[3] * a1); yi = (c[2] * b0) + (c[3] * b1);
    } else if constexpr (K == PK_W) {
        yr = kS2I * (b0 + a1); yi = kS2I * (-a0 + b1);
    } else if constexpr (K == PK_Z) {
        yr = -a1; yi = -b1;
    } else if constexpr (K == PK_S) {
        yr = -b1; yi = a1;
    } else if constexpr (K == PK_SDG) {
        yr = b1; yi = -a1;
    } else if constexpr (K == PK_T) {
        yr = kS2I * (a1 - b1); yi = kS2I * (a1 + b1);
    } else if constexpr (K == PK_TDG) {
        yr = kS2I * (a1 + b1); yi = kS2I * (-a1 + b1);
    } else if constexpr (K == PK_R) {
        yr = -(b1 * c[0]); yi = a1 * c[0];
    } else if constexpr (K == PK_U1) {
        yr = (c[0] * a1) - (c[1] * b1); yi = (c[0] * b1) + (c[1] * a1);
    }
}

// CJ: evaluate on conjugated operands and conjugate the result (slow index).
template <int K, bool CJ>
__host__ __device__ __forceinline__ void eval0(const double* c, double a0, double b0, double a1, double b1,
                                      double& yr, double& yi)
{
    if constexpr (CJ) { b0 = -b0; b1 = -b1; }
    out0<K>(c, a0, b0, a1, b1, yr, yi);
    if constexpr (CJ) yi = -yi;
}

template <int K, bool CJ>
__host__ __device__ __forceinline__ void eval1(const double* c, double a0, double b0, double a1, double b1,
                                      double& yr, double& yi)
{
    if constexpr (CJ) { b0 = -b0; b1 = -b1; }
    out1<K>(c, a0, b0, a1, b1, yr, yi);
    if constexpr (CJ) yi = -yi;
}

}  // namespace dmx
