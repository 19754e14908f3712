// rows.hpp -- the plain method with whole rows of rho on chip (rows.hip): the
// program a segment of gate primitives becomes, its steps' arithmetic, and
// the launcher.  The steps are host functions too, for the CPU check of the
// programs (tests/cpp/row_programs.cpp).
//
// On the column index every row of rho transforms on its own, so a workgroup
// that holds whole rows applies a segment's primitives to them one after the
// other without any other workgroup.  A thread holds 2^K entries of a row
// that differ in K "register" index bits and applies to them, in registers,
// every consecutive primitive whose target is one of those bits; a control or
// the target of a diagonal gate may be any bit, as it only selects entries.
// A regroup step then changes the register bits through LDS.
#pragma once
#pragma clang fp contract(off)

#include <hip/hip_runtime.h>

#include <cstdint>
#include <vector>

#include "pair.hpp"
#include "prim.hpp"

namespace dmx {

// A row of 2^14 entries (256 KB) is the longest that one CU holds.
constexpr int kRowsMaxQubits = 14;

// Dispatch codes of the steps (t, c: register bits).
enum : uint32_t {
    RC_END = 0,
    RC_REGROUP = 1,
    RC_SKIP = 2,                // nothing (keeps a 4x4's records in one chunk)
    RC_DENSE = 4,               // + 4 * kind + t: pair kinds that rewrite both entries
    RC_DIAG = RC_DENSE + 4 * 8, // + 8 * (kind - PK_Z) + t: diagonal kinds; t = 4: on every
                                // entry of the threads that `on` selects
    RC_CX = RC_DIAG + 8 * 7,    // + 4 * t + c: controlled swap
    RC_C2 = RC_CX + 16,         // + p: 4x4 on register bits (2p + 1, 2p); its 32 coefficients
                                // fill this record and the next three
    RC_COUNT = RC_C2 + 2
};

// A wave reads the program a chunk of 12 records (60 lanes x 16 bytes) at a time,
// one chunk ahead of the steps it runs.
constexpr int kRowChunk = 12;

struct RowOp {
    uint32_t code;
    uint32_t on;    // the step applies to threads with (tid & on) == on
    uint32_t pad[2];
    // primitives: PrimOp::c as pairs of words.  Regroup: the LDS places (XORed
    // together) of register bit i in w[i], of thread bit i in w[4 + i].
    uint32_t w[16];
};
static_assert(sizeof(RowOp) == 80, "RowOp layout");

// How n-qubit rows are dealt: a workgroup of 2^(loge - k) threads holds 2^loge
// consecutive entries of a plane (whole rows), 2^k of them per thread.
struct RowShape {
    int k, loge;
    bool split;  // entries stay in registers; regroups pass the two planes through LDS in turn
};
RowShape row_shape(int n);

// LDS place of entry x of a workgroup: every digit of s bits XORed into the
// lowest one.  A place is 16 bytes (s = 3: eight places span the banks) or, split,
// 8 bytes (s = 4); lanes that differ in s index bits with distinct residues
// mod s then fall on different banks.  Linear over XOR.
__host__ __device__ inline uint32_t row_place(uint32_t x, int s, int loge)
{
    uint32_t y = x;
    for (int sh = s; sh < loge; sh += s) y ^= (x >> sh) & ((1u << s) - 1);
    return y;
}

// Appends the program of prims [first, last) (no PK_SUP) on n <= kRowsMaxQubits
// qubits -- its steps, RC_END, and records up to three whole chunks after it
// (what a wave may read ahead); returns the index of its first record.
size_t build_row_program(const std::vector<PrimOp>& prims, size_t first, size_t last, int n,
                         std::vector<RowOp>& out);

// Every row of rho through the program at d_ops, in place.
hipError_t launch_rows(double* re, double* im, const RowOp* d_ops, int n, hipStream_t stream);

// ---- the steps on a thread's 2^K entries (register bit t <-> bit t of the index);
// coef(i): the step's coefficient i; on: whether the step applies to this
// thread (selected without a branch: a divergent one would have the compiler
// lay out the whole dispatch as a chain of predicated blocks) ----

// How many coefficients a pair primitive has.
inline constexpr int row_coefs(int kind)
{
    return kind == PK_C1 ? 8 : kind == PK_RY ? 4 : (kind == PK_RX || kind == PK_U1) ? 2 : kind == PK_R ? 1 : 0;
}

template <int K, int KIND, int T, class Coef>
__host__ __device__ __forceinline__ void row_dense(const Coef& coef, bool on, double* vr, double* vi)
{
    if constexpr (T < K) {
        double c[8] = {};
#pragma unroll
        for (int i = 0; i < row_coefs(KIND); i++) c[i] = coef(i);
#pragma unroll
        for (int i = 0; i < (1 << K); i++) {
            if (i & (1 << T)) continue;
            const int j = i | (1 << T);
            double r0, i0, r1, i1;
            out0<KIND>(c, vr[i], vi[i], vr[j], vi[j], r0, i0);
            out1<KIND>(c, vr[i], vi[i], vr[j], vi[j], r1, i1);
            if constexpr (KIND == PK_X) {  // may be a controlled swap
                r0 = on ? r0 : vr[i], i0 = on ? i0 : vi[i];
                r1 = on ? r1 : vr[j], i1 = on ? i1 : vi[j];
            }
            vr[i] = r0, vi[i] = i0, vr[j] = r1, vi[j] = i1;
        }
    }
}

template <int K, int KIND, int T, class Coef>
__host__ __device__ __forceinline__ void row_diag(const Coef& coef, bool on, double* vr, double* vi)
{
    if constexpr (T < K || T == 4) {
        double c[8] = {};
#pragma unroll
        for (int i = 0; i < row_coefs(KIND); i++) c[i] = coef(i);
#pragma unroll
        for (int i = 0; i < (1 << K); i++) {
            if (T < 4 && !(i & (1 << T))) continue;
            double r1, i1;
            out1<KIND>(c, 0.0, 0.0, vr[i], vi[i], r1, i1);
            if constexpr (T == 4) r1 = on ? r1 : vr[i], i1 = on ? i1 : vi[i];
            vr[i] = r1, vi[i] = i1;
        }
    }
}

template <int K, int T, int C>
__host__ __device__ __forceinline__ void row_cx(double* vr, double* vi)
{
    if constexpr (T < K && C < K && T != C) {
#pragma unroll
        for (int i = 0; i < (1 << K); i++) {
            if ((i & (1 << T)) || !(i & (1 << C))) continue;
            const int j = i | (1 << T);
            const double r = vr[i], m = vi[i];
            vr[i] = vr[j], vi[i] = vi[j];
            vr[j] = r, vi[j] = m;
        }
    }
}

// The 4x4 in the summation order of sweep_quad (sweep.hip).
template <int K, int P, class Coef>
__host__ __device__ __forceinline__ void row_c2(const Coef& coef, double* vr, double* vi)
{
    if constexpr (2 * P + 1 < K) {
        double e[32];
#pragma unroll
        for (int i = 0; i < 32; i++) e[i] = coef(i);
#pragma unroll
        for (int i = 0; i < (1 << K); i++) {
            if (i & (3 << (2 * P))) continue;
            double xr[4], xi[4];
#pragma unroll
            for (int j = 0; j < 4; j++) xr[j] = vr[i | (j << (2 * P))], xi[j] = vi[i | (j << (2 * P))];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const double* er = e + 8 * r;
                double s = (er[0] * xr[0]) - (er[1] * xi[0]);
                s = s + (er[2] * xr[1]);
                s = s - (er[3] * xi[1]);
                s = s + (er[4] * xr[2]);
                s = s - (er[5] * xi[2]);
                s = s + (er[6] * xr[3]);
                s = s - (er[7] * xi[3]);
                double v = (er[0] * xi[0]) + (er[1] * xr[0]);
                v = v + (er[2] * xi[1]);
                v = v + (er[3] * xr[1]);
                v = v + (er[4] * xi[2]);
                v = v + (er[5] * xr[2]);
                v = v + (er[6] * xi[3]);
                v = v + (er[7] * xr[3]);
                vr[i | (r << (2 * P))] = s;
                vi[i | (r << (2 * P))] = v;
            }
        }
    }
}

// Whether a program on 2^k entries per thread has steps of this code.
inline constexpr bool row_code_ok(int k, uint32_t code)
{
    if (code == RC_SKIP) return true;
    if (code >= RC_DENSE && code < RC_DIAG) return (int)(code - RC_DENSE) % 4 < k;
    if (code >= RC_DIAG && code < RC_CX) {
        const int t = (int)(code - RC_DIAG) % 8;
        return t < k || t == 4;
    }
    if (code >= RC_CX && code < RC_C2) {
        const int t = (int)(code - RC_CX) / 4, c = (int)(code - RC_CX) % 4;
        return t != c && t < k && c < k;
    }
    return code >= RC_C2 && code < RC_COUNT && 2 * (int)(code - RC_C2) + 1 < k;
}

inline constexpr int row_codes_below(int k, uint32_t code)
{
    int n = 0;
    for (uint32_t c = 0; c < code; c++) n += row_code_ok(k, c) ? 1 : 0;
    return n;
}

// One primitive step; its code is one of the allowed ones in [LO, HI).  A tree
// of two-way branches: a switch costs the structurised control flow of this
// target a chain of blocks and copies of every entry.
template <int K, uint32_t LO, uint32_t HI, class Coef>
__host__ __device__ __forceinline__ void row_step_in(uint32_t code, const Coef& coef, bool on,
                                                     double* vr, double* vi)
{
    constexpr int count = row_codes_below(K, HI) - row_codes_below(K, LO);
    if constexpr (count == 0) {
    } else if constexpr (!row_code_ok(K, LO)) {
        row_step_in<K, LO + 1, HI>(code, coef, on, vr, vi);
    } else if constexpr (count == 1) {
        if constexpr (LO == RC_SKIP) {
        } else if constexpr (LO < RC_DIAG)
            row_dense<K, (int)(LO - RC_DENSE) / 4, (int)(LO - RC_DENSE) % 4>(coef, on, vr, vi);
        else if constexpr (LO < RC_CX)
            row_diag<K, PK_Z + (int)(LO - RC_DIAG) / 8, (int)(LO - RC_DIAG) % 8>(coef, on, vr, vi);
        else if constexpr (LO < RC_C2)
            row_cx<K, (int)(LO - RC_CX) / 4, (int)(LO - RC_CX) % 4>(vr, vi);
        else
            row_c2<K, (int)(LO - RC_C2)>(coef, vr, vi);
        // a mark that differs from leaf to leaf, so that their last writes are not
        // merged into one through a computed entry (which would put the entries
        // into scratch memory)
        __asm__ volatile("" ::"i"(LO));
    } else {
        constexpr uint32_t mid = (LO + HI) / 2;
        if (code < mid)
            row_step_in<K, LO, mid>(code, coef, on, vr, vi);
        else
            row_step_in<K, mid, HI>(code, coef, on, vr, vi);
    }
}

template <int K, class Coef>
__host__ __device__ __forceinline__ void row_step(uint32_t code, const Coef& coef, bool on, double* vr,
                                                  double* vi)
{
    row_step_in<K, 0, RC_COUNT>(code, coef, on, vr, vi);
}

}  // namespace dmx
