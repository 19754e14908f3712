// rows.hip -- the plain method with whole rows of rho on chip, for gfx950.
//
// k_rows runs a segment's program (rows.hpp) on the column index: a workgroup
// loads whole rows once, applies every primitive of the segment to them in
// the reference's order and with its arithmetic, and stores them once.  Rows
// do not depend on each other, so there is no grid barrier and no pass over
// rho per primitive: a segment's two index passes are this kernel, an
// in-place conjugate transpose and this kernel again.
//
// Bound: from 10 qubits the FP64 VALU (mul and add apart, as the reference
// rounds them: 77-78 % busy at n = 11 and 13) and, between groups of primitives on at
// most K target bits, one LDS round trip of the row; below, the latency of one
// wave's chain of steps (0.3 us each: dispatch, a few dependent FP64
// operations and a third of an LDS round trip).
// Measured against one persistent launch per pass with a grid barrier per
// primitive: 200 gates at n = 6 1.6 -> 0.23 ms, 700 at n = 8 11.8 -> 0.72 ms, 600
// at n = 11 76 -> 2.4 ms, 4 SU(4) layers and 120 gates at n = 13 112 -> 17 ms; against
// one launch per primitive 2130 gates at n = 14 5.84 -> 0.73 s.
#include <hip/hip_runtime.h>

#include "rows.hpp"

namespace dmx {

template <int K, int LOGE, bool SPLIT>
__global__ void __launch_bounds__(1 << (LOGE - K))
    k_rows(double* __restrict__ re, double* __restrict__ im, const RowOp* __restrict__ ops,
           uint64_t entries)
{
    constexpr int kThreads = 1 << (LOGE - K);
    constexpr uint32_t kEntries = 1u << LOGE;
    constexpr int kPer = 1 << K;
    constexpr int kDigit = SPLIT ? 4 : 3;
    // SPLIT: one plane at a time (8-byte places), else both (16-byte places)
    __shared__ double lds[SPLIT ? kEntries : 2 * kEntries];
    double2* const pairs = reinterpret_cast<double2*>(lds);
    const uint32_t tid = threadIdx.x;
    const uint64_t first = (uint64_t)blockIdx.x << LOGE;

    double vr[kPer], vi[kPer];
    uint32_t at = 0, reg[4] = {0, 0, 0, 0};  // LDS places: this thread's entry 0, the register bits
    auto place = [&](int i) {
        return at ^ ((i & 1) ? reg[0] : 0u) ^ ((i & 2) ? reg[1] : 0u) ^ ((i & 4) ? reg[2] : 0u) ^
               ((i & 8) ? reg[3] : 0u);
    };
    auto to_lds = [&](const double* v) {
#pragma unroll
        for (int i = 0; i < kPer; i++) lds[place(i)] = v[i];
    };
    auto from_lds = [&](double* v) {
#pragma unroll
        for (int i = 0; i < kPer; i++) v[i] = lds[place(i)];
    };
    // a plane's rows between memory and LDS (SPLIT: n = 14, every entry there)
    auto plane_in = [&](const double* p) {
#pragma unroll
        for (int i = 0; i < kPer / 2; i++) {
            const uint32_t e = 2 * (tid + i * kThreads);
            const double2 v = *reinterpret_cast<const double2*>(p + first + e);
            const uint32_t x = row_place(e, kDigit, LOGE);
            lds[x] = v.x;
            lds[x ^ 1u] = v.y;
        }
    };
    auto plane_out = [&](double* p) {
#pragma unroll
        for (int i = 0; i < kPer / 2; i++) {
            const uint32_t e = 2 * (tid + i * kThreads);
            const uint32_t x = row_place(e, kDigit, LOGE);
            *reinterpret_cast<double2*>(p + first + e) = make_double2(lds[x], lds[x ^ 1u]);
        }
    };
    if constexpr (!SPLIT) {
#pragma unroll
        for (int i = 0; i < kPer / 2; i++) {
            const uint32_t e = 2 * (tid + i * kThreads);
            double2 r = make_double2(0.0, 0.0), m = r;
            if (first + e < entries) {  // 4^n < 2^LOGE at n <= 3
                r = *reinterpret_cast<const double2*>(re + first + e);
                m = *reinterpret_cast<const double2*>(im + first + e);
            }
            const uint32_t x = row_place(e, kDigit, LOGE);
            pairs[x] = make_double2(r.x, m.x);
            pairs[x ^ 1u] = make_double2(r.y, m.y);
        }
    }

    bool held = false;
    // The program streams through registers: lane l holds bytes 16 l .. of the
    // chunk, the next chunk's load is in flight, and a record's words come by
    // v_readlane (scalar loads one record ahead: 4.2 against 2.8 ms for 600
    // gates at n = 11, as the loads hold the steps' registers).
    const uint4* src = reinterpret_cast<const uint4*>(ops) + (tid & 63u);
    constexpr uint32_t kStride = kRowChunk * sizeof(RowOp) / sizeof(uint4);
    uint4 chunk = src[0], ahead = src[kStride];
    src += 2 * kStride;
    uint32_t r = 0;  // record within the chunk
    auto word = [&](uint32_t d) {  // word d from record r on
        const int lane = (int)(5 * r + d / 4);
        const uint32_t v = (d & 3) == 0 ? chunk.x : (d & 3) == 1 ? chunk.y : (d & 3) == 2 ? chunk.z : chunk.w;
        return (uint32_t)__builtin_amdgcn_readlane((int)v, lane);
    };
    auto coef = [&](uint32_t i) {  // 8 coefficients to a record, after its 4 head words
        const uint32_t d = 20 * (i / 8) + 4 + 2 * (i % 8);
        return __hiloint2double((int)word(d + 1), (int)word(d));
    };
    for (;;) {
        if (r >= (uint32_t)kRowChunk) {
            chunk = ahead;
            ahead = src[0];
            src += kStride;
            r = 0;
        }
        const uint32_t code = word(0);
        if (code == RC_END) break;
        if (code != RC_REGROUP) {
            const uint32_t on = word(1);
            row_step<K>(code, coef, (tid & on) == on, vr, vi);
            r += (code - RC_C2 < 2u) ? 4 : 1;
            continue;
        }
        uint32_t to = 0;
#pragma unroll
        for (int i = 0; i < LOGE - K; i++) to ^= word(8 + i) & (0u - ((tid >> i) & 1u));
        uint32_t place_of[4];
#pragma unroll
        for (int i = 0; i < K; i++) place_of[i] = word(4 + i);
        r++;
        auto move = [&] {
            at = to;
#pragma unroll
            for (int i = 0; i < K; i++) reg[i] = place_of[i];
        };
        if constexpr (SPLIT) {
            const uint32_t at0 = at, r0 = reg[0], r1 = reg[1], r2 = reg[2], r3 = reg[3];
            if (held)
                to_lds(vr);
            else
                plane_in(re);
            __syncthreads();
            move();
            from_lds(vr);
            __syncthreads();
            if (held) {
                at = at0, reg[0] = r0, reg[1] = r1, reg[2] = r2, reg[3] = r3;
                to_lds(vi);
                move();
            } else {
                plane_in(im);
            }
            __syncthreads();
            from_lds(vi);
            __syncthreads();
        } else {
            // every place belongs to one thread per group: one barrier a regroup
            if (held) {
#pragma unroll
                for (int i = 0; i < kPer; i++) pairs[place(i)] = make_double2(vr[i], vi[i]);
            }
            __syncthreads();
            move();
#pragma unroll
            for (int i = 0; i < kPer; i++) {
                const double2 v = pairs[place(i)];
                vr[i] = v.x;
                vi[i] = v.y;
            }
        }
        held = true;
    }
    if (!held) return;  // an empty segment
    if constexpr (SPLIT) {
        to_lds(vr);
        __syncthreads();
        plane_out(re);
        __syncthreads();
        to_lds(vi);
        __syncthreads();
        plane_out(im);
    } else {
#pragma unroll
        for (int i = 0; i < kPer; i++) pairs[place(i)] = make_double2(vr[i], vi[i]);
        __syncthreads();
#pragma unroll
        for (int i = 0; i < kPer / 2; i++) {
            const uint32_t e = 2 * (tid + i * kThreads);
            if (first + e >= entries) continue;
            const uint32_t x = row_place(e, kDigit, LOGE);
            const double2 a = pairs[x], b = pairs[x ^ 1u];
            *reinterpret_cast<double2*>(re + first + e) = make_double2(a.x, b.x);
            *reinterpret_cast<double2*>(im + first + e) = make_double2(a.y, b.y);
        }
    }
}

namespace {

template <int K, int LOGE, bool SPLIT>
void launch(double* re, double* im, const RowOp* d_ops, uint64_t entries, hipStream_t stream)
{
    const unsigned blocks = (unsigned)((entries + (1ull << LOGE) - 1) >> LOGE);
    k_rows<K, LOGE, SPLIT><<<blocks, 1 << (LOGE - K), 0, stream>>>(re, im, d_ops, entries);
}

}  // namespace

hipError_t launch_rows(double* re, double* im, const RowOp* d_ops, int n, hipStream_t stream)
{
    if (n < 1 || n > kRowsMaxQubits) return hipErrorInvalidValue;
    const uint64_t entries = 1ull << (2 * n);
    switch (n <= 8 ? 8 : n) {
    case 8: launch<2, 8, false>(re, im, d_ops, entries, stream); break;
    case 9: launch<2, 10, false>(re, im, d_ops, entries, stream); break;
    case 10: launch<3, 10, false>(re, im, d_ops, entries, stream); break;
    case 11: launch<3, 11, false>(re, im, d_ops, entries, stream); break;
    case 12: launch<3, 12, false>(re, im, d_ops, entries, stream); break;
    case 13: launch<3, 13, false>(re, im, d_ops, entries, stream); break;
    default: launch<4, 14, true>(re, im, d_ops, entries, stream); break;
    }
    return hipGetLastError();
}

}  // namespace dmx
