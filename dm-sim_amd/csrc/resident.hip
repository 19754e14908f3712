// resident.hip -- fused four-qubit blocks on whole rows of rho, for gfx950.
//
// Rows do not depend on each other on the column index, so a workgroup loads
// whole rows (2^n entries, 4 KiB to 32 KiB) into LDS once, applies every block of
// the circuit to their columns with FP64 MFMA and stores them once; a second pass
// does the same to the row index.  A block sweep, one launch per block, moves rho
// through the caches each time and pays a launch: 6 us at 8 qubits and 38 us at 11.
//
// A block is Y = U X on the 16 x 16 tiles of the rows, X's columns the other index
// bits: a lane reads and writes the same four places, so a block takes one barrier
// (none where a wave holds the row, up to 8 qubits).  Index permutations between
// blocks (X, CX, SWAP) only change the places that later records name.
//
// Bound: up to 9 qubits one wave's chain of LDS reads, 12 MFMAs and LDS writes (0.63
// us a block and pass at n = 8, where 256 waves have a SIMD each); from 10 the FP64
// matrix cores, busy 69 % of the time at n = 11 (8.3 us a block and pass for 6.2 at 65
// TFLOP/s; LDS 21 % of the time, 15 % of that bank conflicts), with four waves of two
// tiles, one after the other, which leave registers for five workgroups a CU: with eight
// waves of a tile, two workgroups, 64 % (601 gates 665 -> 638 us a pass, 96 circuits of
// 6 to 11 qubits 16.4 -> 14.9 ms).
// Against one launch per block: 90 blocks at n = 8 586 -> 113 us a run, 30 at n = 11
// 1305 -> 520.
#include <hip/hip_runtime.h>

#include "resident.hpp"

namespace dmx {

namespace {

typedef double d4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ d4 mfma(double a, double b, d4 c)
{
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

}  // namespace

// n <= LOGE; a chunk is 2^C entries, C = LOGE + X, in 2^(C - 8) tiles, dealt to the
// waves in runs.  SLOW: rows and columns of rho exchanged, and conjugated values.  X: as
// many rows more to a chunk as records of 2^LOGE entries have tiles (2^X times), so that
// a SLOW one's columns lie together in memory.
template <int LOGE, int WAVES, bool SLOW, int X = 0>
__device__ __forceinline__ void resident_pass(const ResidentJob& job)
{
    constexpr int C = LOGE + X;
    double* const re = job.re;
    double* const im = job.im;
    const double2* const parts = reinterpret_cast<const double2*>(job.parts);
    const int blocks = job.blocks, n = job.n;
    const ResidentEnd& end = job.end;
    constexpr int kThreads = 64 * WAVES;
    constexpr int kPer = (1 << (C - 8)) / WAVES;  // tiles of a wave
    __shared__ double2 s[1 << C];
    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & 63u, wave = tid >> 6;
    // entry i of the thread's share in memory order: its index in the chunk, its offset
    auto entry = [&](uint32_t i, uint32_t& e) -> uint64_t {
        const uint32_t f = SLOW ? tid + i * kThreads : 2 * (tid + i * kThreads);
        if constexpr (!SLOW) {
            e = f;
            return ((uint64_t)blockIdx.x << C) + f;
        }
        const int rows = C - n;  // 2^rows columns of rho to a chunk, neighbours together
        const uint32_t c = f & ((1u << rows) - 1u), r = f >> rows;
        e = r | c << n;
        return ((uint64_t)r << n) + ((uint64_t)blockIdx.x << rows) + c;
    };

    const double2* src = parts + lane;
    double2 next[kResidentParts];
#pragma unroll
    for (int i = 0; i < kResidentParts; i++) next[i] = src[64 * i];

    if constexpr (SLOW) {
#pragma unroll
        for (int i = 0; i < (1 << C) / kThreads; i++) {
            uint32_t e;
            const uint64_t off = entry(i, e);
            s[row_place(e, 3, C)] = make_double2(re[off], -im[off]);
        }
    } else {
#pragma unroll
        for (int i = 0; i < (1 << C) / kThreads / 2; i++) {
            uint32_t e;
            const uint64_t off = entry(i, e);
            const double2 r = *reinterpret_cast<const double2*>(re + off);
            const double2 m = *reinterpret_cast<const double2*>(im + off);
            const uint32_t x = row_place(e, 3, C);
            s[x] = make_double2(r.x, m.x);
            s[x ^ 1u] = make_double2(r.y, m.y);
        }
    }

    for (int b = 0; b < blocks; b++) {
        const double ur[4] = {next[0].x, next[0].y, next[1].x, next[1].y};
        const double ui[4] = {next[2].x, next[2].y, next[3].x, next[3].y};
        const uint32_t w0 = (uint32_t)__double2loint(next[4].x), w1 = (uint32_t)__double2hiint(next[4].x);
        const uint32_t w2 = (uint32_t)__double2loint(next[4].y);
        const uint32_t c0 = w0 >> 16, c1 = w1 & 0xFFFFu;
        const uint32_t t[3] = {w1 >> 16, w2 & 0xFFFFu, w2 >> 16};
        src += 64 * kResidentParts;
        __syncthreads();
        if (b + 1 < blocks) {
#pragma unroll
            for (int i = 0; i < kResidentParts; i++) next[i] = src[64 * i];
        }
#pragma unroll 1
        for (int u = 0; u < kPer; u++) {
            const uint32_t tile = wave * kPer + u;
            uint32_t x[4] = {w0 & 0xFFFFu};
#pragma unroll
            for (int i = 0; i < LOGE - 8; i++) x[0] ^= (tile >> i) & 1u ? t[i] : 0u;
#pragma unroll
            for (int i = LOGE; i < C; i++) x[0] ^= (tile >> (i - 8)) & 1u ? row_place(1u << i, 3, C) : 0u;
            x[1] = x[0] ^ c0;
            x[2] = x[0] ^ c1;
            x[3] = x[1] ^ c1;
            double2 v[4];
#pragma unroll
            for (int c = 0; c < 4; c++) v[c] = s[x[c]];
            // three real products, p1 = Ur Xr (in yr), p2 = Ui Xi and, in yi, (Ur + Ui) (Xr +
            // Xi) (as four chained by their accumulators 601 gates at n = 11 take
            // 700 us a pass for 651, and the results are a little further off)
            d4 yr = {0, 0, 0, 0}, yi = yr, p2 = yr;
#pragma unroll
            for (int c = 0; c < 4; c++) {
                yr = mfma(ur[c], v[c].x, yr);
                p2 = mfma(ui[c], v[c].y, p2);
                yi = mfma(ur[c] + ui[c], v[c].x + v[c].y, yi);
            }
            yi = yi - yr - p2;
            yr = yr - p2;
#pragma unroll
            for (int r = 0; r < 4; r++) s[x[r]] = make_double2(yr[r], yi[r]);
        }
    }
    __syncthreads();

    auto end_place = [&](uint32_t e) {
        uint32_t x = end.base;
#pragma unroll
        for (int i = 0; i < LOGE; i++) x ^= (e >> i) & 1u ? end.bit[i] : 0u;
#pragma unroll
        for (int i = LOGE; i < C; i++) x ^= (e >> i) & 1u ? row_place(1u << i, 3, C) : 0u;
        return x;
    };
    if constexpr (SLOW) {
#pragma unroll
        for (int i = 0; i < (1 << C) / kThreads; i++) {
            uint32_t e;
            const uint64_t off = entry(i, e);
            const double2 v = s[end_place(e)];
            re[off] = v.x;
            im[off] = -v.y;
        }
    } else {
#pragma unroll
        for (int i = 0; i < (1 << C) / kThreads / 2; i++) {
            uint32_t e;
            const uint64_t off = entry(i, e);
            const uint32_t x = end_place(e);
            const double2 a = s[x], b = s[x ^ end.bit[0]];
            *reinterpret_cast<double2*>(re + off) = make_double2(a.x, b.x);
            *reinterpret_cast<double2*>(im + off) = make_double2(a.y, b.y);
        }
    }
}

template <int LOGE, int WAVES, bool SLOW>
__global__ void __launch_bounds__(64 * WAVES, 5) k_resident(const ResidentJob job)
{
    resident_pass<LOGE, WAVES, SLOW>(job);
}

template <int LOGE, int WAVES, bool SLOW, int X = 0>
__global__ void __launch_bounds__(64 * WAVES, 5) k_resident_batch(const ResidentJob* __restrict__ jobs)
{
    const ResidentJob& job = jobs[blockIdx.y];
    if (blockIdx.x >= 1u << (2 * job.n - LOGE - X)) return;  // a narrower circuit's
    resident_pass<LOGE, WAVES, SLOW, X>(job);
}

hipError_t launch_resident(const ResidentJob& job, bool slow, hipStream_t stream)
{
    const int n = job.n;
    if (n < 4 || n > (slow ? kResidentColumnQubits : kResidentMaxQubits) || job.blocks < 1)
        return hipErrorInvalidValue;
    const int L = resident_log_entries(n);
    const unsigned grid = 1u << (2 * n - L);
    switch (2 * L + (slow ? 1 : 0)) {
    case 16: k_resident<8, 1, false><<<grid, 64, 0, stream>>>(job); break;
    case 17: k_resident<8, 1, true><<<grid, 64, 0, stream>>>(job); break;
    case 18: k_resident<9, 2, false><<<grid, 128, 0, stream>>>(job); break;
    case 19: k_resident<9, 2, true><<<grid, 128, 0, stream>>>(job); break;
    case 20: k_resident<10, 4, false><<<grid, 256, 0, stream>>>(job); break;
    default: k_resident<11, 4, false><<<grid, 256, 0, stream>>>(job); break;
    }
    return hipGetLastError();
}

hipError_t launch_resident_batch(const ResidentJob* d_jobs, int count, int log_entries, bool slow,
                                 int extra, hipStream_t stream)
{
    if (count < 1 || count > 65535 || log_entries < 8 ||
        log_entries > (slow ? kResidentColumnQubits : kResidentMaxQubits))
        return hipErrorInvalidValue;
    const dim3 grid(1u << (log_entries - extra), (unsigned)count);  // n = log_entries: most chunks
    switch (100 * extra + 2 * log_entries + (slow ? 1 : 0)) {
    case 16: k_resident_batch<8, 1, false><<<grid, 64, 0, stream>>>(d_jobs); break;
    case 17: k_resident_batch<8, 1, true><<<grid, 64, 0, stream>>>(d_jobs); break;
    case 117: k_resident_batch<8, 2, true, 1><<<grid, 128, 0, stream>>>(d_jobs); break;
    case 317: k_resident_batch<8, 8, true, 3><<<grid, 512, 0, stream>>>(d_jobs); break;
    case 18: k_resident_batch<9, 2, false><<<grid, 128, 0, stream>>>(d_jobs); break;
    case 319: k_resident_batch<9, 8, true, 3><<<grid, 512, 0, stream>>>(d_jobs); break;
    case 20: k_resident_batch<10, 4, false><<<grid, 256, 0, stream>>>(d_jobs); break;
    case 22: k_resident_batch<11, 4, false><<<grid, 256, 0, stream>>>(d_jobs); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace dmx
