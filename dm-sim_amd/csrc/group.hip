// group.hip -- Hermitian group sweeps for gfx950 (records and index maps:
// group.hpp).
//
// A workgroup (4 waves) takes one 64 x 64 tile at a time: loads into LDS, the
// group's stages there with FP64 MFMA (v_mfma_f64_16x16x4f64), stores of the
// result and its mirror.  Two workgroups per CU (80 KiB of LDS each) overlap one
// another's phases, and a workgroup's next tile is loaded into registers while
// its stages run (not where a five-qubit stage needs the registers).
//
// Bound by both memory and matrix cores: on 14 qubits a sweep without stages
// takes 1150 us (4.3 GB, 3.7 TB/s) and a four-qubit stage keeps the matrix cores busy
// for 430 us (24 MFMAs of 2048 operations per 256 entries, at 64 of the 65-67
// TFLOP/s that a long run of these instructions reaches); a sweep with 2.2 stages on
// average 1690 us.  512 threads, i.e. four waves per SIMD, took longer: the matrix core
// is as busy with two, and each wave's stage setup counts twice.
#include <hip/hip_runtime.h>

#include "group.hpp"

namespace dmx {

namespace {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef double dv2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ d4 mfma(double a, double b, d4 c)
{
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// Doubles of stage matrices kept in LDS beside the tile: with the tile's 64 KiB
// half of a CU's LDS.
constexpr uint32_t kMatsInLds = 2048;

// MFMA lane layout: A[i][k] in lane i + 16k, B[k][j] in lane j + 16k, D[4r + g][j]
// in lane j + 16g register r.  Complex products round as those of the block sweeps
// do: unitaries take three real products combined after their sums, superoperators four.
// Chaining three through one sum (re = K - Ai (Br + Bi), im = K + Ar (Bi - Br) from K = (Ar +
// Ai) Br) lets the accumulators do the additions and is faster where a sweep has
// several stages (2.2 on average at 14 qubits 1577 us for 1689; 40 noisy gates at 12 qubits
// 1350 us a run for 1520), but further off: RMS over rho after those 40 gates 1.76e-15
// for 1.52e-15, where one sweep per channel has 1.58e-15.

// A unitary on four bits: 16 sub-tiles of 16 x 16 (the other two bits of rows
// and columns), wave w those with row part w, two at a time; per sub-tile X =
// T U^T, then T' = conj(U) X (12 + 12 MFMAs; register c of X is the second
// product's B operand).  Places are a lane part, computed once a stage, XORed with
// uniform parts.
template <class Mat>
__device__ __forceinline__ void stage_unitary4(const GroupStage& s, const Mat& mat, int wave, int j,
                                               int kk, double* __restrict__ s_re,
                                               double* __restrict__ s_im)
{
    double ur[4], ui[4];
    uint32_t urow[4], ucol[4];  // places of matrix index 4c as a row, as a column
#pragma unroll
    for (int c = 0; c < 4; c++) {
        ur[c] = mat(j * 16 + 4 * c + kk);
        ui[c] = mat(256 + j * 16 + 4 * c + kk);
        const uint32_t q = group_local(s, 2, 2, c);
        urow[c] = group_row_place(q);
        ucol[c] = group_col_place(q);
    }
    const uint32_t qj = group_local(s, 0, 4, j), qk = group_local(s, 0, 2, kk);
    const uint32_t rd = group_place(qj, qk), wr = group_place(qk, qj);
    const uint32_t row0 = group_row_place(group_local(s, 4, 2, wave));
#pragma unroll 1
    for (int t = 0; t < 2; t++) {
        double tr[2][4], ti[2][4];
        uint32_t base[2];
#pragma unroll
        for (int u = 0; u < 2; u++) {
            base[u] = row0 ^ group_col_place(group_local(s, 4, 2, 2 * t + u));
#pragma unroll
            for (int c = 0; c < 4; c++) {
                tr[u][c] = s_re[rd ^ (base[u] ^ ucol[c])];
                ti[u][c] = s_im[rd ^ (base[u] ^ ucol[c])];
            }
        }
        d4 p[2] = {}, q[2] = {}, k[2] = {}, xr[2], xi[2];
#pragma unroll
        for (int c = 0; c < 4; c++)
#pragma unroll
            for (int u = 0; u < 2; u++) {
                p[u] = mfma(tr[u][c], ur[c], p[u]);
                q[u] = mfma(ti[u][c], ui[c], q[u]);
                k[u] = mfma(tr[u][c] + ti[u][c], ur[c] + ui[c], k[u]);
            }
#pragma unroll
        for (int u = 0; u < 2; u++) {
            xr[u] = p[u] - q[u];
            xi[u] = k[u] - p[u] - q[u];
            p[u] = q[u] = k[u] = d4{0, 0, 0, 0};
        }
#pragma unroll
        for (int c = 0; c < 4; c++)
#pragma unroll
            for (int u = 0; u < 2; u++) {
                p[u] = mfma(ur[c], xr[u][c], p[u]);
                q[u] = mfma(-ui[c], xi[u][c], q[u]);
                k[u] = mfma(ur[c] - ui[c], xr[u][c] + xi[u][c], k[u]);
            }
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const d4 yr = p[u] - q[u];
            const d4 yi = k[u] - p[u] - q[u];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                s_re[wr ^ (base[u] ^ urow[r])] = yr[r];
                s_im[wr ^ (base[u] ^ urow[r])] = yi[r];
            }
        }
    }
}

// A superoperator of two bits: Y = S X with X's rows their 16 (row, column)
// values and its columns 16 values of the other bits; wave w takes the other
// row bits' values 4w..4w+3, two at a time (16 MFMAs each, read and written by the
// same lane).
template <class Mat>
__device__ __forceinline__ void stage_pair(const GroupStage& s, const Mat& mat, int wave, int j, int kk,
                                           double* __restrict__ s_re, double* __restrict__ s_im)
{
    double ur[4], ui[4];
    uint32_t urow[4];
#pragma unroll
    for (int c = 0; c < 4; c++) {
        ur[c] = mat(j * 16 + 4 * c + kk);
        ui[c] = mat(256 + j * 16 + 4 * c + kk);
        urow[c] = group_row_place(group_local(s, 0, 2, c));
    }
    const uint32_t lane = group_col_place(group_local(s, 0, 2, kk) | group_local(s, 2, 4, j));
#pragma unroll 1
    for (int t = 0; t < 2; t++) {
        double tr[2][4], ti[2][4];
        uint32_t base[2];
#pragma unroll
        for (int u = 0; u < 2; u++) {
            base[u] = group_row_place(group_local(s, 2, 4, 4 * wave + 2 * t + u));
#pragma unroll
            for (int c = 0; c < 4; c++) {
                tr[u][c] = s_re[lane ^ (base[u] ^ urow[c])];
                ti[u][c] = s_im[lane ^ (base[u] ^ urow[c])];
            }
        }
        d4 yr[2] = {}, yi[2] = {};
#pragma unroll
        for (int c = 0; c < 4; c++)
#pragma unroll
            for (int u = 0; u < 2; u++) {
                yr[u] = mfma(ur[c], tr[u][c], yr[u]);
                yi[u] = mfma(ur[c], ti[u][c], yi[u]);
            }
#pragma unroll
        for (int c = 0; c < 4; c++)
#pragma unroll
            for (int u = 0; u < 2; u++) {
                yr[u] = mfma(-ui[c], ti[u][c], yr[u]);
                yi[u] = mfma(ui[c], tr[u][c], yi[u]);
            }
#pragma unroll
        for (int u = 0; u < 2; u++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                s_re[lane ^ (base[u] ^ urow[r])] = yr[u][r];
                s_im[lane ^ (base[u] ^ urow[r])] = yi[u][r];
            }
    }
}

// A unitary on five bits: four sub-tiles of 32 x 32, one per wave, as 2 x 2
// parts of 16 x 16 over eight K-chunks.  Column half J of X = T U^T and then of
// T' = conj(U) X; the first half's result waits in registers until the second
// half has read T.  The scheduler is kept from gathering a whole product's
// operands, which would spill.
template <class Mat>
__device__ __forceinline__ void stage_unitary5(const GroupStage& s, const Mat& mat, int wave, int j,
                                               int kk, double* __restrict__ s_re,
                                               double* __restrict__ s_im)
{
    const uint32_t hi = 1u << group_bit(s, 4);
    const uint32_t base =
        group_place((wave & 1) << group_bit(s, 5), (wave >> 1) << group_bit(s, 5));
    const uint32_t hi_row = group_row_place(hi), hi_col = group_col_place(hi);
    const uint32_t qj = group_local(s, 0, 4, j), qk = group_local(s, 0, 2, kk);
    const uint32_t rd = base ^ group_place(qj, qk), wr = base ^ group_place(qk, qj);
    const int mj = j * 32 + kk;
    d4 zr[2], zi[2];  // T'[I][0]
#pragma unroll
    for (int J = 0; J < 2; J++) {
        d4 p[2] = {}, q[2] = {}, k[2] = {}, xr[2], xi[2], yr[2], yi[2];
#pragma unroll 2
        for (int K = 0; K < 8; K++) {
            const uint32_t x = rd ^ group_col_place(group_local(s, 2, 3, K));
            const double ur = mat(mj + 512 * J + 4 * K), ui = mat(1024 + mj + 512 * J + 4 * K);
#pragma unroll
            for (int I = 0; I < 2; I++) {
                const uint32_t xI = I ? x ^ hi_row : x;
                const double tr = s_re[xI], ti = s_im[xI];
                p[I] = mfma(tr, ur, p[I]);
                q[I] = mfma(ti, ui, q[I]);
                k[I] = mfma(tr + ti, ur + ui, k[I]);
            }
        }
#pragma unroll
        for (int I = 0; I < 2; I++) {
            xr[I] = p[I] - q[I];
            xi[I] = k[I] - p[I] - q[I];
            p[I] = q[I] = k[I] = d4{0, 0, 0, 0};
        }
#pragma unroll
        for (int K = 0; K < 8; K++) {
            const double br = xr[K >> 2][K & 3], bi = xi[K >> 2][K & 3];
#pragma unroll
            for (int I = 0; I < 2; I++) {
                const double ur = mat(mj + 512 * I + 4 * K), ui = mat(1024 + mj + 512 * I + 4 * K);
                p[I] = mfma(ur, br, p[I]);
                q[I] = mfma(-ui, bi, q[I]);
                k[I] = mfma(ur - ui, br + bi, k[I]);
            }
            if (K & 1) __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int I = 0; I < 2; I++) {
            yr[I] = p[I] - q[I];
            yi[I] = k[I] - p[I] - q[I];
        }
#pragma unroll
        for (int I = 0; I < 2; I++) {
            if (J == 0) {
                zr[I] = yr[I];
                zi[I] = yi[I];
                continue;
            }
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const uint32_t x = wr ^ group_row_place(group_local(s, 2, 2, r)) ^ (I ? hi_row : 0u);
                s_re[x] = zr[I][r];
                s_im[x] = zi[I][r];
                s_re[x ^ hi_col] = yr[I][r];
                s_im[x ^ hi_col] = yi[I][r];
            }
        }
    }
}

}  // namespace

// FIVE: the group has five-qubit unitaries, whose registers leave no room for
// the next tile's loads: it is loaded when its turn comes.
template <bool FIVE>
__global__ void __launch_bounds__(kGroupThreads, 2)
    k_group(const double* __restrict__ re, const double* __restrict__ im, double* __restrict__ re_out,
            double* __restrict__ im_out, const GroupBlock* __restrict__ blk,
            const GroupStage* __restrict__ all_stages, const double* __restrict__ mats, int n)
{
    __shared__ double s_re[kGroupDim * kGroupDim];
    __shared__ double s_im[kGroupDim * kGroupDim];
    __shared__ double s_mat[kMatsInLds];
    const uint32_t tid = threadIdx.x;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int j = lane & 15, kk = lane >> 4;
    GroupGeom g;
    g.init(*blk, n);
    GroupThread th;
    th.init(g, tid);
    const GroupStage* const stages = all_stages + blk->stage0;
    const int count = (int)blk->stages;
    const uint32_t items = g.items();
    // The group's matrices, one after the other in the pool, as far as they fit.
    // From memory a stage's matrix would be waited for after the next tile's
    // loads, which were issued before it and return in order.
    const uint32_t mat0 = count > 0 ? stages[0].mat : 0;
    const uint32_t mat_end = blk->mat_end;
    for (uint32_t i = tid; i < kMatsInLds && mat0 + i < mat_end; i += kGroupThreads) s_mat[i] = mats[mat0 + i];

    dv2 vr[kGroupReps], vi[kGroupReps];
    GroupItem it;
    uint32_t w = 0;
    bool have = group_slot(items, blockIdx.x, gridDim.x, 0, w);
    auto load = [&] {
        it = group_item(g, w);
#pragma unroll
        for (int rep = 0; rep < kGroupReps; rep++) {
            const uint64_t off = group_load(g, th, it, rep);
            vr[rep] = *reinterpret_cast<const dv2*>(re + off);
            vi[rep] = *reinterpret_cast<const dv2*>(im + off);
        }
    };
    auto store = [&](const GroupItem& at, bool mirror) {
        const double sign = mirror ? -1.0 : 1.0;
#pragma unroll
        for (int rep = 0; rep < kGroupReps; rep++) {
            uint32_t x, dx;
            const uint64_t off = group_store(g, th, at, mirror, rep, x, dx);
            const dv2 r{s_re[x], s_re[x ^ dx]}, m{sign * s_im[x], sign * s_im[x ^ dx]};
            __builtin_nontemporal_store(r, reinterpret_cast<dv2*>(re_out + off));
            __builtin_nontemporal_store(m, reinterpret_cast<dv2*>(im_out + off));
        }
    };
    if (!FIVE && have) load();
    for (uint32_t k = 1; have; k++) {
        if (FIVE) load();
#pragma unroll
        for (int rep = 0; rep < kGroupReps; rep++) {
            const uint32_t x = group_place(th.row + 8 * rep, th.pair), x1 = x ^ group_col_place(1);
            s_re[x] = vr[rep].x;
            s_re[x1] = vr[rep].y;
            s_im[x] = vi[rep].x;
            s_im[x1] = vi[rep].y;
        }
        const GroupItem cur = it;
        have = group_slot(items, blockIdx.x, gridDim.x, k, w);
        if (!FIVE && have) load();
        for (int t = 0; t < count; t++) {
            const GroupStage s = stages[t];
            const uint32_t size = s.kind == GS_UNITARY5 ? 2048u : 512u;
            const bool near = s.mat + size - mat0 <= kMatsInLds;
            __syncthreads();
            auto run = [&](const auto& mat) {
                if (s.kind == GS_UNITARY4)
                    stage_unitary4(s, mat, wave, j, kk, s_re, s_im);
                else if (!FIVE || s.kind == GS_PAIR)
                    stage_pair(s, mat, wave, j, kk, s_re, s_im);
                else if constexpr (FIVE)
                    stage_unitary5(s, mat, wave, j, kk, s_re, s_im);
            };
            if (near)
                run([&](int i) { return s_mat[s.mat - mat0 + i]; });
            else
                run([&](int i) { return mats[s.mat + i]; });
        }
        __syncthreads();
        // one set of stores on every path, so that the wait for the next tile's
        // loads, issued before them, need not wait for the stores as well
        store(cur, !cur.direct);
        if (cur.direct && cur.mirror) store(cur, true);
        __syncthreads();
    }
}

hipError_t launch_group(const double* re, const double* im, double* re_out, double* im_out,
                        const GroupBlock* d_blk, const GroupStage* d_stages, const double* d_mats,
                        int n, bool five, hipStream_t stream)
{
    if (n < 8 || n > 16 || re == re_out || im == im_out) return hipErrorInvalidValue;
    const uint32_t T = 1u << (n - kGroupBits);
    const uint32_t items = T * (T + 1) / 2;
    const uint32_t blocks = items < 512 ? (items + 7) / 8 * 8 : 512;  // two per CU at a time
    if (five)
        k_group<true><<<blocks, kGroupThreads, 0, stream>>>(re, im, re_out, im_out, d_blk, d_stages,
                                                            d_mats, n);
    else
        k_group<false><<<blocks, kGroupThreads, 0, stream>>>(re, im, re_out, im_out, d_blk, d_stages,
                                                             d_mats, n);
    return hipGetLastError();
}

}  // namespace dmx
