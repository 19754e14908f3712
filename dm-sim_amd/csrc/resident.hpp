// resident.hpp -- fused blocks on whole rows of rho held in LDS (resident.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <vector>

#include "fused.hpp"
#include "rows.hpp"

namespace dmx {

// Largest n that runs resident (a row of 2048 entries is 32 KiB, so five
// workgroups fit a CU).  From 12 qubits the Hermitian sweeps, which transform half
// of rho, are the default.
constexpr int kResidentMaxQubits = 11;
// Up to this many qubits the second pass reads and writes columns itself, as
// rho (4 MiB) stays in the caches; above, a conjugate transpose stands between two
// row passes, and rho is held conj-transposed after the run.
constexpr int kResidentColumnQubits = 9;

// A workgroup's chunk: 2^L entries of rho, whole rows (the low n bits of an entry
// number its column, the others its row).
inline int resident_log_entries(int n) { return n > 8 ? n : 8; }

// One block as a wave reads it: part s of lane l at [s * 64 + l].  Lane l =
// i + 16 k holds row i of the 16 x 16 matrix: u[0..1] the real parts of columns
// k, 4 + k and 8 + k, 12 + k, u[2..3] the imaginary ones.  LDS places (row_place)
// compose by XOR: at for the lane, c0 and c1 for the bits of the matrix index that
// the chunk c of four columns numbers, t0, t1, t2 for the bits of the tile's number.
// The lane reads entries (4 c + k) and writes them: the same places.
struct ResidentPart {
    union {
        double u[2];
        struct {
            uint16_t at, c0, c1, t0, t1, t2, pad[2];
        } place;
    };
};
constexpr int kResidentParts = 5;  // four of the matrix, then the places

// The last record: the place of entry 0 and, bit by bit, of an entry's index,
// for the store.
struct ResidentEnd {
    uint32_t base;
    uint32_t bit[11];
};

// The records of a sequence of blocks.  A block's trailing permutation costs
// nothing: it changes which places the index bits mean from there on.
void build_resident(const std::vector<FusedBlock>& blocks, const std::vector<int>& order, int n,
                    std::vector<ResidentPart>& parts, ResidentEnd& end);

// One circuit's rho and its records.
struct ResidentJob {
    double* re;
    double* im;
    const ResidentPart* parts;
    int32_t blocks;
    int32_t n;
    ResidentEnd end;
};

// rho <- rho U^T for the product U of all blocks, 4 <= n <= kResidentMaxQubits;
// slow (n <= kResidentColumnQubits): rho <- conj(U) rho.  In place.
hipError_t launch_resident(const ResidentJob& job, bool slow, hipStream_t stream);

// A batch's column passes run together and stream from memory, where a column alone is
// a strided run of 8-byte accesses: chunks take 2^X times as many columns (extra = X), 64
// bytes side by side at 8 and 9 qubits, 32 at 7.  96 ansatz circuits of 1 / 9 layers, us
// a run with X = 0, 1, 2, 3: 7 qubits 91 / 121, 69 / 110, -, 87 / 189 (waves that
// wait for one another's tiles); 8: 394 / 496, -, 180 / 357, 143 / 353; 9: 1497 / 1887, -,
// 853 / 1394, 572 / 1293; 6: 51 / 66 and 76 / 132 with 0 and 3.
inline int resident_extra(int n, bool slow) { return !slow || n < 7 ? 0 : n == 7 ? 1 : 3; }

// The same for `count` circuits whose chunks have 2^log_entries entries
// (resident_log_entries of every job's n, so one launch takes all widths up to 8), times
// 2^extra (resident_extra of every job's n).
hipError_t launch_resident_batch(const ResidentJob* d_jobs, int count, int log_entries, bool slow,
                                 int extra, hipStream_t stream);

}  // namespace dmx
