// fuse.hpp -- fused execution: gates merged into dense k-qubit blocks, each
// applied to rho's row and column index in one sweep.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <vector>

#include "lower.hpp"
#include "prim.hpp"
#include "fused.hpp"
#include "group.hpp"
#include "prof.hpp"
#include "resident.hpp"

namespace dmx {

class CostModel;  // mlp.hpp

// What the planner chose.  predicted_us is the cost model's estimate of the
// run's launches (0 without a model); greedy_us its estimate for every block
// fused at the default tile width.
struct PlanInfo {
    uint32_t fused_blocks = 0;   // four-qubit blocks run fused
    uint32_t plain_blocks = 0;   // four-qubit blocks run as primitive sweeps on both indices
    uint32_t fused5_blocks = 0;  // five-qubit blocks run fused (a split one counts as its
                                 // four-qubit sub-blocks instead)
    uint32_t channels = 0;       // noise channels (one superoperator sweep each)
    uint32_t perm_blocks = 0;    // fused four-qubit blocks with a trailing permutation
    uint32_t herm_blocks = 0;    // four-qubit blocks run as Hermitian sweeps
    uint32_t relabels = 0;       // relabelling sweeps
    uint32_t grouping = 0;       // 0 least growth, 1 frontier, 2..5 frontier, other scores
    uint32_t tile_hist[9] = {};  // fused blocks per tile width m (4..8)
    double predicted_us = 0.0;
    double greedy_us = 0.0;
};

// One step of a fused plan as the executor runs it (host-side checks).
struct PlanStepView {
    enum Kind { FUSED4, FUSED5, HERM, RELABEL, CHANNEL, OTHER, GROUP } kind;
    const FusedBlock* block;    // FUSED4, HERM, RELABEL: its record as launched
    const FusedBlock5* block5;  // FUSED5
    const PrimOp* prim;         // CHANNEL: its record for the stored orientation (the
                                // conj-transposed one follows it)
    const GroupBlock* group;    // GROUP, with the plan's stages and matrices
    const GroupStage* gstages;
    const double* gmats;
};

// Algorithmic bytes of one Hermitian block sweep (k_fused4_herm) on n >= 8
// qubits: the super-tiles on and above the diagonal read (16 * H(H+1)/2 of
// them, H = 2^(n-8), 64 KiB each); written: every entry, or (half, when the
// next step is another Hermitian sweep) the tiles on and above that sweep's
// diagonal, T(T+1)/2 of the T^2 tiles (T = 2^(n-4)).
inline double herm_bytes(int n, bool half)
{
    const double H = (double)(1ull << (n - 8));
    const double T = (double)(1ull << (n - 4));
    const double rho = 16.0 * (double)(1ull << (2 * n));
    return 16.0 * H * (H + 1.0) / 2.0 * 65536.0 + (half ? rho * (T + 1.0) / (2.0 * T) : rho);
}

struct FusedPlan {
    virtual ~FusedPlan() = default;
    virtual void describe(std::vector<PlanStepView>& out) const = 0;
    virtual int upload(hipStream_t stream) = 0;
    // Whether blocks hold channels (FusedStage): execute then takes rho in its
    // stored orientation only (transposed = false).
    virtual bool staged() const = 0;
    // Whether every block runs on resident rows (resident.hpp) instead of in sweeps.
    virtual bool resident() const = 0;
    // Their records on the host (d_parts not set), for batched launches.
    virtual const std::vector<ResidentPart>& resident_parts() const = 0;
    virtual ResidentJob resident_job() const = 0;
    // Whether execute leaves rho in the other orientation (conj-transposed).
    virtual bool flips() const = 0;
    // Whether execute needs a second pair of planes (blocks with a trailing
    // permutation run out of place).
    virtual bool needs_alt() const = 0;
    // Applies the whole circuit once on `stream`, timing launches into prof.
    // transposed: rho is held conj-transposed (after a plain run), which
    // selects the channel superoperators' records.  rho is in (re, im); an
    // out-of-place sweep writes (re2, im2) and swaps the pairs, so on return
    // (re, im) holds rho again.
    virtual int execute(double*& re, double*& im, double*& re2, double*& im2, int n,
                        bool transposed, hipStream_t stream, LaunchProfiler& prof,
                        uint32_t* launches, uint32_t* sweeps) = 0;
    // After upload: times up to eight of the plan's four-qubit block sweeps (in
    // place, on the scratch planes re, im) at every tile width from 5 to
    // min(8, n) -- and 4 when every sampled block holds qubit 0 -- and gives
    // every block the fastest width where it is admissible.  *chosen = that
    // width (0: no block to time).  Updates info's width histogram.
    virtual int autotune_tiles(int n, double* re, double* im, hipStream_t stream, int* chosen,
                               PlanInfo& info) = 0;
    // Algorithmic bytes of one execute() on n qubits (rho not transposed):
    // the sum of what its launches record in the profiler.
    virtual double bytes(int n) const = 0;
};

// Blocks of a circuit in execution order: order[i] = (0, index into blocks)
// for a block of at most four qubits (padded to four), (2, index into
// blocks5) for a five-qubit block, (3, circuit index) for a channel, which no
// gate crosses.
struct BlockPlan {
    std::vector<FusedBlock> blocks;
    std::vector<std::vector<int>> members;  // circuit indices of each block's gates, in order
    // members[b][0, dense[b]) form the block matrix; the rest are trailing
    // permutation gates (X, CX, SWAP) applied as the block's index map
    std::vector<int> dense;
    std::vector<FusedBlock5> blocks5;
    std::vector<std::vector<int>> members5;
    std::vector<FusedStage> stages;  // of the blocks with channels
    std::vector<std::pair<int, int>> order;
};

// Greedy planning into blocks of at most max(max_k, widest gate) qubits
// (max_k <= 5; blocks below four qubits are padded to four).  fusable = false
// (and no blocks) when the circuit must run the plain method (SRN, n < 4).
// allow_perm (n <= 16): a four-qubit block may also take the X, CX and SWAP
// gates that become ready after it, run as a permutation of its output
// (launch_fused4_perm, out of place).
// herm: the plan runs Hermitian sweeps (k_fused4_herm), whose output map must
// send the block's index bits onto bits 0..3: a trailing CX then joins only if
// its control is not a block bit (after the block's earlier trailing gates)
// while its target is not.
// model: choose among the least-growth grouping, the frontier grouping and the
// frontier grouping scored by the gates' predicted unfused times (all gates,
// multi-qubit gates only, square roots) and by structural scores with heavy
// one-qubit gates, the one whose blocks the network prices cheapest (each the
// cheaper of its fused sweep and its gates unfused); without a model the one
// with fewer sweeps of the first two.  *grouping (may be null) = the choice:
// 0..5 in that order.
// resident: the blocks run on resident rows, all at one price: of the first two
// groupings the one with fewer blocks, whatever the model, and any X, CX or SWAP
// may trail a block.
// fold: a channel is a member of a block like a one-qubit gate, and a block
// with channels runs as stages (unless a gate is wider than four qubits:
// channels then stand between blocks, as without fold).
int plan_blocks(const std::vector<Gate>& circuit, int n, int max_k, BlockPlan& out, bool& fusable,
                bool allow_perm = false, bool herm = false, CostModel* model = nullptr,
                uint32_t* grouping = nullptr, bool fold = false, bool resident = false);

// Relative extra cost of a sweep with a trailing permutation on n qubits:
// about 2.5 us of index-map set-up against the sweep's own time (32 * 4^n bytes
// at ~4.6 TB/s plus ~8 us of launch latency), at least 3 % (measured at n = 8
// and n = 14).
inline double permute_overhead(int n)
{
    const double sweep_us = 32.0 * (double)(1ull << (2 * n)) / 4.6e6 + 8.0;
    const double r = 2.5 / sweep_us;
    return r > 0.03 ? r : 0.03;
}

// From this many qubits a permuting plan is kept without comparison; below, it
// is kept only if its sweeps, each permuting one charged permute_overhead(n)
// extra, are fewer than the in-place plan's.
constexpr int kPermuteSureQubits = 12;
inline bool permuting_pays(int n, double sweeps, double permuting, double sweeps_inplace)
{
    return n >= kPermuteSureQubits || sweeps + permute_overhead(n) * permuting < sweeps_inplace;
}



// Plan of a circuit for the fused executor.  With a cost model, each block is
// priced as a fused launch at every tile width and as its primitive sweeps
// (a five-qubit block: as its member gates re-planned into four-qubit
// blocks), and the cheapest is taken; a plan with five-qubit blocks is kept
// only if predicted faster than the four-qubit plan of the same circuit.
// Without a model, every block is fused at the default tile width (the
// greedy plan).
// tile_bits > 0 fixes every fused block's tile width where that width is
// admissible for the block (tile_bits_ok), and takes precedence over the model.
// herm (n = 8..16, with allow_perm): four-qubit blocks run as Hermitian
// sweeps (k_fused4_herm) with rho's index bits relabelled so that each
// block's output lands in aligned 16-column runs; rho returns to the
// circuit's bit order (k_relabel) before any other step and at the end.
// group (with herm and fold): the whole plan as group sweeps (k_group) of six
// qubits whose stages are the blocks: several blocks of at most max_k qubits
// (five for a five-qubit gate) to a sweep.
// resident (where resident_wanted, with allow_perm): the blocks run on resident
// rows; the model's prices still are those of sweeps.
int build_fused_plan(const std::vector<Gate>& circuit, int n, int max_k, CostModel* model,
                     int tile_bits, bool allow_perm, FusedPlan** out, PlanInfo* info,
                     bool herm = false, bool fold = false, bool group = false,
                     bool resident = false);

// Whether a unitary circuit's blocks may run on resident rows: 4 to
// kResidentMaxQubits qubits, no channels, no gate on more than four qubits, and at
// most four qubits to a block.
bool resident_wanted(const std::vector<Gate>& circuit, int n, int max_k);

// Whether a resident plan of so many blocks, none with a trailing permutation, runs them as
// in-place sweeps after all.  Alone, from 9 qubits the resident passes' two launches (and
// from 10 the conjugate transpose between them) take 30, 41 and 78 us a run with one block
// and 32, 45 and 85 with two (9, 10 and 11 qubits) where one sweep takes 21, 22 and 45 and two
// take 25, 41 and 79 to 83; three take 34, 52 and 113 against 33, 49 and 98.  Below 9 one
// graph launch hides the difference (20 to 24 us either way up to two, 26 against 21 with
// three).  In a batch (96 circuits of 4 to 9 qubits, 64 of 10, 32 of 11) one block takes 37, 39,
// 46, 64, 112, 488, 1651 and 3145 us resident and 26, 24, 29, 50, 91, 295, 696 and 1330 in
// place; two 45 and 51 against 30 and 39 (5 and 6 qubits); three, from 7 to 11, 72, 144,
// 573, 1874 and (four) 3796 against 91, 208, 710, 1622 and 4055.  One rule for both, so
// that a batched rho stays bit-identical to the circuit's own run.  At 4 qubits, where a
// plan is one block, alone both take 24 us, and the resident form is what a test of it runs.
inline bool resident_is_brief(int n, int blocks) { return n > 4 && blocks <= 2; }

// The tile width of such sweeps of one circuit, fastest on circuits of two blocks (us a run at
// widths 6, 7 and 8): 8 qubits 20.4, 23.4 and 30; 9 26.5, 27.7 and 33; 10 46, 36 and 43; 11
// 110, 85 and 81.  Timing the widths at upload would gain up to 2 us a run for 0.5 to 2.5 ms.
inline int brief_tile_bits(int n) { return n < 6 ? n : n <= 9 ? 6 : n == 10 ? 7 : 8; }

// Whether a circuit's Hermitian plan runs as group sweeps.  With channels, from
// 12 qubits: a group holds their whole neighbourhood where a four-qubit block
// with a channel on every gate fills up with channels (a 300-member 12-qubit
// circuit 1680 us in four-qubit blocks with channels, 1520 in groups; below 12 qubits rho
// fits the caches and a sweep costs its launch).  With five-qubit gates, from 13: the five-qubit sweep has no
// Hermitian form (structured circuits 21.5 -> 15.4 ms at 13 qubits, 84 -> 68
// at 14, 354 -> 297 at 15).  Other unitary circuits keep four-qubit sweeps: on
// 2130 gates at 14 qubits 113 group sweeps of 1.69 ms take 193 ms, 181 of the
// others 177, as a group's 2.2 stages occupy the matrix cores for 1 ms that
// overlaps its 1.1 ms of memory traffic only in part.
bool group_wanted(const std::vector<Gate>& circuit, int n);

// From this many qubits the engine folds channels into blocks.  A noisy
// 318-member circuit at 8 qubits takes 9 sweeps instead of 138 and 180 channel
// sweeps (1.32 -> 0.22 ms a run with its downloads), one of 164 members at 12
// qubits 12 instead of 182 launches (16.1 -> 1.95 ms).  It would pay below as well: 100
// gates with a channel on every operand take 558, 694 and 688 us at 4, 5 and 6 qubits
// and would take 31, 47 and 45.  There a plan stays at one launch per block and channel
// because a test at 6 qubits counts them, and no setting asks for channels as barriers.
constexpr int kFoldChannelQubits = 7;

// Smallest n for Hermitian plans, and the smallest where the engine uses
// them by default.
constexpr int kHermMinQubits = 8;
constexpr int kHermAutoQubits = 12;

}  // namespace dmx
