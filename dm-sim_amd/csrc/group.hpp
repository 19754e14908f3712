// group.hpp -- Hermitian group sweeps (k_group, group.hip): several blocks on
// up to six qubits applied in one sweep of rho.  Records, and the index maps,
// which the kernel shares with their CPU check (tests/cpp/group_maps.cpp).
//
// A sweep is on six index bits (qmask; bit 0 among them, so column pairs stay
// together).  Its tiles are the 64 x 64 entries over those bits with the other
// row and column bits fixed (free parts r, c); rho is Hermitian, so only the
// tiles with r <= c are read and transformed, and each result is written where
// the next sweep reads it, in place of the tile, in place of its mirror
// (conjugate transpose), or both.  Tiles pass through the group's stages in
// LDS.  The output map phi(x) = L x ^ b, chosen by the host, sends the span of
// qmask onto bits 0..5: tiles and mirrors land in 64 rows x one aligned run of
// 64 columns (512 bytes).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace dmx {

constexpr int kGroupBits = 6;
constexpr int kGroupDim = 1 << kGroupBits;
constexpr int kGroupThreads = 256;
constexpr int kGroupReps = kGroupDim * kGroupDim / 2 / kGroupThreads;  // column pairs a thread moves

// LDS place (in doubles) of local row a, column b of a tile.  16 lanes that read
// or write one row's or one column's entries over four of the six bits should
// hit 16 different eight-byte banks: the low four bits of the place are the XOR of
// one vector per bit of a and b, any four of the first five of which are
// independent (sets with the sixth conflict two ways at worst).  Linear over
// XOR, so places combine from lane and uniform parts.
__host__ __device__ inline uint32_t group_mix(uint32_t x)
{
    return (x & 15u) ^ (0u - ((x >> 4) & 1u) & 15u) ^ (0u - ((x >> 5) & 1u) & 5u);
}
__host__ __device__ inline uint32_t group_row_place(uint32_t a) { return (a << 6) | group_mix(a); }
__host__ __device__ inline uint32_t group_col_place(uint32_t b) { return (b & 48u) | group_mix(b); }
__host__ __device__ inline uint32_t group_place(uint32_t a, uint32_t b)
{
    return group_row_place(a) ^ group_col_place(b);
}

// One stage on a group's six local bits (bit t <-> the t-th lowest of qmask).
// bits: the local bits it acts on, lowest matrix index bit first, then the
// others, four bits each.  Matrices are row-major planes re, im at mat (doubles
// from the plan's pool).
enum GroupStageKind : uint32_t {
    GS_UNITARY4 = 0,  // 16 x 16 on four bits, both sides
    GS_UNITARY5 = 1,  // 32 x 32 on five bits, both sides
    GS_PAIR = 2       // superoperator of two bits u, v: 16 x 16 on the entries that differ in
                      // them, index 4 * (row bits v, u) + (column bits v, u)
};
struct GroupStage {
    uint32_t kind;
    uint32_t bits;
    uint32_t mat;
    uint32_t pad;
};

struct GroupBlock {
    uint32_t qmask;
    uint32_t stage0, stages;
    uint32_t next_q;   // the next group's qmask in this sweep's output order (half writes), 0 = write all
    uint32_t perm_b;
    uint32_t perm_L[16];
    uint32_t finv[6];  // inverse of f (f(a) = L on local index a), by columns
    uint32_t mat_end;  // where the stages' matrices (from stages[stage0].mat on) end in the pool
    uint32_t pad[4];
};
static_assert(sizeof(GroupBlock) == 128, "GroupBlock layout");

__host__ __device__ inline uint32_t group_bit(const GroupStage& s, int i) { return (s.bits >> (4 * i)) & 15u; }

// The low `count` bits of v on the stage's bits first, first + 1, ...
__host__ __device__ inline int group_local(const GroupStage& s, int first, int count, int v)
{
    int x = 0;
#pragma unroll
    for (int i = 0; i < count; i++) x |= ((v >> i) & 1) << group_bit(s, first + i);
    return x;
}

__host__ __device__ inline uint32_t group_deposit(uint32_t v, uint32_t mask)
{
    uint32_t out = 0;
    for (uint32_t m = mask; m; m &= m - 1) {
        if (v & 1u) out |= m & (~m + 1u);
        v >>= 1;
    }
    return out;
}

struct GroupGeom {
    uint64_t dim;
    uint32_t qmask, T;         // T = 2^(n - 6) free parts
    uint32_t free_bit[10];     // bit i of a free part: its index bit ...
    uint32_t free_img[10];     // ... and that bit's image under L
    uint32_t pb, finv[6];
    uint64_t rep_row[kGroupReps];  // row offset of local row 8 rep
    uint32_t rep_inv[kGroupReps];  // inv(8 rep)
    bool half;
    uint32_t hi_keep;          // bits >= 6 outside next_q

    __host__ __device__ void init(const GroupBlock& b, int n)
    {
        dim = 1ull << n;
        qmask = b.qmask;
        T = 1u << (n - kGroupBits);
        uint32_t m = (uint32_t)(dim - 1) & ~qmask;
#pragma unroll
        for (int i = 0; i < 10; i++) {
            const uint32_t bit = m & (~m + 1u);  // 0 once they are used up
            m &= m - 1u;
            free_bit[i] = bit;
            uint32_t img = 0;
#pragma unroll
            for (int q = 0; q < 16; q++) img ^= ((bit >> q) & 1u) ? b.perm_L[q] : 0u;
            free_img[i] = img;
        }
#pragma unroll
        for (int q = 0; q < 6; q++) finv[q] = b.finv[q];
        pb = b.perm_b;
#pragma unroll
        for (uint32_t rep = 0; rep < kGroupReps; rep++) {
            rep_row[rep] = (uint64_t)group_deposit(8u * rep, qmask) * dim;
            rep_inv[rep] = inv(8u * rep);
        }
        half = b.next_q != 0;
        hi_keep = (uint32_t)(dim - 1) & ~63u & ~b.next_q;
    }
    __host__ __device__ uint32_t inv(uint32_t p) const  // p < 64
    {
        uint32_t y = 0;
#pragma unroll
        for (int q = 0; q < 6; q++) y ^= ((p >> q) & 1u) ? finv[q] : 0u;
        return y;
    }
    __host__ __device__ uint32_t items() const { return T * (T + 1) / 2; }
};

// One work item: the tile of free parts r <= c, as index bits and as images
// under phi, and the local index that the images' low bits stand for.  It is
// written in its place (direct), in its mirror's, or both.
struct GroupItem {
    uint32_t rphys, cphys, R0, C0;
    bool direct, mirror;
};

// The triangle r <= c folded into a (T + 1) x T/2 rectangle: row a holds
// (a, a..T-1) then (T-1-a, T-1-a..T-1).
__host__ __device__ inline GroupItem group_item(const GroupGeom& g, uint32_t w)
{
    GroupItem it;
    const uint32_t a = w / (g.T + 1), bc = w % (g.T + 1);
    const bool first = bc < g.T - a;
    const uint32_t r = first ? a : g.T - 1 - a;
    const uint32_t c = r + (first ? bc : bc - (g.T - a));
    it.rphys = it.cphys = 0;
    it.R0 = it.C0 = g.pb;
#pragma unroll
    for (int i = 0; i < 10; i++) {
        const uint32_t rb = 0u - ((r >> i) & 1u), cb = 0u - ((c >> i) & 1u);
        it.rphys |= rb & g.free_bit[i];
        it.cphys |= cb & g.free_bit[i];
        it.R0 ^= rb & g.free_img[i];
        it.C0 ^= cb & g.free_img[i];
    }
    // the next sweep reads (x, y) with x <= y outside its bits: decided by the
    // high parts, or (equal) by bits inside the tile: then both are written
    const uint32_t rk = it.R0 & g.hi_keep, ck = it.C0 & g.hi_keep;
    it.direct = !g.half || rk <= ck;
    it.mirror = r != c && (!g.half || ck <= rk);
    return it;
}

// Schedule: a read's runs are as short as 32 bytes where few of the sweep's bits
// are the lowest index bits; the items that share their lines -- consecutive c
// -- go to one XCD (workgroups are dealt to the 8 XCDs round-robin) together,
// kGroupChunk at a time.  Slot s = block / 8 + k * (grid / 8) of an XCD (k-th
// pass of a workgroup's loop) takes item (s / chunk) * 8 * chunk + XCD * chunk +
// s % chunk.  False once the items are used up (then for every later k as
// well).  The grid is a multiple of 8.
constexpr uint32_t kGroupChunk = 16;
__host__ __device__ inline bool group_slot(uint32_t items, uint32_t block, uint32_t grid, uint32_t k,
                                           uint32_t& w)
{
    const uint32_t s = (block >> 3) + k * (grid >> 3);
    w = (s / kGroupChunk) * (8 * kGroupChunk) + (block & 7u) * kGroupChunk + s % kGroupChunk;
    return w < items;
}

// Per-thread constants (thread tid of 256): loads and stores move the column
// pair `pair`, pair + 1 of rows row + 8 rep.
struct GroupThread {
    uint32_t pair;  // 2 (tid % 32)
    uint32_t row;   // tid / 32
    uint64_t load;  // offset of the pair of row `row` in a tile at 0
    uint64_t store; // the same in an output tile
    uint32_t ip, ir;  // inv(pair), inv(row)

    __host__ __device__ void init(const GroupGeom& g, uint32_t tid)
    {
        pair = 2 * (tid & 31u);
        row = tid >> 5;
        load = group_deposit(pair, g.qmask) + (uint64_t)group_deposit(row, g.qmask) * g.dim;
        store = pair + (uint64_t)row * g.dim;
        ip = g.inv(pair);
        ir = g.inv(row);
    }
};

// Load rep: offset of the pair in a plane; it is local row row + 8 rep, columns
// pair, pair + 1.
__host__ __device__ inline uint64_t group_load(const GroupGeom& g, const GroupThread& t,
                                               const GroupItem& it, int rep)
{
    return (uint64_t)it.rphys * g.dim + it.cphys + g.rep_row[rep] + t.load;
}

// Stores of the tile (mirror: of its conjugate transpose in the mirror's place).
// Store rep: offset of the output pair; its two sources are the LDS places x and
// x ^ dx (conjugated for the mirror).
__host__ __device__ inline uint64_t group_store(const GroupGeom& g, const GroupThread& t,
                                                const GroupItem& it, bool mirror, int rep, uint32_t& x,
                                                uint32_t& dx)
{
    const uint32_t X0 = mirror ? it.C0 : it.R0, Y0 = mirror ? it.R0 : it.C0;  // output rows, columns
    const uint32_t s = t.ir ^ g.rep_inv[rep] ^ g.inv(X0 & 63u), k = t.ip ^ g.inv(Y0 & 63u);
    x = mirror ? group_place(k, s) : group_place(s, k);
    dx = mirror ? group_place(g.finv[0], 0) : group_place(0, g.finv[0]);
    return (uint64_t)((X0 & ~63u) + 8u * (uint32_t)rep) * g.dim + (Y0 & ~63u) + t.store;
}

// Algorithmic bytes of one sweep on n qubits: the tiles on and above the
// diagonal read; written, every entry or (half) the tiles on and above the
// next sweep's diagonal.
inline double group_bytes(int n, bool half)
{
    const double T = (double)(1ull << (n - kGroupBits));
    const double up = T * (T + 1.0) / 2.0 * 65536.0;
    return up + (half ? up : 16.0 * (double)(1ull << (2 * n)));
}

// One sweep from (re, im) into (re_out, im_out), n = 8..16; no overlap.  five:
// whether the group has a GS_UNITARY5 stage.
hipError_t launch_group(const double* re, const double* im, double* re_out, double* im_out,
                        const GroupBlock* d_blk, const GroupStage* d_stages, const double* d_mats,
                        int n, bool five, hipStream_t stream);

}  // namespace dmx
