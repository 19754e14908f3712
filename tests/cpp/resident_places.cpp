// The records of the resident block executor (dm-sim_amd/csrc/resident.hpp),
// executed on the CPU lane by lane and tile by tile: every block's lanes and tiles
// take each place of the chunk exactly once, and the rows afterwards are those of
// the blocks and their permutations applied one after the other.
#include <cmath>
#include <complex>
#include <cstdio>
#include <random>
#include <vector>

#include "resident.hpp"

using namespace dmx;
typedef std::complex<double> cd;

namespace {

std::mt19937 rng(7);

FusedBlock random_block(int n)
{
    FusedBlock fb = {};
    while (__builtin_popcount(fb.qmask) < 4) fb.qmask |= 1u << (rng() % n);
    std::normal_distribution<double> g(0.0, 0.25);
    for (int i = 0; i < 256; i++) fb.ur[i] = g(rng), fb.ui[i] = g(rng);
    fb.perm_on = rng() % 4 != 0;
    if (!fb.perm_on) return fb;
    fb.perm_b = rng() % (1u << n);
    for (int q = 0; q < n; q++) fb.perm_L[q] = 1u << q;
    for (int i = 0; i < 3 * n; i++) {  // L as a product of CX
        const int c = rng() % n, t = rng() % n;
        if (c == t) continue;
        for (int q = 0; q < n; q++)
            if ((fb.perm_L[q] >> c) & 1u) fb.perm_L[q] ^= 1u << t;
    }
    return fb;
}

void apply(const FusedBlock& fb, int n, std::vector<cd>& row)
{
    int q[4], k = 0;
    for (int i = 0; i < n; i++)
        if ((fb.qmask >> i) & 1u) q[k++] = i;
    auto local = [&](uint32_t x) {
        uint32_t v = 0;
        for (int t = 0; t < 4; t++) v |= ((x >> q[t]) & 1u) << t;
        return v;
    };
    std::vector<cd> out(row.size());
    for (uint32_t x = 0; x < row.size(); x++) {
        cd sum = 0;
        for (uint32_t v = 0; v < 16; v++) {
            uint32_t y = x & ~fb.qmask;
            for (int t = 0; t < 4; t++) y |= ((v >> t) & 1u) << q[t];
            sum += cd(fb.ur[16 * local(x) + v], fb.ui[16 * local(x) + v]) * row[y];
        }
        uint32_t to = x;
        if (fb.perm_on) {
            to = fb.perm_b;
            for (int i = 0; i < n; i++)
                if ((x >> i) & 1u) to ^= fb.perm_L[i];
        }
        out[to] = sum;
    }
    row = out;
}

bool run(int n, int count)
{
    std::vector<FusedBlock> blocks;
    std::vector<int> order;
    for (int i = 0; i < count; i++) blocks.push_back(random_block(n));
    for (int i = 0; i < count; i++) order.push_back(count - 1 - i);
    std::vector<ResidentPart> parts;
    ResidentEnd end;
    build_resident(blocks, order, n, parts, end);
    const int L = resident_log_entries(n), tiles = 1 << (L - 8);
    std::vector<cd> chunk(1u << L), lds(1u << L);
    std::normal_distribution<double> g;
    for (auto& v : chunk) v = cd(g(rng), g(rng));
    for (uint32_t e = 0; e < chunk.size(); e++) lds[row_place(e, 3, L)] = chunk[e];
    for (int b = 0; b < count; b++) {
        const ResidentPart* const rec = parts.data() + (size_t)b * kResidentParts * 64;
        std::vector<int> seen(lds.size(), 0);
        for (int t = 0; t < tiles; t++) {
            cd x[16][16], u[16][16];
            uint32_t at[64][4];
            for (int lane = 0; lane < 64; lane++) {
                const int j = lane & 15, k = lane >> 4;
                const auto& p = rec[4 * 64 + lane].place;
                for (int c = 0; c < 4; c++) {
                    uint32_t y = p.at ^ (c & 1 ? p.c0 : 0) ^ (c & 2 ? p.c1 : 0) ^ (t & 1 ? p.t0 : 0) ^
                                 (t & 2 ? p.t1 : 0) ^ (t & 4 ? p.t2 : 0);
                    if (y >= lds.size() || seen[y]++) return false;
                    at[lane][c] = y;
                    x[4 * c + k][j] = lds[y];
                    u[j][4 * c + k] = cd(rec[(c / 2) * 64 + lane].u[c % 2],
                                         rec[(2 + c / 2) * 64 + lane].u[c % 2]);
                }
            }
            for (int lane = 0; lane < 64; lane++)
                for (int r = 0; r < 4; r++) {
                    cd sum = 0;
                    for (int k = 0; k < 16; k++) sum += u[4 * r + (lane >> 4)][k] * x[k][lane & 15];
                    lds[at[lane][r]] = sum;
                }
        }
    }
    for (uint32_t row = 0; row < (1u << (L - n)); row++) {
        std::vector<cd> want(chunk.begin() + (row << n), chunk.begin() + ((row + 1) << n));
        for (int b : order) apply(blocks[b], n, want);
        for (uint32_t e = 0; e < (1u << n); e++) {
            uint32_t x = end.base;
            for (int i = 0; i < L; i++)
                if (((e | row << n) >> i) & 1u) x ^= end.bit[i];
            if (std::abs(lds[x] - want[e]) > 1e-12) return false;
        }
    }
    return true;
}

}  // namespace

int main()
{
    int ok = 0;
    for (int n = 4; n <= kResidentMaxQubits; n++)
        for (int count : {1, 2, 9}) {
            if (!run(n, count)) {
                std::printf("n = %d, %d blocks: wrong\n", n, count);
                return 1;
            }
            ok++;
        }
    std::printf("%d cases OK\n", ok);
}
