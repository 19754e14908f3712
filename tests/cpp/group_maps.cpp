// Group sweeps (dm-sim_amd/csrc/group.hpp) on the CPU, thread by thread with the
// kernel's own index maps, on plans from dmx::build_fused_plan: the schedule
// takes every item once for several grids, every load is an entry that the
// sweep before wrote (the rest is poisoned), every store lies inside the planes
// and no entry is written twice, and the run's result equals the circuit's
// gates and channels applied one after the other to a random Hermitian matrix.
// Prints "<cases> cases OK", or the first violation and exits nonzero.
#include <cmath>
#include <complex>
#include <cstdio>
#include <cstring>
#include <limits>
#include <random>
#include <vector>

#include "fuse.hpp"
#include "herm.hpp"
#include "lower.hpp"

using namespace dmx;
using cd = std::complex<double>;
using Mat = std::vector<cd>;

namespace {

// A <- conj(G) A G^T for G on bits q (q[t] <-> matrix index bit t) of a d x d matrix.
void unitary(Mat& A, int d, const std::vector<int>& q, const std::vector<cd>& G)
{
    const int k = (int)q.size(), D = 1 << k;
    int mask = 0;
    for (int b : q) mask |= 1 << b;
    std::vector<int> at(D, 0);
    for (int s = 0; s < D; s++)
        for (int t = 0; t < k; t++)
            if ((s >> t) & 1) at[s] |= 1 << q[t];
    std::vector<cd> v(D);
    for (int side = 0; side < 2; side++)
        for (int other = 0; other < d; other++)
            for (int base = 0; base < d; base++) {
                if (base & mask) continue;
                auto e = [&](int s) -> cd& {
                    return side ? A[(size_t)(base | at[s]) * d + other] : A[(size_t)other * d + (base | at[s])];
                };
                for (int s = 0; s < D; s++) v[s] = e(s);
                for (int r = 0; r < D; r++) {
                    cd y = 0;
                    for (int s = 0; s < D; s++) y += (side ? std::conj(G[r * D + s]) : G[r * D + s]) * v[s];
                    e(r) = y;
                }
            }
}

// The superoperator S on bits lo, hi (row and column): index 4 * (row bits) + (column bits).
void super(Mat& A, int d, const std::vector<int>& q, const std::vector<cd>& S)
{
    const int k = (int)q.size(), D = 1 << k;
    int mask = 0;
    for (int b : q) mask |= 1 << b;
    auto at = [&](int s) {
        int x = 0;
        for (int t = 0; t < k; t++)
            if ((s >> t) & 1) x |= 1 << q[t];
        return x;
    };
    std::vector<cd> v(D * D);
    for (int r0 = 0; r0 < d; r0++)
        for (int c0 = 0; c0 < d; c0++) {
            if ((r0 & mask) || (c0 & mask)) continue;
            for (int s = 0; s < D * D; s++) v[s] = A[(size_t)(r0 | at(s / D)) * d + (c0 | at(s % D))];
            for (int i = 0; i < D * D; i++) {
                cd y = 0;
                for (int s = 0; s < D * D; s++) y += S[i * D * D + s] * v[s];
                A[(size_t)(r0 | at(i / D)) * d + (c0 | at(i % D))] = y;
            }
        }
}

int fail(const char* what, int n, int seed)
{
    std::printf("FAIL %s (n=%d seed=%d)\n", what, n, seed);
    return 1;
}

}  // namespace

int main()
{
    int cases = 0, fives = 0, pairs = 0, perms = 0;
    for (int n = 8; n <= 10; n++)
        for (int seed = 0; seed < (n < 10 ? 4 : 2); seed++) {
            std::mt19937 rng(50 * n + seed);
            std::normal_distribution<double> g01(0.0, 1.0);
            const bool noisy = seed % 2;
            std::vector<Gate> circ;
            for (int i = 0; i < 70; i++) {
                Gate g;
                if (noisy && rng() % 3 == 0) {
                    // one Kraus operator: A' = conj(K) A K^T keeps Hermitian matrices Hermitian
                    g.op = OP_KRAUS;
                    g.qb[0] = rng() % n;
                    g.mre.assign(32, 0.0), g.mim.assign(32, 0.0);
                    for (int t = 0; t < 2; t++) {
                        cd K[4];
                        for (cd& v : K) v = 0.5 * cd(g01(rng), g01(rng));
                        for (int i4 = 0; i4 < 16; i4++) {
                            const int a = i4 >> 3, b = (i4 >> 2) & 1, a2 = (i4 >> 1) & 1, b2 = i4 & 1;
                            const cd s = std::conj(K[2 * a + a2]) * K[2 * b + b2];
                            g.mre[i4] += s.real(), g.mim[i4] += s.imag();
                        }
                    }
                } else {
                    const int ops[] = {OP_U3, OP_H, OP_CX, OP_CX, OP_SWAP, OP_X, OP_CU1, OP_RYY, OP_CCX,
                                       OP_C3X, OP_C4X};
                    g.op = i == 20 ? (int)OP_C4X : ops[rng() % (i % 10 == 0 ? 11 : 9)];
                    g.theta = g01(rng), g.phi = g01(rng), g.lambda = g01(rng);
                    for (int j = 0; j < op_arity(g.op); j++)
                        for (bool again = true; again;) {
                            g.qb[j] = rng() % n;
                            again = false;
                            for (int k = 0; k < j; k++) again = again || g.qb[k] == g.qb[j];
                        }
                }
                circ.push_back(g);
            }
            const int d = 1 << n;
            Mat A((size_t)d * d);
            for (int r = 0; r < d; r++)
                for (int c = 0; c <= r; c++) {
                    A[(size_t)r * d + c] = cd(g01(rng), r == c ? 0.0 : g01(rng));
                    A[(size_t)c * d + r] = std::conj(A[(size_t)r * d + c]);
                }
            Mat W = A;
            for (const Gate& g : circ) {
                std::vector<cd> G;
                if (g.op == OP_KRAUS) {
                    for (int i = 0; i < 16; i++) G.push_back(cd(g.mre[i], g.mim[i]));
                    super(W, d, {(int)g.qb[0]}, G);
                    continue;
                }
                int k = 0;
                std::vector<uint32_t> q;
                std::vector<double> re, im;
                gate_matrix(g, k, q, re, im);
                for (size_t i = 0; i < re.size(); i++) G.push_back(cd(re[i], im[i]));
                unitary(W, d, std::vector<int>(q.rbegin(), q.rend()), G);
            }
            FusedPlan* plan = nullptr;
            PlanInfo info;
            if (build_fused_plan(circ, n, 4, nullptr, 0, true, &plan, &info, true, true, true) || !plan)
                return fail("plan", n, seed);
            std::vector<PlanStepView> steps;
            plan->describe(steps);
            const cd poison(std::numeric_limits<double>::quiet_NaN(), 0.0);
            Mat B;
            for (const PlanStepView& v : steps) {
                B.assign((size_t)d * d, poison);
                std::vector<char> wrote((size_t)d * d, 0);
                if (v.kind == PlanStepView::RELABEL) {
                    auto to = [&](int x) {
                        int y = 0;
                        for (int q = 0; q < n; q++)
                            if ((x >> q) & 1) y |= (int)v.block->perm_L[q];
                        return y;
                    };
                    for (int r = 0; r < d; r++)
                        for (int c = 0; c < d; c++) B[(size_t)to(r) * d + to(c)] = A[(size_t)r * d + c];
                    A.swap(B);
                    continue;
                }
                if (v.kind != PlanStepView::GROUP) return fail("step kind", n, seed);
                const GroupBlock& b = *v.group;
                GroupGeom g;
                g.init(b, n);
                perms += b.perm_b != 0;
                for (uint32_t grid : {8u, 24u, 128u, 512u}) {
                    std::vector<int> seen(g.items(), 0);
                    for (uint32_t blk = 0; blk < grid; blk++) {
                        uint32_t w = 0, k = 0;
                        while (group_slot(g.items(), blk, grid, k++, w)) seen[w]++;
                    }
                    for (int s : seen)
                        if (s != 1) return fail("schedule", n, seed);
                }
                for (uint32_t w = 0; w < g.items(); w++) {
                    const GroupItem it = group_item(g, w);
                    Mat T(64 * 64, poison);
                    for (uint32_t tid = 0; tid < (uint32_t)kGroupThreads; tid++) {
                        GroupThread th;
                        th.init(g, tid);
                        for (int rep = 0; rep < kGroupReps; rep++) {
                            const uint32_t a = th.row + 8 * rep;
                            const uint64_t off = group_load(g, th, it, rep);
                            if (off + 1 >= A.size() || (off & 1) || a >= 64) return fail("load", n, seed);
                            T[a * 64 + th.pair] = A[off];
                            T[a * 64 + th.pair + 1] = A[off + 1];
                        }
                    }
                    for (const cd& x : T)
                        if (std::isnan(x.real())) return fail("read of an unwritten entry", n, seed);
                    for (uint32_t s = b.stage0; s < b.stage0 + b.stages; s++) {
                        const GroupStage& st = v.gstages[s];
                        const int k = st.kind == GS_PAIR ? 2 : st.kind == GS_UNITARY4 ? 4 : 5;
                        const int size = st.kind == GS_UNITARY5 ? 1024 : 256;
                        std::vector<int> q;
                        uint32_t all = 0;
                        for (int i = 0; i < 6; i++) all |= 1u << group_bit(st, i);
                        if (all != 63u) return fail("stage bits", n, seed);
                        for (int i = 0; i < k; i++) q.push_back((int)group_bit(st, i));
                        std::vector<cd> G(size);
                        for (int i = 0; i < size; i++) G[i] = cd(v.gmats[st.mat + i], v.gmats[st.mat + size + i]);
                        if (st.kind == GS_PAIR)
                            super(T, 64, q, G);
                        else
                            unitary(T, 64, q, G);
                        fives += st.kind == GS_UNITARY5;
                        pairs += st.kind == GS_PAIR;
                    }
                    Mat P(4096, poison);  // the tile in its LDS places
                    for (uint32_t a = 0; a < 64; a++)
                        for (uint32_t c = 0; c < 64; c++) P[group_place(a, c)] = T[a * 64 + c];
                    for (const cd& x : P)
                        if (std::isnan(x.real())) return fail("places", n, seed);
                    auto put = [&](uint64_t off, cd x0, cd x1) {
                        if (off + 1 >= B.size() || (off & 1) || wrote[off]++ || wrote[off + 1]++) return false;
                        B[off] = x0, B[off + 1] = x1;
                        return true;
                    };
                    for (uint32_t tid = 0; tid < (uint32_t)kGroupThreads; tid++) {
                        GroupThread th;
                        th.init(g, tid);
                        for (int rep = 0; rep < kGroupReps; rep++) {
                            for (int m = 0; m < 2; m++) {
                                // as the kernel: one set always, the mirror's too where both are on
                                if (m == 0 ? !it.direct && !it.mirror : !(it.direct && it.mirror)) continue;
                                const bool mirror = m || !it.direct;
                                uint32_t x, dx;
                                const uint64_t off = group_store(g, th, it, mirror, rep, x, dx);
                                if (x >= 4096 || (x ^ dx) >= 4096) return fail("place", n, seed);
                                const cd v0 = P[x], v1 = P[x ^ dx];
                                if (!put(off, mirror ? std::conj(v0) : v0, mirror ? std::conj(v1) : v1))
                                    return fail("store", n, seed);
                            }
                        }
                    }
                    if (!it.direct && !it.mirror) return fail("item without a store", n, seed);
                }
                A.swap(B);
            }
            double err = 0, big = 0;
            for (size_t i = 0; i < A.size(); i++) {
                if (!(std::abs(A[i] - W[i]) <= err)) err = std::abs(A[i] - W[i]);
                big = std::max(big, std::abs(W[i]));
            }
            if (!(err <= 1e-11 * big)) return std::printf("FAIL result n=%d seed=%d: %g of %g\n", n, seed, err, big), 1;
            delete plan;
            cases++;
        }
    if (!fives || !pairs || !perms) return std::printf("FAIL coverage %d %d %d\n", fives, pairs, perms), 1;
    std::printf("%d cases OK\n", cases);
    return 0;
}
