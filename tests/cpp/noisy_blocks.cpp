// Blocks with channels among their gates (dmx::plan_blocks with fold), on the
// CPU: the blocks in execution order, their tiles taken through the stage
// records as fused.hpp defines them and their trailing index maps, against the
// circuit's gates and channels one after the other on a random matrix.
// Prints "<cases> cases OK", or the first violation and exits nonzero.
#include <cmath>
#include <complex>
#include <cstdio>
#include <cstring>
#include <random>
#include <vector>

#include "fuse.hpp"
#include "lower.hpp"

using dmx::Gate;
using cd = std::complex<double>;
using Mat = std::vector<cd>;  // dim x dim, the stored A = conj(rho)

namespace {

// A <- conj(G) A G^T for G on qubits q (q[0]: the high bit of its index).
void unitary(Mat& A, int n, const std::vector<uint32_t>& q, const std::vector<cd>& G)
{
    const int k = (int)q.size(), d = 1 << k, dim = 1 << n;
    auto at = [&](int base, int s) {
        for (int j = 0; j < k; j++)
            if ((s >> (k - 1 - j)) & 1) base |= 1 << q[j];
        return base;
    };
    uint32_t mask = 0;
    for (uint32_t b : q) mask |= 1u << b;
    std::vector<cd> v(d);
    for (int side = 0; side < 2; side++)
        for (int other = 0; other < dim; other++)
            for (int base = 0; base < dim; base++) {
                if (base & mask) continue;
                for (int s = 0; s < d; s++) {
                    const int x = at(base, s);
                    v[s] = side ? A[(size_t)x * dim + other] : A[(size_t)other * dim + x];
                }
                for (int r = 0; r < d; r++) {
                    cd y = 0;
                    for (int s = 0; s < d; s++) y += (side ? std::conj(G[r * d + s]) : G[r * d + s]) * v[s];
                    const int x = at(base, r);
                    (side ? A[(size_t)x * dim + other] : A[(size_t)other * dim + x]) = y;
                }
            }
}

void channel(Mat& A, int n, const Gate& g)
{
    const int dim = 1 << n, b = 1 << g.qb[0];
    for (int r = 0; r < dim; r++)
        for (int c = 0; c < dim; c++) {
            if ((r & b) || (c & b)) continue;
            cd v[4], y[4];
            for (int s = 0; s < 4; s++) v[s] = A[(size_t)(r | (s & 2 ? b : 0)) * dim + (c | (s & 1 ? b : 0))];
            for (int i = 0; i < 4; i++) {
                y[i] = 0;
                for (int j = 0; j < 4; j++) y[i] += cd(g.mre[4 * i + j], g.mim[4 * i + j]) * v[j];
            }
            for (int s = 0; s < 4; s++) A[(size_t)(r | (s & 2 ? b : 0)) * dim + (c | (s & 1 ? b : 0))] = y[s];
        }
}

int deposit(int v, uint32_t mask)
{
    int out = 0;
    for (uint32_t m = mask; m; m &= m - 1, v >>= 1)
        if (v & 1) out |= (int)(m & (~m + 1));
    return out;
}

// One stage on every tile of the block on qmask.
void stage(Mat& A, int n, uint32_t qmask, const dmx::FusedStage& st)
{
    std::vector<cd> S(256);
    for (int i = 0; i < 256; i++) S[i] = cd(st.re[i], st.im[i]);
    std::vector<uint32_t> q;
    for (int b = n - 1; b >= 0; b--)
        if ((qmask >> b) & 1u) q.push_back((uint32_t)b);
    if (st.whole) {
        unitary(A, n, q, S);
        return;
    }
    const int dim = 1 << n;
    auto bits = [&](int lo, int hi, int v) { return (v & 1) << lo | (v >> 1) << hi; };
    for (int r0 = 0; r0 < dim; r0++)
        for (int c0 = 0; c0 < dim; c0++) {
            if ((r0 & qmask) || (c0 & qmask)) continue;
            for (int sp = 0; sp < 16; sp++) {
                cd v[16];
                auto at = [&](int s) -> cd& {
                    const int r = bits(st.u, st.v, s >> 2) | bits(st.x, st.y, sp >> 2);
                    const int c = bits(st.u, st.v, s & 3) | bits(st.x, st.y, sp & 3);
                    return A[(size_t)(r0 | deposit(r, qmask)) * dim + (c0 | deposit(c, qmask))];
                };
                for (int s = 0; s < 16; s++) v[s] = at(s);
                for (int i = 0; i < 16; i++) {
                    cd y = 0;
                    for (int j = 0; j < 16; j++) y += S[16 * i + j] * v[j];
                    at(i) = y;
                }
            }
        }
}

}  // namespace

int main()
{
    int cases = 0, folded = 0, whole = 0;
    for (int n = 4; n <= 7; n++)
        for (int seed = 0; seed < 12; seed++) {
            std::mt19937 rng(1000 * n + seed);
            std::normal_distribution<double> g01(0.0, 1.0);
            auto pick = [&](int k) {
                std::vector<uint32_t> q;
                while ((int)q.size() < k) {
                    const uint32_t b = rng() % n;
                    bool seen = false;
                    for (uint32_t o : q) seen = seen || o == b;
                    if (!seen) q.push_back(b);
                }
                return q;
            };
            const int per_channel = 1 + seed % 4;  // every member to every fourth a channel
            std::vector<Gate> circ;
            for (int i = 0; i < 40; i++) {
                Gate g;
                if ((int)(rng() % (per_channel + 1)) == 0) {
                    g.op = dmx::OP_KRAUS;
                    g.qb[0] = rng() % n;
                    g.mre.resize(32), g.mim.resize(32);
                    for (int t = 0; t < 32; t++) g.mre[t] = 0.3 * g01(rng), g.mim[t] = 0.3 * g01(rng);
                } else {
                    const int ops[] = {dmx::OP_U3, dmx::OP_H, dmx::OP_CX, dmx::OP_CX, dmx::OP_SWAP,
                                       dmx::OP_X, dmx::OP_CU1, dmx::OP_RYY, dmx::OP_CCX, dmx::OP_C3X};
                    g.op = ops[rng() % (seed % 3 == 0 ? 10 : 8)];
                    g.theta = g01(rng), g.phi = g01(rng), g.lambda = g01(rng);
                    const std::vector<uint32_t> q = pick(dmx::op_arity(g.op));
                    for (size_t j = 0; j < q.size(); j++) g.qb[j] = q[j];
                }
                circ.push_back(g);
            }
            const int dim = 1 << n;
            Mat A((size_t)dim * dim);
            for (cd& v : A) v = cd(g01(rng), g01(rng));
            Mat W = A;
            for (const Gate& g : circ) {
                if (g.op == dmx::OP_KRAUS) {
                    channel(W, n, g);
                    continue;
                }
                int k = 0;
                std::vector<uint32_t> q;
                std::vector<double> re, im;
                dmx::gate_matrix(g, k, q, re, im);
                std::vector<cd> G(re.size());
                for (size_t i = 0; i < re.size(); i++) G[i] = cd(re[i], im[i]);
                unitary(W, n, q, G);
            }
            dmx::BlockPlan bp;
            bool fusable = false;
            if (dmx::plan_blocks(circ, n, 1 + seed % 5, bp, fusable, seed % 2, false, nullptr, nullptr,
                                 true) || !fusable)
                return std::printf("FAIL plan n=%d seed=%d\n", n, seed), 1;
            for (const auto& o : bp.order) {
                if (o.first != 0) return std::printf("FAIL step kind n=%d seed=%d\n", n, seed), 1;
                const dmx::FusedBlock& b = bp.blocks[o.second];
                if (b.stages == 0) {
                    dmx::FusedStage st;
                    st.whole = 1;
                    std::memcpy(st.re, b.ur, sizeof(st.re));
                    std::memcpy(st.im, b.ui, sizeof(st.im));
                    stage(A, n, b.qmask, st);
                }
                if ((size_t)b.stage0 + b.stages > bp.stages.size())
                    return std::printf("FAIL records n=%d seed=%d\n", n, seed), 1;
                for (uint32_t i = 0; i < b.stages; i++) {
                    const dmx::FusedStage& st = bp.stages[b.stage0 + i];
                    if (!st.whole && ((1u << st.u) | (1u << st.v) | (1u << st.x) | (1u << st.y)) != 15u)
                        return std::printf("FAIL bits n=%d seed=%d\n", n, seed), 1;
                    stage(A, n, b.qmask, st);
                    folded++;
                    whole += st.whole;
                }
                if (b.perm_on) {
                    Mat P((size_t)dim * dim);
                    auto pi = [&](int x) {
                        uint32_t y = b.perm_b;
                        for (int q = 0; q < n; q++)
                            if ((x >> q) & 1) y ^= b.perm_L[q];
                        return y;
                    };
                    for (int r = 0; r < dim; r++)
                        for (int c = 0; c < dim; c++) P[(size_t)pi(r) * dim + pi(c)] = A[(size_t)r * dim + c];
                    A.swap(P);
                }
            }
            double err = 0, big = 0;
            for (size_t i = 0; i < A.size(); i++) {
                err = std::max(err, std::abs(A[i] - W[i]));
                big = std::max(big, std::abs(W[i]));
            }
            if (!(err <= 1e-11 * big)) return std::printf("FAIL result n=%d seed=%d: %g of %g\n", n, seed, err, big), 1;
            cases++;
        }
    if (folded < 200 || whole == 0) return std::printf("FAIL coverage %d %d\n", folded, whole), 1;
    std::printf("%d cases OK\n", cases);
    return 0;
}
