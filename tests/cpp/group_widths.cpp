// Stage widths of group plans (dmx::build_fused_plan with group): no unitary acts on more
// qubits than the fusion width allows or its widest gate has, no superoperator on two
// where the width is one.  Prints "<cases> cases OK", or the first violation.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <memory>
#include <random>
#include <vector>

#include "fuse.hpp"
#include "lower.hpp"

using dmx::Gate;

namespace {

// The qubits on which the d x d matrix (re, im) is not the identity: bit b counts unless
// M = M' (x) 1 there.
int support(const double* re, const double* im, int d)
{
    int count = 0;
    for (int b = 1; b < d; b <<= 1) {
        bool plain = true;
        for (int i = 0; i < d; i++)
            for (int j = 0; j < d; j++) {
                const int x = i * d + j, y = (i ^ b) * d + (j ^ b);
                if ((i & b) != (j & b))
                    plain = plain && re[x] == 0 && im[x] == 0;
                else
                    plain = plain && std::abs(re[x] - re[y]) < 1e-12 && std::abs(im[x] - im[y]) < 1e-12;
            }
        count += plain ? 0 : 1;
    }
    return count;
}

}  // namespace

int main()
{
    int cases = 0, fives = 0;
    for (int wide = 0; wide < 2; wide++)
        for (int noise = wide ? 0 : 1; noise < 2; noise++)
            for (int k = 1; k <= 5; k++) {
                const int n = 13;
                std::mt19937 rng(100 * wide + 10 * noise + k);
                std::vector<Gate> c;
                int widest = 2;
                for (int g = 0; g < 60; g++) {
                    Gate x;
                    const int ops[] = {dmx::OP_U3, dmx::OP_RZZ, dmx::OP_RXX, dmx::OP_U3, dmx::OP_RYY, dmx::OP_C4X};
                    x.op = ops[wide && g % 20 == 7 ? 5 : rng() % 5];
                    widest = std::max(widest, dmx::op_arity(x.op));
                    std::vector<uint32_t> q(n);
                    for (int i = 0; i < n; i++) q[i] = (uint32_t)i;
                    std::shuffle(q.begin(), q.end(), rng);
                    for (int j = 0; j < dmx::op_arity(x.op); j++) x.qb[j] = q[j];
                    x.theta = 0.1 * (g + 1), x.phi = 0.4, x.lambda = 0.7;
                    c.push_back(x);
                    if (noise && g % 9 == 4) {
                        Gate e;
                        e.op = dmx::OP_KRAUS;
                        e.qb[0] = q[0];
                        e.mre.assign(16, 0.0), e.mim.assign(16, 0.0);
                        for (int i = 0; i < 4; i++) e.mre[5 * i] = i % 3 ? 0.9 : 1.0;
                        c.push_back(e);
                    }
                }
                dmx::FusedPlan* p = nullptr;
                dmx::PlanInfo info;
                if (dmx::build_fused_plan(c, n, k, nullptr, 0, true, &p, &info, true, true, true) || !p)
                    return std::printf("FAIL plan\n"), 1;
                std::unique_ptr<dmx::FusedPlan> hold(p);
                std::vector<dmx::PlanStepView> steps;
                p->describe(steps);
                for (const auto& v : steps) {
                    if (v.kind != dmx::PlanStepView::GROUP) continue;
                    for (uint32_t i = v.group->stage0; i < v.group->stage0 + v.group->stages; i++) {
                        const dmx::GroupStage& s = v.gstages[i];
                        const int bits = s.kind == dmx::GS_UNITARY5 ? 5 : 4, d = 1 << bits;
                        int on = support(v.gmats + s.mat, v.gmats + s.mat + d * d, d);
                        if (s.kind == dmx::GS_PAIR)  // index 4 * row bits + column bits: a qubit has two
                            on = (on + 1) / 2;
                        fives += s.kind == dmx::GS_UNITARY5 ? 1 : 0;
                        if (on > std::max(k, widest))
                            return std::printf("FAIL wide %d noise %d k %d: a stage on %d\n", wide, noise, k, on), 1;
                        if (!wide && k < 5 && s.kind == dmx::GS_UNITARY5)
                            return std::printf("FAIL wide %d noise %d k %d: five\n", wide, noise, k), 1;
                    }
                }
                cases++;
            }
    if (!fives) return std::printf("FAIL coverage\n"), 1;
    std::printf("%d cases OK\n", cases);
    return 0;
}
