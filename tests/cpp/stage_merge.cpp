// Channel-free stages of a block with channels (dmx::plan_blocks with fold): a run of
// superoperators of two qubits, 16 matrix instructions each, becomes one unitary of the
// block, 24, from two on; a single one stays.  Prints "OK" or what differs.
#include <cstdio>
#include <vector>

#include "fuse.hpp"
#include "lower.hpp"

using dmx::Gate;

int main()
{
    auto gate = [](int op, uint32_t a, uint32_t b) {
        Gate g;
        g.op = op;
        g.qb[0] = a, g.qb[1] = b;
        g.theta = 0.3, g.phi = 0.2, g.lambda = 0.1;
        return g;
    };
    Gate noise;
    noise.op = dmx::OP_KRAUS;
    noise.qb[0] = 0;
    noise.mre.assign(16, 0.0), noise.mim.assign(16, 0.0);
    for (int i = 0; i < 4; i++) noise.mre[5 * i] = i % 3 ? 0.9 : 1.0;
    for (int pairs = 1; pairs <= 3; pairs++) {
        std::vector<Gate> c = {gate(dmx::OP_RZZ, 0, 1), noise, gate(dmx::OP_RXX, 1, 2)};
        if (pairs > 1) c.push_back(gate(dmx::OP_RZZ, 2, 3));
        if (pairs > 2) c.push_back(gate(dmx::OP_RXX, 3, 1));
        dmx::BlockPlan bp;
        bool fusable = false;
        if (dmx::plan_blocks(c, 4, 4, bp, fusable, false, false, nullptr, nullptr, true) || !fusable ||
            bp.blocks.size() != 1)
            return std::printf("plan of %d pairs\n", pairs), 1;
        std::vector<int> whole;
        for (const dmx::FusedStage& s : bp.stages) whole.push_back((int)s.whole);
        const std::vector<int> want = pairs == 1 ? std::vector<int>{0, 0} : std::vector<int>{0, 1};
        if (whole != want) return std::printf("%d pairs: %zu stages\n", pairs, whole.size()), 1;
    }
    std::printf("OK\n");
    return 0;
}
