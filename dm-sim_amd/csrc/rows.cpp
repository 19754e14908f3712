// rows.cpp -- programs of the resident-row plain method (rows.hpp, host side).
#include "rows.hpp"

#include <algorithm>
#include <cstring>

namespace dmx {

// More entries per thread mean fewer regroups but longer steps.  Up to 9
// qubits a run is one wave's chain of steps long whatever their number (256
// rows of 8 qubits on 1024 SIMDs), so steps are short; from 10 the waves
// share the SIMDs.  Fastest of 2, 3 and 4 register bits on random and
// hardware-efficient circuits (400 gates up to 10 qubits, 200 above, us a
// run): 8 qubits 301/240 against 360/287 with three; 9: 384/299 (1024 entries
// a workgroup) against 398/319; 10: 504/454 with three against 589/542 and
// 616/501; 11: 872/703 against 1084/932 and 1036/841; 13: 13876/11757 with
// three, 14608/11470 with four.
RowShape row_shape(int n)
{
    if (n <= 8) return {2, 8, false};
    if (n == 9) return {2, 10, false};
    if (n <= 13) return {3, n, false};
    return {4, 14, true};
}

namespace {

// Consecutive primitives and the register bits they need: C2 operands as
// pairs (high, low) on neighbouring register bits, other targets anywhere.
struct RowGroup {
    std::vector<std::pair<int, int>> pairs;
    std::vector<int> singles;
    size_t first = 0, last = 0;

    bool has(int q) const
    {
        for (const auto& p : pairs)
            if (p.first == q || p.second == q) return true;
        return std::find(singles.begin(), singles.end(), q) != singles.end();
    }

    // Takes the register bits of primitive p if they fit into k; false (and
    // unchanged) if they do not.
    bool take(const PrimOp& p, int k)
    {
        if (p.kind == PK_C2) {
            for (const auto& pr : pairs)
                if (pr.first == p.q0 && pr.second == p.q1) return true;
            for (const auto& pr : pairs)
                for (int q : {p.q0, p.q1})
                    if (pr.first == q || pr.second == q) return false;
            std::vector<int> rest;
            for (int q : singles)
                if (q != p.q0 && q != p.q1) rest.push_back(q);
            if (2 * (pairs.size() + 1) + rest.size() > (size_t)k) return false;
            pairs.push_back({p.q0, p.q1});
            singles = rest;
            return true;
        }
        if (pos1_only(p.kind) || has(p.q0)) return true;
        if (2 * pairs.size() + singles.size() >= (size_t)k) return false;
        singles.push_back(p.q0);
        return true;
    }
};

}  // namespace

size_t build_row_program(const std::vector<PrimOp>& prims, size_t first, size_t last, int n,
                         std::vector<RowOp>& out)
{
    const RowShape sh = row_shape(n);
    const int s = sh.split ? 4 : 3;
    const size_t start = out.size();
    for (size_t at = first; at < last;) {
        RowGroup g;
        g.first = at;
        while (at < last && g.take(prims[at], sh.k)) at++;
        g.last = at;
        // register bits: pairs first, then singles, then free bits to fill up,
        // taken from the residue class (mod s) that has the most left
        int reg[4] = {-1, -1, -1, -1};
        uint32_t used = 0;
        int nr = 0;
        for (const auto& p : g.pairs) {
            reg[nr++] = p.second;
            reg[nr++] = p.first;
        }
        for (int q : g.singles) reg[nr++] = q;
        for (int i = 0; i < nr; i++) used |= 1u << reg[i];
        auto left = [&](int cls) {
            int c = 0;
            for (int b = cls; b < sh.loge; b += s) c += !((used >> b) & 1u);
            return c;
        };
        auto fullest = [&](uint32_t skip) {
            int best = -1;
            for (int cls = 0; cls < s; cls++)
                if (!((skip >> cls) & 1u) && left(cls) > 0 && (best < 0 || left(cls) > left(best)))
                    best = cls;
            return best;
        };
        auto take_bit = [&](int cls) {
            int b = cls;
            while ((used >> b) & 1u) b += s;
            used |= 1u << b;
            return b;
        };
        while (nr < sh.k) reg[nr++] = take_bit(fullest(0));
        // thread bits: runs of s of them with distinct residues
        std::vector<int> thr;
        uint32_t run = 0;
        while ((int)thr.size() < sh.loge - sh.k) {
            int cls = fullest(run);
            if (cls < 0) {
                run = 0;
                cls = fullest(0);
            }
            run |= 1u << cls;
            if (run == (1u << s) - 1) run = 0;
            thr.push_back(take_bit(cls));
        }
        RowOp rg = {};
        rg.code = RC_REGROUP;
        for (int i = 0; i < sh.k; i++) rg.w[i] = row_place(1u << reg[i], s, sh.loge);
        for (int i = 0; i < (int)thr.size(); i++) rg.w[4 + i] = row_place(1u << thr[i], s, sh.loge);
        out.push_back(rg);
        auto reg_of = [&](int q) {
            for (int i = 0; i < sh.k; i++)
                if (reg[i] == q) return i;
            return -1;
        };
        auto thread_bit = [&](int q) {
            return 1u << (std::find(thr.begin(), thr.end(), q) - thr.begin());
        };
        for (size_t i = g.first; i < g.last; i++) {
            const PrimOp& p = prims[i];
            RowOp op = {};
            std::memcpy(op.w, p.c, sizeof(op.w));
            const int t = reg_of(p.q0);
            if (p.kind == PK_C2) {
                RowOp skip = {};
                skip.code = RC_SKIP;
                while ((out.size() - start) % kRowChunk > kRowChunk - 4) out.push_back(skip);
                op.code = RC_C2 + (uint32_t)(t / 2);
                for (int r = 0; r < 3; r++) {
                    out.push_back(op);
                    op.code = RC_SKIP;
                    std::memcpy(op.w, p.c + 8 * (r + 1), sizeof(op.w));
                }
            } else if (pos1_only(p.kind)) {
                op.code = RC_DIAG + 8 * (uint32_t)(p.kind - PK_Z) + (t < 0 ? 4u : (uint32_t)t);
                if (t < 0) op.on = thread_bit(p.q0);
            } else if (p.q1 >= 0 && reg_of(p.q1) >= 0) {
                op.code = RC_CX + 4 * (uint32_t)t + (uint32_t)reg_of(p.q1);
            } else {
                op.code = RC_DENSE + 4 * (uint32_t)p.kind + (uint32_t)t;
                if (p.q1 >= 0) op.on = thread_bit(p.q1);
            }
            out.push_back(op);
        }
    }
    const RowOp end = {};
    out.insert(out.end(), 1 + 3 * kRowChunk, end);
    return start;
}

}  // namespace dmx
