// The resident-row programs (dm-sim_amd/csrc/rows.hpp), executed on the CPU
// thread by thread with the kernel's own step functions: at every regroup each
// of the workgroup's LDS places belongs to exactly one (thread, register
// entry), and the rows afterwards equal, bit for bit, the primitives applied
// one after the other to each row.
#include <cstdio>
#include <cstring>
#include <random>
#include <vector>

#include "rows.hpp"

using namespace dmx;

namespace {

template <int KIND>
void pair_sweep(const PrimOp& p, int n, double* re, double* im)
{
    for (uint32_t x = 0; x < (1u << n); x++) {
        if ((x >> p.q0) & 1u) continue;
        if (p.q1 >= 0 && !((x >> p.q1) & 1u)) continue;
        const uint32_t y = x | (1u << p.q0);
        double r0 = re[x], i0 = im[x], r1, i1;
        if (!pos1_only(KIND)) out0<KIND>(p.c, re[x], im[x], re[y], im[y], r0, i0);
        out1<KIND>(p.c, re[x], im[x], re[y], im[y], r1, i1);
        re[x] = r0, im[x] = i0, re[y] = r1, im[y] = i1;
    }
}

void apply(const PrimOp& p, int n, double* re, double* im)
{
    switch (p.kind) {
#define CASE(K) case K: pair_sweep<K>(p, n, re, im); return;
        CASE(PK_C1) CASE(PK_X) CASE(PK_Y) CASE(PK_H) CASE(PK_SRN) CASE(PK_RX) CASE(PK_RY) CASE(PK_W)
        CASE(PK_Z) CASE(PK_S) CASE(PK_SDG) CASE(PK_T) CASE(PK_TDG) CASE(PK_R) CASE(PK_U1)
#undef CASE
    default: break;
    }
    for (uint32_t x = 0; x < (1u << n); x++) {
        if (((x >> p.q0) & 1u) || ((x >> p.q1) & 1u)) continue;
        double vr[4], vi[4];
        uint32_t at[4];
        for (uint32_t j = 0; j < 4; j++) {
            at[j] = x | ((j >> 1) << p.q0) | ((j & 1u) << p.q1);
            vr[j] = re[at[j]], vi[j] = im[at[j]];
        }
        row_c2<2, 0>([&](int i) { return p.c[i]; }, vr, vi);
        for (int j = 0; j < 4; j++) re[at[j]] = vr[j], im[at[j]] = vi[j];
    }
}

template <int K>
bool run(const std::vector<RowOp>& prog, size_t at, int loge, bool split, std::vector<double>& re,
         std::vector<double>& im)
{
    const int threads = 1 << (loge - K), per = 1 << K, s = split ? 4 : 3;
    const uint32_t entries = 1u << loge;
    std::vector<double> lr(entries), li(entries);
    for (uint32_t e = 0; e < entries; e++) lr[row_place(e, s, loge)] = re[e], li[row_place(e, s, loge)] = im[e];
    std::vector<double> vr(entries), vi(entries);
    std::vector<uint32_t> place(entries);
    bool held = false;
    const size_t start = at;
    for (;; at++) {
        if (at + 3 * kRowChunk >= prog.size()) return false;  // what the kernel may read ahead
        const RowOp& op = prog[at];
        if (op.code >= RC_COUNT) return false;
        if (op.code != RC_END && op.code != RC_REGROUP && !row_code_ok(K, op.code)) return false;
        if (op.code == RC_END || op.code == RC_REGROUP) {
            if (held)
                for (uint32_t e = 0; e < entries; e++) lr[place[e]] = vr[e], li[place[e]] = vi[e];
            if (op.code == RC_END) break;
            std::vector<int> seen(entries, 0);
            for (int t = 0; t < threads; t++) {
                uint32_t base = 0;
                for (int i = 0; i < loge - K; i++)
                    if ((t >> i) & 1) base ^= op.w[4 + i];
                for (int i = 0; i < per; i++) {
                    uint32_t x = base;
                    for (int b = 0; b < K; b++)
                        if ((i >> b) & 1) x ^= op.w[b];
                    if (x >= entries || seen[x]++) return false;
                    place[t * per + i] = x;
                    vr[t * per + i] = lr[x], vi[t * per + i] = li[x];
                }
            }
            held = true;
            continue;
        }
        if (!held) return false;
        const bool c2 = op.code - RC_C2 < 2u;
        if (c2 && (at - start) % kRowChunk > kRowChunk - 4) return false;
        auto coef = [&](int i) {
            double v;
            std::memcpy(&v, (&op)[i / 8].w + 2 * (i % 8), 8);
            return v;
        };
        for (int t = 0; t < threads; t++)
            row_step<K>(op.code, coef, ((uint32_t)t & op.on) == op.on, &vr[t * per], &vi[t * per]);
        if (c2) at += 3;
    }
    for (uint32_t e = 0; e < entries; e++) re[e] = lr[row_place(e, s, loge)], im[e] = li[row_place(e, s, loge)];
    return true;
}

}  // namespace

int main()
{
    int cases = 0;
    for (int n = 1; n <= kRowsMaxQubits; n++)
        for (int seed = 0; seed < 3; seed++) {
            std::mt19937_64 rng(100 * n + seed);
            std::uniform_real_distribution<double> u(-1, 1);
            // seed 0: every kind; 1: mostly 4x4 and controlled swaps; 2: one primitive
            std::vector<PrimOp> prims(seed == 2 ? 1 : n > 11 ? 60 : 150);
            for (PrimOp& p : prims) {
                std::memset(&p, 0, sizeof(p));
                for (double& c : p.c) c = u(rng);
                p.q0 = (int)(rng() % n);
                p.q1 = -1;
                const bool two = n > 1 && rng() % (seed == 1 ? 2 : 8) == 0;
                p.kind = two ? PK_C2 : (int)(rng() % (PK_U1 + 1));
                if (seed == 1 && !two && rng() % 2) p.kind = PK_X;
                if (p.kind == PK_C2 || (p.kind == PK_X && n > 1 && rng() % 3))
                    do p.q1 = (int)(rng() % n);
                    while (p.q1 == p.q0);
            }
            std::vector<RowOp> prog;
            build_row_program(prims, 0, prims.size() / 2, n, prog);
            const size_t at = build_row_program(prims, 0, prims.size(), n, prog);
            const RowShape sh = row_shape(n);
            const uint32_t entries = 1u << sh.loge;
            std::vector<double> re(entries), im(entries);
            for (uint32_t e = 0; e < entries; e++) re[e] = u(rng), im[e] = u(rng);
            std::vector<double> wr = re, wi = im;
            for (uint32_t row = 0; row < entries; row += 1u << n)
                for (const PrimOp& p : prims) apply(p, n, &wr[row], &wi[row]);
            bool ok = sh.loge >= n && sh.loge - sh.k <= 10;
            if (sh.k == 2)
                ok = ok && run<2>(prog, at, sh.loge, sh.split, re, im);
            else if (sh.k == 3)
                ok = ok && run<3>(prog, at, sh.loge, sh.split, re, im);
            else
                ok = ok && run<4>(prog, at, sh.loge, sh.split, re, im);
            if (!ok || std::memcmp(re.data(), wr.data(), 8 * entries) ||
                std::memcmp(im.data(), wi.data(), 8 * entries)) {
                printf("n = %d seed = %d: %s\n", n, seed, ok ? "rows differ" : "bad program");
                return 1;
            }
            cases++;
        }
    printf("%d cases OK\n", cases);
    return 0;
}
