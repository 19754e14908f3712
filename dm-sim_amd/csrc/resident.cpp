// resident.cpp -- records of the resident block executor (resident.hpp).
#include "resident.hpp"

#include <cstring>
#include <utility>

namespace dmx {

void build_resident(const std::vector<FusedBlock>& blocks, const std::vector<int>& order, int n,
                    std::vector<ResidentPart>& parts, ResidentEnd& end)
{
    const int L = resident_log_entries(n);
    auto place = [&](uint32_t x) { return row_place(x, 3, L); };
    // logical index x of a row is held as entry (xor of col[q] over x's bits) ^ off
    uint32_t col[kResidentMaxQubits], off = 0;
    for (int q = 0; q < n; q++) col[q] = 1u << q;
    parts.clear();
    parts.reserve(order.size() * kResidentParts * 64);
    for (const int index : order) {
        const FusedBlock& fb = blocks[index];
        uint32_t b[4], rest[kResidentMaxQubits];
        int nb = 0, nr = 0;
        for (int q = 0; q < n; q++) {
            if ((fb.qmask >> q) & 1u)
                b[nb++] = place(col[q]);
            else
                rest[nr++] = place(col[q]);
        }
        for (int q = n; q < L; q++) rest[nr++] = place(1u << q);
        // Lane bits 0..2 are to differ on the banks (8 places of 16 bytes): bits
        // with new residues first.
        uint32_t span = 1;  // residues reached so far, as a set
        for (int i = 0; i < 3; i++) {
            for (int r = i; r < nr; r++)
                if (!((span >> (rest[r] & 7u)) & 1u)) {
                    std::swap(rest[r], rest[i]);
                    break;
                }
            uint32_t more = span;
            for (uint32_t s = 0; s < 8; s++)
                if ((span >> s) & 1u) more |= 1u << (s ^ (rest[i] & 7u));
            span = more;
        }
        const uint32_t base = place(off);
        const size_t at = parts.size();
        parts.resize(at + kResidentParts * 64);
        ResidentPart* const rec = parts.data() + at;
        for (int lane = 0; lane < 64; lane++) {
            const int j = lane & 15, k = lane >> 4;
            for (int c = 0; c < 4; c++) {
                rec[(c / 2) * 64 + lane].u[c % 2] = fb.ur[16 * j + 4 * c + k];
                rec[(2 + c / 2) * 64 + lane].u[c % 2] = fb.ui[16 * j + 4 * c + k];
            }
            uint32_t x = base;
            for (int i = 0; i < 4; i++)
                if ((j >> i) & 1) x ^= rest[i];
            for (int i = 0; i < 2; i++)
                if ((k >> i) & 1) x ^= b[i];
            ResidentPart& p = rec[4 * 64 + lane];
            std::memset(&p, 0, sizeof(p));
            p.place.at = (uint16_t)x;
            p.place.c0 = (uint16_t)b[2];
            p.place.c1 = (uint16_t)b[3];
            if (nr > 4) p.place.t0 = (uint16_t)rest[4];
            if (nr > 5) p.place.t1 = (uint16_t)rest[5];
            if (nr > 6) p.place.t2 = (uint16_t)rest[6];
        }
        if (!fb.perm_on) continue;
        // The permutation sends x to L x + perm_b: from here on index y is what
        // L^-1 (y + perm_b) was.  L^-1 by elimination on (L, col) column by column.
        uint32_t lin[kResidentMaxQubits], im[kResidentMaxQubits];
        for (int q = 0; q < n; q++) {
            lin[q] = fb.perm_L[q];
            im[q] = col[q];
        }
        for (int q = 0; q < n; q++) {
            int p = q;
            while (p < n - 1 && !((lin[p] >> q) & 1u)) p++;
            std::swap(lin[p], lin[q]);
            std::swap(im[p], im[q]);
            for (int r = 0; r < n; r++)
                if (r != q && ((lin[r] >> q) & 1u)) {
                    lin[r] ^= lin[q];
                    im[r] ^= im[q];
                }
        }
        for (int q = 0; q < n; q++) {
            col[q] = im[q];
            if ((fb.perm_b >> q) & 1u) off ^= col[q];
        }
    }
    std::memset(&end, 0, sizeof(end));
    end.base = place(off);
    for (int q = 0; q < L; q++) end.bit[q] = place(q < n ? col[q] : 1u << q);
}

}  // namespace dmx
