// CPU model of the gate-net engine's LDS kernel: plans a program blob with
// rf_gnplan.h for planes of ``pb`` bytes and runs the wavefront programs over
// them, one stimulus at a time (one byte a plane: the plan's addresses divided
// by its width). Built by tests/test_gnplan.py with the host compiler.
#include <cstdlib>
#include <cstring>
#include <new>
#include <vector>

#include "rf_gnplan.h"

// Allocations left before one fails (negative: none does). Linked
// -Bsymbolic, so only this file's allocations come here.
static long g_left = -1;
void* operator new(size_t n) {
    if (g_left >= 0 && g_left-- == 0) throw std::bad_alloc();
    if (void* p = malloc(n ? n : 1)) return p;
    throw std::bad_alloc();
}
void operator delete(void* p) noexcept { free(p); }
void operator delete(void* p, size_t) noexcept { free(p); }

using namespace gnplan;

namespace {
uint64_t mix(uint64_t x) {
    uint64_t z = x + 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}
uint32_t op(uint32_t m, uint32_t a, uint32_t b) {   // operator masks p, q, n
    const uint32_t t = m & 1 ? a & ~b : a;
    return (m & 2 ? t ^ b : t & b) ^ (m >> 2);
}
}  // namespace

// The plane width that plan_program chooses when its allocation ``left`` fails;
// *used: the allocations it made.
extern "C" uint32_t gnplan_width(const uint32_t* h, uint32_t nwaves, uint64_t lds_bytes, long left, long* used) {
    Plan p;
    g_left = left >= 0 ? left : 1l << 40;
    const long l0 = g_left;
    const uint32_t pb = plan_program(h, nwaves, lds_bytes, &p);
    *used = l0 - g_left;
    g_left = -1;
    return pb;
}

// info[0..6]: slots, state slots, levels, wavefront rows, rows evaluated,
// wavefront rows of a batch, live RAMs. Returns 0, 1 when the program is not planned, 2
// when a level's rows read a slot that the same level writes, 3 when the
// wavefronts' barriers differ, 4 when a batch's row position is wrong, 5 when a
// class's operator is, 6 when an address is no plane's.
extern "C" int gnplan_run(const uint32_t* h, uint32_t nwaves, uint32_t pb, uint64_t seed, const uint32_t* budgets,
                          uint32_t n, uint64_t* hashes, uint32_t* info) {
    Net net;
    if (!read_net(h, net)) return 1;
    Planner pl(net, nwaves);
    pl.schedule();
    const Plan p = pl.emit(pb);
    info[5] = p.batch;
    info[6] = p.n_ram_live;
    bool off = false;
    const auto at = [&](uint32_t address) {   // the plane's slot
        if (address % pb || address / pb >= p.nslots) off = true;
        return off ? 0u : address / pb;
    };
    info[0] = p.nslots;
    info[1] = p.nstate;
    info[2] = p.levels;
    info[3] = p.wave_rows;
    info[4] = 0;
    const uint32_t n_pi = h[H_PI], n_po = h[H_PO], depth = h[H_DEPTH], width = h[H_WIDTH], ab = h[H_ABITS];
    for (uint32_t s = 0; s < n; ++s) {
        std::vector<uint8_t> L(p.nslots, 0xa5);
        memset(L.data(), 0, p.nstate);
        std::vector<uint64_t> mem((size_t)h[H_RAMS] * depth, 0);
        uint64_t hash = 0xcbf29ce484222325ull;
        auto gen = [&](uint32_t c) {
            for (uint32_t i = 0; i < n_pi; ++i) {
                const uint64_t w = mix(seed ^ (s * 0x9E3779B97F4A7C15ull) ^ ((uint64_t)c << 8) ^ (i / 64));
                L[p.a0 + i] = (w >> (i % 64)) & 1;
            }
        };
        gen(0);
        for (uint32_t k = 0; budgets[s] && k <= budgets[s]; ++k) {
            std::vector<uint32_t> rj(nwaves, 0), ri(nwaves, 0);
            for (uint32_t level = 0; level < p.levels; ++level) {
                std::vector<uint8_t> written(p.nslots, 0), read(p.nslots, 0);
                for (uint32_t w = 0; w < nwaves; ++w) {
                    const uint32_t* wt = &p.words[4 * w];
                    for (bool bar = false; !bar;) {
                        if (rj[w] == wt[1]) {
                            if (level + 1 != p.levels) return 3;
                            break;
                        }
                        const uint32_t* d = &p.words[wt[0] + 4 * rj[w]++];
                        const uint32_t* ahead = &p.words[wt[0] + 4 * ((rj[w] - 1 + kUnroll) % wt[1])];
                        if (d[2] != ahead[3] || (((d[0] >> 3) & 511) && d[3] != ri[w])) return 4;
                        const uint32_t per = p.batch == 1 ? 64 : 128;
                        if (((d[0] >> 3) & 511) > 64 * p.batch) return 4;
                        const uint32_t cls = d[0] & 7, n = (d[0] >> 3) & 511;
                        bar = d[0] >> 31;
                        for (uint32_t i = 0; i < n; ++i) {
                            const uint32_t to = p.batch == 1 ? i : i / 128 * 128 + 2 * (i % 64) + i % 128 / 64;
                            const uint64_t row = p.rows[per * (size_t)(wt[2] + ri[w]) + to];
                            const uint32_t a = at(row & 0x3ffff), c = at((row >> 18) & 0x3ffff), b = at(row >> 46);
                            const uint32_t m = (row >> 36) & 63;
                            ++info[4];
                            read[a] = 1;
                            if (cls == kCopy) {
                                L[b] = L[a];
                                written[b] = 1;
                                continue;
                            }
                            read[b] = 1;
                            if (cls == kPair || cls == kMux) read[c] = 1;
                            uint32_t v = cls == kMux ? (L[a] ? L[b] : L[c]) : op(m & 7, L[a], L[b]);
                            if (cls >= kOp && (m & 7) != op_bits(cls - kOp)) return 5;
                            if (cls == kPair) v = op(m >> 3, v, L[c]);
                            const uint32_t to_slot = at(d[1] + i * pb);
                            L[to_slot] = v & 1;
                            written[to_slot] = 1;
                        }
                        ri[w] += (n + per - 1) / per;
                    }
                }
                for (uint32_t i = 0; i < p.nslots; ++i)
                    if (written[i] && read[i]) return 2;
            }
            for (uint32_t w = 0; w < nwaves; ++w)
                if (rj[w] != p.words[4 * w + 1]) return 3;
            if (k) {
                uint64_t v = 0;
                for (uint32_t i = 0; i < n_po; ++i) v |= (uint64_t)L[at(p.words[p.off_po + i])] << i;
                const int nb = n_po <= 8 ? 1 : n_po <= 16 ? 2 : n_po <= 32 ? 4 : 8;
                for (int i = 0; i < nb; ++i) hash = (hash ^ ((v >> (8 * i)) & 0xff)) * 0x100000001b3ull;
            }
            for (uint32_t r = 0; r < p.n_ram_live; ++r) {
                const uint32_t* rw = &p.words[p.off_ram + r * p.ram_words];
                uint64_t addr = 0, wd = 0;
                for (uint32_t i = 0; i < ab; ++i) addr |= (uint64_t)L[at(rw[2 + i])] << i;
                for (uint32_t i = 0; i < width; ++i) wd |= (uint64_t)L[at(rw[2 + ab + 1 + i])] << i;
                uint64_t* m = &mem[(size_t)rw[0] * depth];
                const uint64_t old = addr < depth ? m[addr] : 0;
                if (L[at(rw[2 + ab])] && addr < depth) m[addr] = wd;
                for (uint32_t i = 0; i < width; ++i) L[at(rw[1] + i * pb)] = (old >> i) & 1;
            }
            for (uint32_t i = 0; i < n_pi; ++i) L[p.b0 + i] = L[p.a0 + i];
            gen(k + 1);
        }
        if (off) return 6;
        hashes[s] = hash;
    }
    return 0;
}
