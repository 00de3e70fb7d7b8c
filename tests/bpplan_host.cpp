// CPU model of the planned per-cycle program of the bit-plane kernel: program
// M of a blob is evaluated from the same planes by its own records and by the
// plan of rf_bpplan.h, then both tables (commit, hash, ports). Built by
// tests/test_bpplan.py with the host compiler.
#include <cstring>
#include <vector>

#include "rf_bpplan.h"

using namespace bpplan;

namespace {
uint32_t ev(uint32_t x) { return x + (x & 1); }
uint64_t rd(const std::vector<uint64_t>& L, uint32_t ref) {
    const uint64_t v = L[ref & 0x7fffffffu];
    return ref >> 31 ? ~v : v;
}
}  // namespace

// Section offsets as tests compute them (rtlflow_amd.bitplane.sections): sec =
// {in, state, lev M, gates M, commit M, hash M, ports M}. out0 / out1:
// state planes after the commit, then every hash and port reference.
// info: rounds, wavefront rows, generic rows, rounds of the program as stated.
// Returns 0; 1 not planned; 2 a round reads what its level writes; 3 slots or
// rounds out of range; 4 rows of a classed wavefront carry inversions.
extern "C" int bpplan_run(const uint32_t* b, const uint32_t* sec, uint32_t threads, const uint64_t* planes,
                          uint64_t* out0, uint64_t* out1, uint32_t* info) {
    Source s{};
    s.blob = b;
    s.byte_form = (b[1] >> 16) != 0;
    s.nslots = b[2];
    s.n_in = b[3];
    s.n_state = b[4];
    s.n_hash = b[6];
    s.nlev = b[9];
    s.n_commit = b[16];
    s.off_in = sec[0];
    s.off_state = sec[1];
    s.off_lev = sec[2];
    s.off_gates = sec[3];
    s.off_commit = sec[4];
    s.off_hash = sec[5];
    s.off_ports = sec[6];
    const Plan p = Planner(s, threads, 48).run();
    info[3] = 0;
    for (uint32_t l = 0; l < s.nlev; ++l) info[3] += (b[s.off_lev + l + 1] - b[s.off_lev + l] + threads - 1) / threads;
    if (!p.ok) return 1;
    info[0] = p.nr;
    info[1] = p.rows;
    info[2] = p.generic;
    const auto fields = [&](const uint32_t* g, uint32_t* f) {   // dst, s, x, ix, y, iy
        if (s.byte_form) {
            f[0] = (g[0] & 0xffff) / 8, f[1] = (g[0] >> 16) / 8, f[2] = (g[1] & 0xfff8) / 8, f[3] = g[1] & 1;
            f[4] = ((g[1] >> 16) & 0xfff8) / 8, f[5] = (g[1] >> 16) & 1;
        } else {
            f[0] = g[0] & 0xffff, f[1] = g[0] >> 16, f[2] = g[1] & 0x7fff, f[3] = (g[1] >> 15) & 1;
            f[4] = (g[1] >> 16) & 0x7fff, f[5] = g[1] >> 31;
        }
    };
    const auto finish = [&](std::vector<uint64_t>& L, const uint32_t* com, uint32_t nc, const uint32_t* h,
                            const uint32_t* q, uint64_t* out) {
        std::vector<uint64_t> refs;
        for (uint32_t k = 0, o = 0; k < s.n_hash; ++k, o += 2 + h[o + 1])
            for (uint32_t i = 0; i < h[o + 1]; ++i) refs.push_back(rd(L, h[o + 2 + i]));
        const uint32_t np = q[1];
        q += 2;
        for (uint32_t r = 0; r < np; ++r) {
            const uint32_t n = q[0] == 0 ? q[2] : 1 + q[2] + q[3];
            for (uint32_t i = 0; i < n; ++i) refs.push_back(rd(L, q[4 + i]));
            q += (q[0] == 0 ? 4 : 5) + q[2] + q[3];
        }
        std::vector<uint64_t> next(nc);
        for (uint32_t k = 0; k < nc; ++k) next[k] = rd(L, com[2 * k + 1]);
        for (uint32_t k = 0; k < nc; ++k) L[com[2 * k]] = next[k];
        for (uint32_t k = 0; k < s.n_state; ++k) {
            const uint32_t* sl = b + s.off_state + 6 * k;
            for (uint32_t i = 0; i < sl[4]; ++i) *out++ = L[sl[5] + i];
        }
        for (uint64_t v : refs) *out++ = v;
    };
    std::vector<uint64_t> A(planes, planes + s.nslots), B = A;
    for (uint32_t k = 0; k < b[s.off_lev + s.nlev]; ++k) {   // levels in order: no level reads its own writes
        uint32_t f[6];
        fields(b + s.off_gates + 2 * k, f);
        const uint64_t x = f[3] ? ~A[f[2]] : A[f[2]], y = f[5] ? ~A[f[4]] : A[f[4]];
        A[f[0]] = (A[f[1]] & x) | (~A[f[1]] & y);
    }
    finish(A, b + s.off_commit, s.n_commit, b + s.off_hash, b + s.off_ports, out0);
    if (p.nr > 48) return 3;
    std::vector<uint8_t> wr(s.nslots, 0), re(s.nslots, 0);
    for (uint32_t r = 0; r < p.nr; ++r) {
        for (uint32_t t = 0; t < threads; ++t) {
            uint32_t cls = 0, f[6];
            for (uint32_t k = 0; k < 4; ++k) cls |= (uint32_t)((p.cls[4 * (t / 64) + k] >> r) & 1) << k;
            if (!(cls & 8)) continue;
            cls &= 7;
            fields(&p.recs[((size_t)r * threads + t) * 2], f);
            if (f[0] >= s.nslots || f[1] >= s.nslots || f[2] >= s.nslots || f[4] >= s.nslots) return 3;
            if (cls != GENERIC && (f[3] || f[5])) return 4;
            const uint64_t S = B[f[1]], X = f[3] ? ~B[f[2]] : B[f[2]], Y = f[5] ? ~B[f[4]] : B[f[4]];
            re[f[1]] = re[f[2]] = 1;
            if (cls >= MUX) re[f[4]] = 1;
            uint64_t v;
            switch (cls) {
                case AND: v = S & X; break;
                case ANDN: v = S & ~X; break;
                case NOR: v = ~(S | X); break;
                case XOR: v = S ^ X; break;
                case MUXN: v = (S & ~X) | (~S & Y); break;
                default: v = (S & X) | (~S & Y);
            }
            if (wr[f[0]] && B[f[0]] != v) return 2;
            B[f[0]] = v;
            wr[f[0]] = 1;
        }
        if ((p.bar >> r) & 1) {
            for (uint32_t i = 0; i < s.nslots; ++i)
                if (wr[i] && re[i]) return 2;
            std::fill(wr.begin(), wr.end(), 0);
            std::fill(re.begin(), re.end(), 0);
        }
    }
    finish(B, p.commit.data(), (uint32_t)p.commit.size() / 2, p.hash.data(), p.ports.data(), out1);
    return 0;
}
