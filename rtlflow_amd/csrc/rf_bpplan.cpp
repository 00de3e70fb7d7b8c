// rf_bpplan.cpp -- the bit-plane planner as the compiler's host library
// (rtlflow_amd/bitplane.py, plan): a design's plans are written into its
// library beside the blob they are made from.
#include "rf_bpplan.h"

#include <cstring>
#include <exception>

namespace {
// sec: word offsets of {inputs, state, levels M, gates M, commit M, hash M,
// ports M} (rtlflow_amd.bitplane.sections).
bpplan::Source source(const uint32_t* b, const uint32_t* sec) {
    bpplan::Source s{};
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
    return s;
}
}  // namespace

// The plan of program M for ``threads`` threads, at most ``cap`` words of it
// into ``out``. Returns its words; 0: none better than the program's own
// records.
extern "C" uint64_t rf_bpplan_make(const uint32_t* blob, const uint32_t* sec, uint32_t threads, uint32_t* out,
                                   uint64_t cap) {
    try {
        const bpplan::Plan p = bpplan::Planner(source(blob, sec), threads, bpplan::max_rounds(threads)).run();
        if (!p.ok || !p.classed || !p.nr) return 0;
        const std::vector<uint32_t> w = bpplan::pack(p, threads);
        memcpy(out, w.data(), 4 * (w.size() < cap ? w.size() : cap));
        return w.size();
    } catch (const std::exception&) {
        return 0;
    }
}

// Whether ``words`` are a plan of the program that the runtime takes.
extern "C" int rf_bpplan_check(const uint32_t* blob, const uint32_t* sec, uint32_t threads, const uint32_t* words,
                               uint64_t n) {
    return bpplan::check(source(blob, sec), threads, words, n);
}
