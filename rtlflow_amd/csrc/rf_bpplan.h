// rf_bpplan.h -- planner of the bit-plane kernel's per-cycle program: program
// M of a blob (generic gate records, level by level) becomes rounds of
// wavefront rows. Plain C++ (no GPU), so the CPU tests run it. The design's
// build plans (rf_bpplan.cpp) and writes the plans beside the blob: planning
// takes about 0.6 us a gate (net2 5 ms), more than a plan saves in 10,000
// cycles, so no run pays for it. The runtime makes only the unplanned form
// (as_stated, a copy: 0.02 ms) itself, for workgroup sizes and libraries
// without a plan.
//
// The generic record dst = s ? (x ^ ix) : (y ^ iy) reads three planes and
// takes 12 VALU instructions whatever the gate is. Here 64 gates of one class
// form a wavefront row whose operators are scalar control flow: a two-input
// gate reads two planes and takes 5 VALU instructions, a multiplexer 6. The
// inversions go into the planes' polarity: a value is kept inverted when its
// class gives that, and the gates that read it are classed accordingly. Next
// states written in place keep the state's own polarity; a gate that would
// need its complement there, and the remainders of classes that do not fill a
// wavefront row when a level would otherwise take another round, stay generic
// records.
#pragma once
#include <stdint.h>

#include <algorithm>
#include <vector>

namespace bpplan {

// Classes of a wavefront row (operands s, x, y as the record's fields).
enum { AND = 0, ANDN = 1, NOR = 2, XOR = 3, MUX = 4, MUXN = 5, GENERIC = 6, CLASSES = 7 };
// s & x, s & ~x, ~(s | x), s ^ x, s ? x : y, s ? ~x : y, the generic record.

constexpr uint32_t kNone = 0xffffffffu;

// The sections of a blob the plan is made from (word offsets).
struct Source {
    const uint32_t* blob;
    bool byte_form;
    uint32_t nslots, n_in, off_in, n_state, off_state;
    uint32_t nlev, off_lev, off_gates;         // program M
    uint32_t n_commit, off_commit;             // after program M
    uint32_t n_hash, off_hash, off_ports;      // of program M
};

struct Plan {
    bool ok = false;
    bool classed = false;              // not just the program's own records
    uint32_t nr = 0;                   // rounds
    uint64_t bar = 0;                  // bit i: a barrier follows round i
    std::vector<uint32_t> recs;        // [round][thread] two words
    std::vector<uint64_t> cls;         // [wavefront][4]: bit i of word b < 3 is bit b of round i's class, of word 3: it has a row
    std::vector<uint32_t> commit;      // {state slot, source slot | inverted << 31}
    std::vector<uint32_t> hash, ports; // program M's tables with the plan's slots
    uint32_t rows = 0, generic = 0;    // wavefront rows, of which generic
};

// Rounds of register-resident records that the kernels of a workgroup size
// hold (rf_bitplane.hip).
inline uint32_t max_rounds(uint32_t threads) { return threads < 256 ? 0u : threads >= 1024 ? 40u : 48u; }

// A plan as words: this header, then at word kHdr the records, the classes,
// the commit pairs, the hash and the port tables (offsets from the start).
enum { P_MAGIC, P_THREADS, P_NR, P_BAR_LO, P_BAR_HI, P_CLS, P_COMMIT, P_NCOMMIT, P_HASH, P_PORTS, P_TOTAL };
constexpr uint32_t kHdr = 12, kMagic = 0x4c504252u;   // 'RBPL'
inline std::vector<uint32_t> pack(const Plan& p, uint32_t threads) {
    std::vector<uint32_t> w(kHdr, 0);
    w[P_MAGIC] = kMagic;
    w[P_THREADS] = threads;
    w[P_NR] = p.nr;
    w[P_BAR_LO] = (uint32_t)p.bar;
    w[P_BAR_HI] = (uint32_t)(p.bar >> 32);
    w.insert(w.end(), p.recs.begin(), p.recs.end());
    w[P_CLS] = (uint32_t)w.size();
    for (uint64_t c : p.cls) w.insert(w.end(), {(uint32_t)c, (uint32_t)(c >> 32)});
    w[P_COMMIT] = (uint32_t)w.size();
    w[P_NCOMMIT] = (uint32_t)p.commit.size() / 2;
    w.insert(w.end(), p.commit.begin(), p.commit.end());
    w[P_HASH] = (uint32_t)w.size();
    w.insert(w.end(), p.hash.begin(), p.hash.end());
    w[P_PORTS] = (uint32_t)w.size();
    w.insert(w.end(), p.ports.begin(), p.ports.end());
    w[P_TOTAL] = (uint32_t)w.size();
    return w;
}

// Whether words [w, w + n) are a plan of program M of ``s`` for ``threads``
// threads: every section inside, every slot a kernel addresses below nslots
// (a record's fields on rows that run, the tables' references), and tables of
// the program's own shape.
inline bool check(const Source& s, uint32_t threads, const uint32_t* w, uint64_t n) {
    if (n < kHdr || w[P_MAGIC] != kMagic || w[P_THREADS] != threads || w[P_TOTAL] != n || (n >> 31)) return false;
    const uint32_t nr = w[P_NR], nw = threads / 64;
    if (!nr || nr > max_rounds(threads) || w[P_CLS] != kHdr + (uint64_t)nr * threads * 2 ||
        w[P_COMMIT] != w[P_CLS] + (uint64_t)nw * 8 || w[P_HASH] != w[P_COMMIT] + 2ull * w[P_NCOMMIT] ||
        w[P_PORTS] < w[P_HASH] || w[P_PORTS] > n)
        return false;
    if (!((w[nr > 32 ? P_BAR_HI : P_BAR_LO] >> ((nr - 1) % 32)) & 1)) return false;   // the last round ends in a barrier
    for (uint32_t r = 0; r < nr; ++r)
        for (uint32_t v = 0; v < nw; ++v) {
            uint32_t cls = 0;
            for (uint32_t k = 0; k < 4; ++k) cls |= ((w[w[P_CLS] + 8 * v + 2 * k + r / 32] >> (r % 32)) & 1) << k;
            if (!(cls & 8)) continue;
            if ((cls & 7) >= CLASSES) return false;
            for (uint32_t t = 64 * v; t < 64 * v + 64; ++t) {
                const uint32_t* g = w + kHdr + 2 * ((uint64_t)r * threads + t);
                for (uint32_t k = 0; k < 4; ++k) {
                    uint32_t f = (g[k / 2] >> (16 * (k % 2))) & 0xffffu;
                    if (s.byte_form ? (k < 2 && (f & 7)) || (f >> 3) >= s.nslots
                                    : (k < 2 ? f : f & 0x7fffu) >= s.nslots)
                        return false;
                }
            }
        }
    const auto slot = [&](uint32_t ref) { return (ref & 0x7fffffffu) < s.nslots; };
    for (uint32_t k = 0; k < w[P_NCOMMIT]; ++k) {
        const uint32_t* c = w + w[P_COMMIT] + 2 * k;
        if (c[0] >= s.nslots || !slot(c[1])) return false;
    }
    const uint32_t *b = s.blob + s.off_hash, *h = w + w[P_HASH], *he = w + w[P_PORTS];
    for (uint32_t k = 0; k < s.n_hash; ++k) {
        if (he - h < (int64_t)b[1] + 2 || h[0] != b[0] || h[1] != b[1]) return false;
        for (uint32_t i = 0; i < b[1]; ++i)
            if (!slot(h[2 + i])) return false;
        h += 2 + b[1];
        b += 2 + b[1];
    }
    b = s.blob + s.off_ports;
    const uint32_t* q = w + w[P_PORTS];
    if (h != he || n - w[P_PORTS] != b[0] || q[0] != b[0] || q[1] != b[1]) return false;
    uint32_t at = 2;
    for (uint32_t r = 0; r < b[1]; ++r) {
        const uint32_t na = b[at + 2], n2 = b[at + 3], refs = b[at] == 0 ? na : 1 + na + n2;
        const uint32_t size = (b[at] == 0 ? 4u : 5u) + na + n2;
        for (uint32_t i = 0; i < size; ++i)
            if (i >= 4 && i < 4 + refs ? !slot(q[at + i]) : q[at + i] != b[at + i]) return false;
        at += size;
    }
    return true;
}

class Planner {
public:
    Planner(const Source& s, uint32_t threads, uint32_t rounds)
        : s_(s), nt_(threads), nw_(threads / 64), maxr_(rounds) {}

    // The plan of classed rows; when the program is not of the lowering's form
    // or its values need more slots than it has, its own records as generic
    // rows. Not ok: more rounds than the kernels hold.
    Plan run() {
        // (a round holds one gate per thread)
        if (s_.blob[s_.off_lev + s_.nlev] > (uint64_t)nt_ * maxr_) return Plan();
        if (parse() && tables()) {
            for (bool delay : {true, false}) {
                Plan p;
                set_levels(delay);
                if (least_rounds() > maxr_) continue;
                classify();
                if (!place(p)) continue;
                emit_tables(p);
                p.ok = p.classed = true;
                return p;
            }
        }
        return as_stated();
    }

    // The program's own records as generic rows: no more work than a copy.
    Plan as_stated() const {
        Plan p;
        const uint32_t* b = s_.blob;
        p.cls.assign((size_t)nw_ * 4, 0);
        for (uint32_t l = 0; l < s_.nlev; ++l) p.nr += (b[s_.off_lev + l + 1] - b[s_.off_lev + l] + nt_ - 1) / nt_;
        if (p.nr > maxr_) return Plan();
        p.recs.resize((size_t)p.nr * nt_ * 2, 0);
        uint32_t r = 0;
        for (uint32_t l = 0; l < s_.nlev; ++l) {
            const uint32_t lo = b[s_.off_lev + l], hi = b[s_.off_lev + l + 1];
            for (uint32_t k = lo; k < hi; k += nt_, ++r) {
                const uint32_t n = std::min(hi - k, nt_);
                uint32_t* rec = &p.recs[(size_t)r * nt_ * 2];
                std::copy_n(b + s_.off_gates + 2 * k, 2 * n, rec);
                for (uint32_t w = 0; 64 * w < n; ++w) {
                    mark(p, w, r, GENERIC);
                    p.rows++;
                    p.generic++;
                }
                // idle lanes repeat the last record
                for (uint32_t t = n; t % 64; ++t) std::copy_n(rec + 2 * (n - 1), 2, rec + 2 * t);
            }
            if (hi > lo) p.bar |= 1ull << (r - 1);
        }
        p.commit.assign(b + s_.off_commit, b + s_.off_commit + 2 * s_.n_commit);
        uint32_t o = s_.off_hash;
        for (uint32_t k = 0; k < s_.n_hash; ++k) o += 2 + b[o + 1];
        p.hash.assign(b + s_.off_hash, b + o);
        p.ports.assign(b + s_.off_ports, b + s_.off_ports + b[s_.off_ports]);
        p.ok = true;
        return p;
    }

private:
    enum Kind : uint8_t { LEAF, K_AND, K_XOR, K_MUX, K_COPY };
    struct Val {
        Kind kind = LEAF;
        uint32_t in[3] = {0, 0, 0};   // literals 2 * value + inverted
        uint32_t nin = 0, o = 0;      // o: the value is the inverted operator
        uint32_t level = 0, asap = 0, last = 0, readers = 0;
        uint32_t slot = kNone;
        uint32_t target = kNone;      // state slot written in place
        bool keep = false;            // read after the last level
        uint32_t states = kNone;      // state planes that take it: the first of takes_
        // class row
        uint8_t cls = 0, inv = 0, pol = 0;
        uint32_t s = 0, x = 0, y = 0;
    };
    struct Field {
        uint32_t dst, s, x, ix, y, iy;
    };
    struct Take {
        uint32_t slot, inv, next;   // state slot, inverted; the value's next one in takes_
    };
    void add_state(Val& v, uint32_t slot, uint32_t inv) {
        uint32_t* at = &v.states;   // (kept in the order added: the first that can be is written in place)
        while (*at != kNone) at = &takes_[*at].next;
        *at = (uint32_t)takes_.size();
        takes_.push_back({slot, inv, kNone});
    }

    uint32_t zero() const { return zero_; }
    uint32_t leaf(uint32_t slot) {
        if (cur_[slot] == kNone) {
            Val v;
            v.slot = slot;
            cur_[slot] = (uint32_t)v_.size();
            if (!slot) zero_ = cur_[slot];
            v_.push_back(v);
        }
        return cur_[slot];
    }
    Field field(uint32_t k) const {
        const uint32_t* g = s_.blob + s_.off_gates + 2 * k;
        if (s_.byte_form)
            return {(g[0] & 0xffffu) / 8, (g[0] >> 16) / 8, (g[1] & 0xfff8u) / 8, g[1] & 1u, ((g[1] >> 16) & 0xfff8u) / 8,
                    (g[1] >> 16) & 1u};
        return {g[0] & 0xffffu, g[0] >> 16, g[1] & 0x7fffu, (g[1] >> 15) & 1u, (g[1] >> 16) & 0x7fffu, g[1] >> 31};
    }
    static Val op(Kind k, uint32_t o, std::initializer_list<uint32_t> in) {
        Val v;
        v.kind = k;
        v.o = o;
        for (uint32_t i : in) v.in[v.nin++] = i;
        return v;
    }
    Val simplify(const Field& f) {
        const uint32_t z = leaf(0);
        const uint32_t s = 2 * leaf(f.s), x = 2 * leaf(f.x) + f.ix, y = 2 * leaf(f.y) + f.iy;
        const bool cx = (x >> 1) == z, cy = (y >> 1) == z;
        if (cx && cy) return f.ix == f.iy ? op(K_COPY, 0, {x}) : op(K_COPY, 0, {s ^ f.iy});
        if (cx) return f.ix ? op(K_AND, 1, {s ^ 1, y ^ 1}) : op(K_AND, 0, {s ^ 1, y});
        if (cy) return f.iy ? op(K_AND, 1, {s, x ^ 1}) : op(K_AND, 0, {s, x});
        if ((x >> 1) == (y >> 1)) return f.ix == f.iy ? op(K_COPY, 0, {x}) : op(K_XOR, f.iy, {s, x & ~1u});
        return op(K_MUX, 0, {s, x, y});
    }

    // Program M in single assignment; false when it is not of the form the
    // lowering writes (a gate into an input slot, a slot out of order).
    bool parse() {
        const uint32_t* b = s_.blob;
        cur_.assign(s_.nslots, kNone);
        is_state_.assign(s_.nslots, 0);
        nfixed_ = 1;
        for (uint32_t k = 0; k < s_.n_in; ++k) {
            const uint32_t* ic = b + s_.off_in + 4 * k;
            nfixed_ = std::max(nfixed_, std::max(ic[2], ic[3]) + ic[1]);
        }
        for (uint32_t k = 0; k < s_.n_state; ++k) {
            const uint32_t* sl = b + s_.off_state + 6 * k;
            nfixed_ = std::max(nfixed_, sl[5] + sl[4]);
            for (uint32_t i = 0; i < sl[4]; ++i) is_state_[sl[5] + i] = 1;
        }
        v_.reserve(b[s_.off_lev + s_.nlev] + nfixed_);
        std::vector<std::pair<uint32_t, uint32_t>> now;
        for (uint32_t l = 0; l < s_.nlev; ++l) {
            now.clear();
            for (uint32_t k = b[s_.off_lev + l]; k < b[s_.off_lev + l + 1]; ++k) {
                const Field f = field(k);
                for (uint32_t r : {f.s, f.x, f.y})
                    if (r >= nfixed_ && cur_[r] == kNone) return false;
                Val v = simplify(f);
                now.push_back({f.dst, (uint32_t)v_.size()});
                v_.push_back(v);
            }
            for (const auto& w : now) {
                if (w.first < nfixed_) {
                    if (!is_state_[w.first]) return false;
                    add_state(v_[w.second], w.first, 0);
                }
                cur_[w.first] = w.second;
            }
        }
        return true;
    }

    // The tables that read values after the last level.
    bool tables() {
        const uint32_t* b = s_.blob;
        for (uint32_t k = 0; k < s_.n_commit; ++k) {
            const uint32_t* c = b + s_.off_commit + 2 * k;
            const uint32_t v = cur_[c[1] & 0x7fffffffu];
            if (c[0] >= nfixed_ || !is_state_[c[0]] || v == kNone || v_[v].kind == LEAF) return false;
            add_state(v_[v], c[0], c[1] >> 31);
        }
        bool ok = true;
        const auto keep = [&](uint32_t ref) {
            const uint32_t v = leaf(ref & 0x7fffffffu);
            // a state or input plane may change under the lane work
            if (v_[v].kind == LEAF && v != leaf(0)) ok = false;
            v_[v].keep = true;
        };
        each_ref(keep);
        return ok;
    }
    // Every slot reference of the hash and port tables of program M.
    template <typename F>
    void each_ref(const F& fn) const {
        const uint32_t* b = s_.blob;
        uint32_t o = s_.off_hash;
        for (uint32_t k = 0; k < s_.n_hash; ++k) {
            for (uint32_t i = 0; i < b[o + 1]; ++i) fn(b[o + 2 + i]);
            o += 2 + b[o + 1];
        }
        const uint32_t* q = b + s_.off_ports + 2;
        for (uint32_t r = 0; r < b[s_.off_ports + 1]; ++r) {
            const uint32_t na = q[2], n2 = q[3], refs = q[0] == 0 ? na : 1 + na + n2;
            for (uint32_t i = 0; i < refs; ++i) fn(q[4 + i]);
            q += (q[0] == 0 ? 4u : 5u) + na + n2;
        }
    }

    void set_levels(bool delay) {
        lmax_ = 0;
        for (Val& v : v_) {
            v.readers = v.pol = v.inv = 0;
            v.target = kNone;
            if (v.kind != LEAF) v.slot = kNone;
        }
        for (Val& v : v_) {
            if (v.kind == LEAF) continue;
            uint32_t l = 0;
            for (uint32_t k = 0; k < v.nin; ++k) {
                Val& x = v_[v.in[k] >> 1];
                l = std::max(l, x.level);
                x.readers++;
            }
            v.level = v.asap = l + 1;
            lmax_ = std::max(lmax_, v.level);
        }
        const auto scan = [&]() {
            for (Val& v : v_) v.last = 0;
            for (const Val& v : v_)
                for (uint32_t k = 0; k < v.nin; ++k) {
                    Val& x = v_[v.in[k] >> 1];
                    x.last = std::max(x.last, v.level);
                }
        };
        std::vector<uint32_t> leaf_of(s_.nslots, kNone);   // state slot -> its value before the edge
        for (uint32_t i = 0; i < v_.size(); ++i)
            if (v_[i].kind == LEAF) leaf_of[v_[i].slot] = i;
        const auto last_read = [&](uint32_t slot) { return leaf_of[slot] == kNone ? 0u : v_[leaf_of[slot]].last; };
        scan();
        // next states that nothing else reads move past the last reader of
        // their state, so that they can be written in place
        for (int it = 0; it < 2 && delay; ++it) {
            for (Val& v : v_) {
                if (v.keep || v.states == kNone || v.readers) continue;
                uint32_t want = kNone;
                for (uint32_t k = v.states; k != kNone; k = takes_[k].next)
                    want = std::min(want, last_read(takes_[k].slot) + 1);
                v.level = std::min(lmax_, std::max(v.asap, want));
            }
            scan();
        }
        if (delay) {
            pack_levels();
            scan();
        }
        for (Val& v : v_) {
            for (uint32_t k = v.states; k != kNone; k = takes_[k].next)
                if (v.target == kNone && !takes_[k].inv && last_read(takes_[k].slot) < v.level) v.target = takes_[k].slot;
            if (v.keep) v.last = lmax_ + 1;
            for (uint32_t k = v.states; k != kNone; k = takes_[k].next)
                if (takes_[k].slot != v.target) v.last = lmax_ + 1;
        }
    }

    // Rounds that the levels need at the least (classes that leave wavefront
    // rows partly empty can need more).
    uint32_t least_rounds() const {
        std::vector<uint32_t> n(lmax_ + 1, 0);
        for (const Val& v : v_)
            if (v.kind != LEAF) n[v.level]++;
        uint32_t r = 0;
        for (uint32_t x : n) r += (x + nt_ - 1) / nt_;
        return r;
    }

    // A level's rows past its last full round of threads move on to the next
    // level where their readers allow it, when that saves a round.
    void pack_levels() {
        std::vector<uint32_t> latest(v_.size(), lmax_), n(lmax_ + 2, 0);
        std::vector<std::vector<uint32_t>> at(lmax_ + 2);
        for (uint32_t i = (uint32_t)v_.size(); i-- > 0;) {
            if (v_[i].kind == LEAF) continue;
            for (uint32_t k = 0; k < v_[i].nin; ++k) {
                uint32_t& x = latest[v_[i].in[k] >> 1];
                x = std::min(x, v_[i].level - 1);
            }
        }
        // (readers are at their final or a later level, so ``latest`` holds)
        for (uint32_t i = 0; i < v_.size(); ++i)
            if (v_[i].kind != LEAF) at[v_[i].level].push_back(i);
        for (uint32_t l = 1; l < lmax_; ++l) {
            const uint32_t over = (uint32_t)at[l].size() % nt_, next = (uint32_t)at[l + 1].size();
            if (!over || at[l].size() < nt_) continue;
            // free room in the next level, or at least no round more than here
            if ((next + over + nt_ - 1) / nt_ > (next + nt_ - 1) / nt_ + 1) continue;
            std::vector<uint32_t> go;
            for (size_t k = at[l].size(); k-- > 0 && go.size() < over;)
                if (latest[at[l][k]] > l) go.push_back(at[l][k]);
            if (go.size() < over) continue;
            std::vector<char> gone(v_.size(), 0);
            for (uint32_t i : go) {
                gone[i] = 1;
                v_[i].level = l + 1;
                at[l + 1].push_back(i);
            }
            at[l].erase(std::remove_if(at[l].begin(), at[l].end(), [&](uint32_t i) { return gone[i]; }), at[l].end());
        }
    }

    // Class, operands and polarity of every value (operands come first).
    void classify() {
        for (Val& v : v_) {
            if (v.kind == LEAF) continue;
            uint32_t id[3], in[3];
            for (uint32_t k = 0; k < v.nin; ++k) {
                id[k] = v.in[k] >> 1;
                in[k] = (v.in[k] & 1) ^ v_[id[k]].pol;
            }
            switch (v.kind) {
                case K_COPY:
                    v.cls = AND, v.s = v.x = id[0], v.pol = in[0] ^ v.o;
                    break;
                case K_AND:
                    v.s = id[0], v.x = id[1], v.pol = v.o;
                    if (in[0] && in[1]) v.cls = NOR;
                    else if (!in[0] && !in[1]) v.cls = AND;
                    else {
                        v.cls = ANDN;
                        if (in[0]) std::swap(v.s, v.x);
                    }
                    break;
                case K_XOR:
                    v.cls = XOR, v.s = id[0], v.x = id[1], v.pol = in[0] ^ in[1] ^ v.o;
                    break;
                default: {   // K_MUX
                    v.s = id[0], v.x = id[1], v.y = id[2];
                    uint32_t ix = in[1], iy = in[2];
                    if (in[0]) std::swap(v.x, v.y), std::swap(ix, iy);
                    v.cls = ix == iy ? MUX : MUXN;
                    v.pol = iy ^ v.o;
                }
            }
            if (v.target != kNone && v.pol) v.inv = 1, v.pol = 0;   // in place: generic, complemented
        }
    }

    uint32_t reads(const Val& v) const { return v.cls == MUX || v.cls == MUXN ? 3u : 2u; }

    // Rounds, row order and slots, level by level.
    bool place(Plan& p) {
        std::vector<std::vector<uint32_t>> at(lmax_ + 1);
        for (uint32_t i = 0; i < v_.size(); ++i)
            if (v_[i].kind != LEAF) at[v_[i].level].push_back(i);
        std::vector<std::vector<uint32_t>> ends(lmax_ + 2);
        std::vector<std::vector<uint32_t>> free(32);
        uint32_t top = nfixed_;
        count_banks();
        banks_.assign(4, Banks(s_.nslots));
        p.cls.assign((size_t)nw_ * 4, 0);
        for (uint32_t l = 1; l <= lmax_; ++l) {
            // temporaries last read at an earlier level are free
            for (uint32_t i : ends[l - 1]) free[v_[i].slot % 32].push_back(v_[i].slot);
            std::vector<std::vector<uint32_t>> grp(CLASSES);
            for (uint32_t i : at[l]) grp[v_[i].inv ? (uint32_t)GENERIC : v_[i].cls].push_back(i);
            pool_remainders(grp);
            std::vector<std::pair<uint32_t, std::vector<uint32_t>>> wr;   // class, values
            for (uint32_t c = 0; c < CLASSES; ++c) {
                spread(grp[c], c);
                for (size_t k = 0; k < grp[c].size(); k += 64)
                    wr.push_back({c, {grp[c].begin() + k, grp[c].begin() + std::min(grp[c].size(), k + 64)}});
            }
            const uint32_t rounds = ((uint32_t)wr.size() + nw_ - 1) / nw_;
            if (p.nr + rounds > maxr_) return false;
            p.recs.resize((size_t)(p.nr + rounds) * nt_ * 2, 0);
            for (uint32_t k = 0; k < wr.size(); ++k) {
                // the last round's idle wavefronts are the first ones
                const uint32_t r = p.nr + k / nw_, w = nw_ - 1 - k % nw_;
                mark(p, w, r, wr[k].first);
                p.rows++;
                p.generic += wr[k].first == GENERIC;
                uint32_t held = 0;
                const auto& rows = wr[k].second;
                for (uint32_t t = 0; t < 64; ++t) {
                    if (t % 32 == 0) {
                        held = 0;   // bank pairs of this half's destinations
                        for (uint32_t j = t; j < std::min<size_t>(rows.size(), t + 32); ++j)
                            if (v_[rows[j]].target != kNone) held |= 1u << (v_[rows[j]].target % 32);
                    }
                    uint32_t* rec = &p.recs[((size_t)r * nt_ + w * 64 + t) * 2];
                    if (t >= rows.size()) {
                        // idle lanes repeat the last row
                        rec[0] = rec[-2];
                        rec[1] = rec[-1];
                        continue;
                    }
                    Val& v = v_[rows[t]];
                    if (v.target != kNone) {
                        v.slot = v.target;
                    } else {
                        v.slot = take(free, held, top, rows[t]);
                        if (top > s_.nslots) return false;
                        held |= 1u << (v.slot % 32);
                        if (v.last <= lmax_) ends[std::max(v.last, l)].push_back(rows[t]);
                    }
                    write(rec, wr[k].first == GENERIC ? generic(v) : plain(v));
                }
            }
            p.nr += rounds;
            if (rounds) p.bar |= 1ull << (p.nr - 1);
        }
        return true;
    }

    static void mark(Plan& p, uint32_t wave, uint32_t round, uint32_t cls) {
        for (uint32_t bit = 0; bit < 4; ++bit)
            if (((cls | 8u) >> bit) & 1) p.cls[4 * wave + bit] |= 1ull << round;
    }

    // Classes' last rows that do not fill a wavefront row become generic,
    // smallest first, while that saves the level a round.
    void pool_remainders(std::vector<std::vector<uint32_t>>& grp) const {
        size_t full = 0, rest = grp[GENERIC].size();
        std::vector<std::pair<size_t, uint32_t>> rem;
        for (uint32_t c = AND; c < GENERIC; ++c) {
            full += grp[c].size() / 64;
            if (grp[c].size() % 64) rem.push_back({grp[c].size() % 64, c});
        }
        size_t all = rest;
        for (const auto& r : rem) all += r.first;
        const size_t least = (full + (all + 63) / 64 + nw_ - 1) / nw_ * nw_;
        std::sort(rem.begin(), rem.end());
        for (size_t k = 0; k < rem.size(); ++k) {
            if (full + (rem.size() - k) + (rest + 63) / 64 <= least) break;
            auto& from = grp[rem[k].second];
            grp[GENERIC].insert(grp[GENERIC].end(), from.end() - rem[k].first, from.end());
            from.resize(from.size() - rem[k].first);
            rest += rem[k].first;
        }
    }

    // The value's record: without inversions, and generic (also of a class
    // row that joins a generic wavefront row).
    Field plain(const Val& v) const {
        return {v.slot, v_[v.s].slot, v_[v.x].slot, 0, v.cls >= MUX ? v_[v.y].slot : v_[v.x].slot, 0};
    }
    Field generic(const Val& v) const {
        const uint32_t s = v_[v.s].slot, x = v_[v.x].slot, y = v_[v.y].slot, o = v.inv;
        switch (v.cls) {
            case AND: return {v.slot, s, x, o, 0, o};
            case ANDN: return {v.slot, s, x, o ^ 1, 0, o};
            case NOR: return {v.slot, s, 0, o, x, o ^ 1};
            case XOR: return {v.slot, s, x, o ^ 1, x, o};
            case MUX: return {v.slot, s, x, o, y, o};
            default: return {v.slot, s, x, o ^ 1, y, o};
        }
    }
    void write(uint32_t* rec, const Field& f) const {
        if (s_.byte_form) {
            rec[0] = 8 * f.dst | (8 * f.s) << 16;
            rec[1] = (8 * f.x | f.ix) | (8 * f.y | f.iy) << 16;
        } else {
            rec[0] = f.dst | f.s << 16;
            rec[1] = (f.x | f.ix << 15) | (f.y | f.iy << 15) << 16;
        }
    }

    // How often the operands of a level's class rows name each bank pair:
    // a temporary takes the bank pair its readers use least, so that 32 of
    // them can be found without two slots in one (the operands of a
    // commutative class count together).
    uint32_t* bank_use(const Val& v, uint32_t k) {
        const uint32_t op = v.cls == MUX || v.cls == MUXN ? k : v.cls == ANDN ? k : 0u;
        return &use_[(((size_t)v.level * CLASSES + (v.inv ? (uint32_t)GENERIC : v.cls)) * 3 + op) * 32];
    }
    void count_banks() {
        use_.assign((size_t)(lmax_ + 1) * CLASSES * 3 * 32, 0);
        rd_at_.assign(v_.size() + 1, 0);
        const auto each = [&](const auto& fn) {
            for (Val& v : v_) {
                if (v.kind == LEAF) continue;
                const uint32_t op[3] = {v.s, v.x, v.y};
                for (uint32_t k = 0; k < reads(v); ++k) fn(v, k, op[k]);
            }
        };
        each([&](Val& v, uint32_t k, uint32_t i) {
            const Val& x = v_[i];
            if (x.kind == LEAF || x.target != kNone)
                bank_use(v, k)[(x.kind == LEAF ? x.slot : x.target) % 32]++;
            else
                ++rd_at_[i + 1];
        });
        for (size_t i = 1; i < rd_at_.size(); ++i) rd_at_[i] += rd_at_[i - 1];
        rd_use_.resize(rd_at_.back());
        std::vector<uint32_t> to(rd_at_);
        each([&](Val& v, uint32_t k, uint32_t i) {
            if (v_[i].kind != LEAF && v_[i].target == kNone) rd_use_[to[i]++] = (uint32_t)(bank_use(v, k) - use_.data());
        });
    }
    // A slot for value ``i``: a free one or the next new one, its bank pair
    // not in ``held`` (the destinations of its 32 lanes).
    uint32_t take(std::vector<std::vector<uint32_t>>& free, uint32_t held, uint32_t& top, uint32_t i) {
        uint32_t cost[32];
        for (uint32_t r = 0; r < 32; ++r) cost[r] = 63 - (uint32_t)std::min<size_t>(63, free[r].size());
        for (uint32_t k = rd_at_[i]; k < rd_at_[i + 1]; ++k) {
            const uint32_t* u = &use_[rd_use_[k]];
            for (uint32_t r = 0; r < 32; ++r) cost[r] += 64 * u[r];
        }
        uint32_t best = kNone, least = kNone;
        for (int any = held == kNone ? 1 : 0; any < 2 && best == kNone; ++any)
            for (uint32_t r = 0; r < 32; ++r) {
                if ((((held >> r) & 1) && !any) || (free[r].empty() && top + 32 > s_.nslots)) continue;
                if (cost[r] < least) least = cost[r], best = r;
            }
        if (best == kNone) return top++;   // past the program's slots: the plan fails
        for (uint32_t k = rd_at_[i]; k < rd_at_[i + 1]; ++k) use_[rd_use_[k] + best]++;
        if (free[best].empty()) {
            while (top % 32 != best) {
                free[top % 32].push_back(top);
                ++top;
            }
            return top++;
        }
        const uint32_t s = free[best].back();
        free[best].pop_back();
        return s;
    }

    // Bank pairs that 32 lanes' accesses of one kind meet: LDS serves 32 lanes'
    // 64-bit accesses at a time, in as many passes as the most slots that
    // differ in one bank pair (slot modulo 32; equal slots are one access).
    struct Banks {
        std::vector<uint32_t> at;   // per slot: the set it was last put in
        uint32_t set = 0;
        uint8_t n[32];
        uint8_t most;
        explicit Banks(uint32_t nslots) : at(nslots, 0) {}
        void clear() {
            ++set;
            std::fill(n, n + 32, 0);
            most = 0;
        }
        // 256 for another pass, plus the slots already in the bank pair
        uint32_t cost(uint32_t s) const {
            if (at[s] == set) return 0;
            const uint32_t c = n[s % 32];
            return c + (c == most ? 256u : 0u);
        }
        void put(uint32_t s) {
            if (at[s] == set) return;
            at[s] = set;
            most = std::max(most, ++n[s % 32]);
        }
    };

    // The rows of a class of a level ordered: each next row is the one whose
    // operands (and fixed destination) need the fewest further passes of the
    // current 32 lanes; a commutative gate's operands may swap.
    void spread(std::vector<uint32_t>& g, uint32_t cls) {
        struct Cand {
            uint32_t s, x, y, dst, val;
        };
        std::vector<Cand> left(g.size());
        for (size_t k = 0; k < g.size(); ++k) {
            const Val& v = v_[g[k]];
            const Field f = cls == GENERIC ? generic(v) : plain(v);
            left[k] = {f.s, f.x, f.y, v.target, g[k]};
        }
        const bool swaps = cls == AND || cls == NOR || cls == XOR, three = cls >= MUX;
        Banks &bs = banks_[0], &bx = banks_[1], &by = banks_[2], &bd = banks_[3];
        for (size_t k = 0; k < left.size(); ++k) {
            if (k % 32 == 0)
                for (Banks& b : banks_) b.clear();
            size_t best = k;
            uint32_t least = kNone;
            bool swap = false;
            // (the first row of a half: any)
            const size_t end = k % 32 ? left.size() : k + 1;
            for (size_t j = k; j < end && least; ++j) {
                const Cand& c = left[j];
                uint32_t w = c.dst != kNone ? bd.cost(c.dst) : 0u;
                if (three) w += by.cost(c.y);
                const uint32_t w0 = w + bs.cost(c.s) + bx.cost(c.x);
                if (w0 < least) least = w0, best = j, swap = false;
                if (swaps) {
                    const uint32_t w1 = w + bs.cost(c.x) + bx.cost(c.s);
                    if (w1 < least) least = w1, best = j, swap = true;
                }
            }
            std::swap(left[k], left[best]);
            Cand& c = left[k];
            if (swap) {
                std::swap(c.s, c.x);
                std::swap(v_[c.val].s, v_[c.val].x);
            }
            if (c.dst != kNone) bd.put(c.dst);
            if (three) by.put(c.y);
            bs.put(c.s);
            bx.put(c.x);
            g[k] = c.val;
        }
    }

    // Slot reference of a table entry (inversion in bit 31).
    uint32_t ref(uint32_t old) const {
        const Val& v = v_[cur_[old & 0x7fffffffu]];
        return v.slot | ((old >> 31) ^ v.pol) << 31;
    }
    void emit_tables(Plan& p) const {
        const uint32_t* b = s_.blob;
        std::vector<std::pair<uint32_t, uint32_t>> com;
        for (const Val& v : v_)
            for (uint32_t k = v.states; k != kNone; k = takes_[k].next)
                if (takes_[k].slot != v.target) com.push_back({takes_[k].slot, v.slot | (takes_[k].inv ^ v.pol) << 31});
        spread_commit(com);
        for (const auto& c : com) p.commit.insert(p.commit.end(), {c.first, c.second});
        uint32_t o = s_.off_hash;
        for (uint32_t k = 0; k < s_.n_hash; ++k) {
            p.hash.insert(p.hash.end(), {b[o], b[o + 1]});
            for (uint32_t i = 0; i < b[o + 1]; ++i) p.hash.push_back(ref(b[o + 2 + i]));
            o += 2 + b[o + 1];
        }
        const uint32_t* q = b + s_.off_ports;
        p.ports.assign(q, q + q[0]);
        uint32_t at = 2;
        for (uint32_t r = 0; r < q[1]; ++r) {
            const uint32_t kind = q[at], na = q[at + 2], n2 = q[at + 3], refs = kind == 0 ? na : 1 + na + n2;
            for (uint32_t i = 0; i < refs; ++i) p.ports[at + 4 + i] = ref(q[at + 4 + i]);
            at += (kind == 0 ? 4u : 5u) + na + n2;
        }
    }
    // Commit pairs ordered like rows: reads and writes of each 32 spread over
    // the bank pairs.
    void spread_commit(std::vector<std::pair<uint32_t, uint32_t>>& c) const {
        std::vector<Banks> bk(2, Banks(s_.nslots));
        for (size_t k = 0; k < c.size(); ++k) {
            if (k % 32 == 0) bk[0].clear(), bk[1].clear();
            size_t best = k;
            uint32_t least = kNone;
            for (size_t j = k; j < c.size() && least && (j == k || k % 32); ++j) {
                const uint32_t w = bk[0].cost(c[j].first) + bk[1].cost(c[j].second & 0x7fffffffu);
                if (w < least) least = w, best = j;
            }
            std::swap(c[k], c[best]);
            bk[0].put(c[k].first);
            bk[1].put(c[k].second & 0x7fffffffu);
        }
    }

    const Source s_;
    const uint32_t nt_, nw_, maxr_;
    std::vector<Val> v_;
    std::vector<Take> takes_;
    std::vector<uint32_t> cur_;     // slot -> value it holds
    std::vector<char> is_state_;
    std::vector<uint32_t> use_;                    // bank_use()
    std::vector<uint32_t> rd_at_, rd_use_;         // of a temporary i: its readers' rows of use_, rd_use_[rd_at_[i] ..)
    std::vector<Banks> banks_;                     // of spread(): s, x, y, fixed destinations
    uint32_t nfixed_ = 0, lmax_ = 0, zero_ = kNone;
};

}  // namespace bpplan
