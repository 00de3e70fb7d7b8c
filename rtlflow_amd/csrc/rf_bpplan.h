// rf_bpplan.h -- host planner of the bit-plane kernel's per-cycle program:
// program M of a blob (generic gate records, level by level) becomes rounds
// of wavefront rows. Plain C++ (no GPU), so the CPU tests run it.
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
    uint32_t nr = 0;                   // rounds
    uint64_t bar = 0;                  // bit i: a barrier follows round i
    std::vector<uint32_t> recs;        // [round][thread] two words
    std::vector<uint64_t> cls;         // [wavefront][4]: bit i of word b < 3 is bit b of round i's class, of word 3: it has a row
    std::vector<uint32_t> commit;      // {state slot, source slot | inverted << 31}
    std::vector<uint32_t> hash, ports; // program M's tables with the plan's slots
    uint32_t rows = 0, generic = 0;    // wavefront rows, of which generic
};

class Planner {
public:
    Planner(const Source& s, uint32_t threads, uint32_t max_rounds)
        : s_(s), nt_(threads), nw_(threads / 64), maxr_(max_rounds) {}

    // The plan of classed rows; when the program is not of the lowering's form
    // or its values need more slots than it has, its own records as generic
    // rows. Not ok: more rounds than max_rounds.
    Plan run() {
        if (parse() && tables()) {
            for (bool delay : {true, false}) {
                Plan p;
                set_levels(delay);
                classify();
                if (!place(p)) continue;
                emit_tables(p);
                p.ok = true;
                return p;
            }
        }
        return as_stated();
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
        std::vector<uint32_t> states; // (state slot << 1 | inverted) that take it
        // class row
        uint8_t cls = 0, inv = 0, pol = 0;
        uint32_t s = 0, x = 0, y = 0;
    };
    struct Field {
        uint32_t dst, s, x, ix, y, iy;
    };

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
                    v_[w.second].states.push_back(2 * w.first);
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
            v_[v].states.push_back(2 * c[0] + (c[1] >> 31));
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
                if (v.keep || v.states.empty() || v.readers) continue;
                uint32_t want = kNone;
                for (uint32_t st : v.states) want = std::min(want, last_read(st >> 1) + 1);
                v.level = std::min(lmax_, std::max(v.asap, want));
            }
            scan();
        }
        if (delay) {
            pack_levels();
            scan();
        }
        for (Val& v : v_) {
            for (uint32_t st : v.states)
                if (v.target == kNone && !(st & 1) && last_read(st >> 1) < v.level) v.target = st >> 1;
            if (v.keep) v.last = lmax_ + 1;
            for (uint32_t st : v.states)
                if ((st >> 1) != v.target) v.last = lmax_ + 1;
        }
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
        p.cls.assign((size_t)nw_ * 4, 0);
        for (uint32_t l = 1; l <= lmax_; ++l) {
            // temporaries last read at an earlier level are free
            for (uint32_t i : ends[l - 1]) free[v_[i].slot % 32].push_back(v_[i].slot);
            std::vector<std::vector<uint32_t>> grp(CLASSES);
            for (uint32_t i : at[l]) grp[v_[i].inv ? (uint32_t)GENERIC : v_[i].cls].push_back(i);
            pool_remainders(grp);
            std::vector<std::pair<uint32_t, std::vector<uint32_t>>> wr;   // class, values
            for (uint32_t c = 0; c < CLASSES; ++c)
                for (size_t k = 0; k < grp[c].size(); k += 64) {
                    spread(grp[c], k, c);
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

    // The program's own records as generic rows.
    Plan as_stated() const {
        Plan p;
        const uint32_t* b = s_.blob;
        p.cls.assign((size_t)nw_ * 4, 0);
        for (uint32_t l = 0; l < s_.nlev; ++l) {
            const uint32_t lo = b[s_.off_lev + l], hi = b[s_.off_lev + l + 1];
            for (uint32_t k = lo; k < hi; k += nt_, ++p.nr) {
                if (p.nr >= maxr_) return Plan();
                p.recs.resize((size_t)(p.nr + 1) * nt_ * 2, 0);
                for (uint32_t w = 0; w < nw_ && k + 64 * w < hi; ++w) {
                    mark(p, w, p.nr, GENERIC);
                    p.rows++;
                    p.generic++;
                    for (uint32_t t = 0; t < 64; ++t) {
                        const uint32_t* g = b + s_.off_gates + 2 * std::min(k + 64 * w + t, hi - 1);
                        uint32_t* rec = &p.recs[((size_t)p.nr * nt_ + w * 64 + t) * 2];
                        rec[0] = g[0];
                        rec[1] = g[1];
                    }
                }
            }
            if (hi > lo) p.bar |= 1ull << (p.nr - 1);
        }
        p.commit.assign(b + s_.off_commit, b + s_.off_commit + 2 * s_.n_commit);
        uint32_t o = s_.off_hash;
        for (uint32_t k = 0; k < s_.n_hash; ++k) o += 2 + b[o + 1];
        p.hash.assign(b + s_.off_hash, b + o);
        p.ports.assign(b + s_.off_ports, b + s_.off_ports + b[s_.off_ports]);
        p.ok = true;
        return p;
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
        readers_.assign(v_.size(), {});
        for (uint32_t i = 0; i < v_.size(); ++i) {
            Val& v = v_[i];
            if (v.kind == LEAF) continue;
            const uint32_t op[3] = {v.s, v.x, v.y};
            for (uint32_t k = 0; k < reads(v); ++k) {
                const Val& x = v_[op[k]];
                if (x.kind == LEAF || x.target != kNone)
                    bank_use(v, k)[(x.kind == LEAF ? x.slot : x.target) % 32]++;
                else
                    readers_[op[k]].push_back(4 * i + k);
            }
        }
    }
    // A slot for value ``i``: a free one or the next new one, its bank pair
    // not in ``held`` (the destinations of its 32 lanes).
    uint32_t take(std::vector<std::vector<uint32_t>>& free, uint32_t held, uint32_t& top, uint32_t i) {
        uint32_t best = kNone, least = kNone;
        for (int any = held == kNone ? 1 : 0; any < 2 && best == kNone; ++any)
            for (uint32_t r = 0; r < 32; ++r) {
                if ((((held >> r) & 1) && !any) || (free[r].empty() && top + 32 > s_.nslots)) continue;
                uint32_t c = 0;
                for (uint32_t rd : readers_[i]) c += bank_use(v_[rd / 4], rd % 4)[r];
                c = c * 64 + 63 - (uint32_t)std::min<size_t>(63, free[r].size());
                if (c < least) least = c, best = r;
            }
        if (best == kNone) return top++;   // past the program's slots: the plan fails
        for (uint32_t rd : readers_[i]) bank_use(v_[rd / 4], rd % 4)[best]++;
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
        uint32_t slot[32][8];
        uint8_t n[32];
        uint8_t most;
        void clear() {
            std::fill(n, n + 32, 0);
            most = 0;
        }
        bool has(uint32_t s) const {
            const uint32_t r = s % 32;
            for (uint32_t i = 0; i < n[r]; ++i)
                if (slot[r][i] == s) return true;
            return false;
        }
        // 256 for another pass, plus the slots already in the bank pair
        uint32_t cost(uint32_t s) const {
            if (has(s)) return 0;
            const uint32_t c = n[s % 32];
            return c + (c == most ? 256u : 0u);
        }
        void put(uint32_t s) {
            const uint32_t r = s % 32;
            if (has(s)) return;
            if (n[r] < 8) slot[r][n[r]++] = s;
            most = std::max(most, n[r]);
        }
    };

    // Rows g[k0 .. k0 + 64) chosen from g[k0 ..) and ordered: each next row is
    // the one whose operands (and fixed destination) need the fewest further
    // passes of the current 32 lanes; a commutative gate's operands may swap.
    void spread(std::vector<uint32_t>& g, size_t k0, uint32_t cls) {
        Banks bk[4];
        const size_t end = std::min(g.size(), k0 + 64);
        for (size_t k = k0; k < end; ++k) {
            if ((k - k0) % 32 == 0)
                for (Banks& b : bk) b.clear();
            size_t best = k;
            uint32_t least = kNone;
            bool swap = false;
            for (size_t j = k; j < g.size() && least; ++j) {
                const Val& v = v_[g[j]];
                const Field f = cls == GENERIC ? generic(v) : plain(v);
                uint32_t c = v.target != kNone ? bk[3].cost(v.target) : 0u;
                if (cls >= MUX) c += bk[2].cost(f.y);
                const uint32_t c0 = c + bk[0].cost(f.s) + bk[1].cost(f.x);
                if (c0 < least) least = c0, best = j, swap = false;
                if (cls == AND || cls == NOR || cls == XOR) {
                    const uint32_t c1 = c + bk[0].cost(f.x) + bk[1].cost(f.s);
                    if (c1 < least) least = c1, best = j, swap = true;
                }
                if ((k - k0) % 32 == 0) break;   // the first row of a half: any
            }
            std::swap(g[k], g[best]);
            Val& v = v_[g[k]];
            if (swap) std::swap(v.s, v.x);
            const Field f = cls == GENERIC ? generic(v) : plain(v);
            if (v.target != kNone) bk[3].put(v.target);
            if (cls >= MUX) bk[2].put(f.y);
            bk[0].put(f.s);
            bk[1].put(f.x);
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
            for (uint32_t st : v.states)
                if ((st >> 1) != v.target) com.push_back({st >> 1, v.slot | ((st & 1) ^ v.pol) << 31});
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
    static void spread_commit(std::vector<std::pair<uint32_t, uint32_t>>& c) {
        Banks bk[2];
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
    std::vector<uint32_t> cur_;     // slot -> value it holds
    std::vector<char> is_state_;
    std::vector<uint32_t> use_;                    // bank_use()
    std::vector<std::vector<uint32_t>> readers_;   // of a temporary: 4 * value + operand
    uint32_t nfixed_ = 0, lmax_ = 0, zero_ = kNone;
};

}  // namespace bpplan
