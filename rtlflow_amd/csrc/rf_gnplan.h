// rf_gnplan.h -- host planner of the gate-net engine's LDS form: a program of
// gate records (rf_gatenet.hip) becomes wavefront programs whose node values
// live in one workgroup's LDS. Plain C++ (no GPU), so the CPU tests run it.
//
// What the plan does to the netlist:
//
//  * Only live logic stays: gates that an output, a flip-flop or a RAM port
//    that itself reaches an output depends on (a random netlist keeps about a
//    third of its gates).
//  * One program per clock cycle evaluates the outputs of cycle n (clk = 1,
//    inputs of cycle n in plane set B) and the next state of cycle n + 1
//    (clk = 0, inputs in set A) together: both read the same flip-flop and RAM
//    planes, so gates that read no input are evaluated once.
//  * Rows. A row is what one thread evaluates: one gate, or a two-input gate
//    together with the one two-input gate that alone reads its value (at most
//    three operands, so the value in between costs no LDS access).
//  * Classes. Rows are single gates, pairs or multiplexers; 64 rows of one
//    class form a wavefront row. A single's or pair's operators are bits of the
//    row (classes per operator would leave most wavefront rows partly empty),
//    but a level's single gates of one operator are a class of their own when
//    they fill a batch: 3 VALU instructions a row instead of 8.
//  * Batches. A wavefront takes up to four wavefront rows of one class at a
//    time, so that their operand reads are in flight together; the batches of
//    a level go to the least loaded wavefront.
//  * Destinations. A batch writes consecutive slots from one base: the
//    destination costs no bits in the row and its writes share banks.
//    Flip-flops are numbered by the row that writes them, so the next state
//    goes straight into the flip-flop's slot when no row at or after its level
//    reads the old value; the other flip-flops are copied by commit rows after
//    the last level.
//  * Temporaries are reused: a batch's slots are free after the last level
//    that reads one of them (rows of a class are sorted by that level).
//  * Banks. LDS serves accesses of at most 4 bytes 32 lanes at a time over 32
//    banks, in as many passes as the most dwords in one bank: the rows of a
//    class whose slots die together are ordered so that each 32 of them read
//    distinct banks as far as possible.
#pragma once
#include <stdint.h>

#include <algorithm>
#include <exception>
#include <map>
#include <vector>

namespace gnplan {

// Header words of a program blob (layout: rf_gatenet.hip).
enum {
    H_MAGIC, H_VERSION, H_NODES, H_PI, H_FF, H_RAMBITS, H_PO, H_RAMS, H_DEPTH, H_WIDTH, H_ABITS,
    H_LEV_FULL, H_LEV_CONE, H_REC_FULL, H_REC_CONE, H_MTASKS, H_OFF_LEV_FULL, H_OFF_LEV_CONE,
    H_OFF_FF, H_OFF_PO, H_OFF_RAM, H_OFF_REC_FULL, H_OFF_REC_CONE, H_OFF_MT, H_OFF_PREDS,
    H_OFF_REC_MT, H_REC_MT, H_TOTAL, H_WORDS = 32
};
constexpr uint32_t kDstMask = (1u << 29) - 1;   // of a record's first word; the type above it

// Row classes: a single gate a k b, the pair (a k1 b) k2 c, the multiplexer
// a ? b : c, single gates of one operator (kOp + k), the copy of a to address
// b (commit rows). Operators k: 0 AND, 1 OR, 2 XOR, 3 NAND.
constexpr uint32_t kSingle = 0, kPair = 1, kMux = 2, kOp = 3, kCopy = 7, kClasses = 8;
// Cost of a wavefront row in VALU instructions plus LDS passes (its share of
// the CU), for the balance between wavefronts.
inline uint32_t row_cost(uint32_t cls) {
    return cls == kSingle ? 16u : cls == kPair ? 27u : cls == kMux ? 17u : cls == kCopy ? 8u : 11u;
}
// What a wavefront does beside a cycle's first levels, in the same measure:
// the next inputs and the hash (level 1), a RAM's read data (level kRamLevels).
constexpr uint32_t kInputCost = 150, kHashCost = 200, kRamCost = 100;

// A row: three operand byte addresses of at most 18 bits, a in bits 0..17, c
// in 18..35, b in 46..63; operator masks of k1 in bits 36..38 and k2 in bits
// 39..41. With masks p, q, n: a k b = (p ? a & ~b : a), then (q ? ^ : &) b,
// inverted when n.
constexpr uint32_t kAddrBits = 18;
inline uint64_t op_bits(uint32_t k) { return k == 0 ? 0u : k == 1 ? 3u : k == 2 ? 2u : 4u; }
inline uint64_t pack_row(uint32_t a, uint32_t b, uint32_t c, uint32_t k1, uint32_t k2) {
    return (uint64_t)a | ((uint64_t)c << 18) | ((uint64_t)b << 46) | (op_bits(k1) << 36) | (op_bits(k2) << 39);
}

// A batch of a wavefront's program, four words: class in bits 0..2, rows in
// 3..11 (at most 64 times the plan's wavefront rows per batch; 0: none), bit
// 31: a workgroup barrier follows; the first destination's byte address; the
// position in the wavefront's row stream (in lines) of the batch kUnroll
// places on, cyclically; its own position. A line is what 64 lanes load at
// once: one wavefront row of 8 bytes a lane, or with batches of kBatch
// wavefront rows two of them interleaved, 16 bytes a lane (the vector cache
// serves 4 lanes a cycle whatever they load).
// RAM data read at a cycle's edge reaches its planes within the next cycle's
// first levels (the RAM's wavefronts write them before the barrier that ends
// level kRamLevels): rows that read it come after.
constexpr uint32_t kRamLevels = 1;
constexpr uint32_t kBatch = 4;     // most wavefront rows of a batch
constexpr uint32_t kUnroll = 3;    // a wavefront's batches are a multiple of this

struct Gate {
    uint32_t type;       // 0 AND, 1 OR, 2 XOR, 3 NAND, 4 MUX
    uint32_t in[3];      // node ids (the program's)
    uint32_t level;      // level in the full evaluation, from 1
};

// The netlist as the program states it. def[node]: index into gates of the
// gate that drives the node, or kNone.
constexpr uint32_t kNone = 0xffffffffu;
struct Net {
    uint32_t nodes = 0, n_pi = 0, n_ff = 0, n_rams = 0, abits = 0, width = 0;
    std::vector<Gate> gates;
    std::vector<uint32_t> def;
    std::vector<uint32_t> ff_d, po, ram;   // ram: [n_rams][abits + 1 + width]
};

// The program's netlist for the LDS planner. False when the records are not a
// plain levelised netlist (a node driven twice, an operand that no lower
// level drives, an output cone that lacks a gate): such programs run level by
// level in the order they state.
inline bool read_net(const uint32_t* h, Net& net) {
    net.nodes = h[H_NODES];
    net.n_pi = h[H_PI];
    net.n_ff = h[H_FF];
    net.n_rams = h[H_RAMS];
    net.abits = h[H_ABITS];
    net.width = h[H_WIDTH];
    const uint32_t g0 = net.n_pi + net.n_ff + h[H_RAMBITS];
    const auto nin = [](uint32_t ty) { return ty == 4 ? 3u : 2u; };
    net.def.assign(net.nodes, kNone);
    net.gates.resize(h[H_REC_FULL]);
    const uint32_t* rec = h + h[H_OFF_REC_FULL];
    const uint32_t* lev = h + h[H_OFF_LEV_FULL];
    for (uint32_t l = 0; l < h[H_LEV_FULL]; ++l) {
        for (uint32_t k = lev[l]; k < lev[l + 1]; ++k) {
            const uint32_t* r = rec + 4 * k;
            Gate& g = net.gates[k];
            g.type = r[0] >> 29;
            g.level = l + 1;
            for (uint32_t j = 0; j < 3; ++j) g.in[j] = r[1 + j];
            for (uint32_t j = 0; j < nin(g.type); ++j)
                if (g.in[j] >= g0 && net.def[g.in[j]] == kNone) return false;
        }
        for (uint32_t k = lev[l]; k < lev[l + 1]; ++k) {
            uint32_t& d = net.def[rec[4 * k] & kDstMask];
            if (d != kNone) return false;
            d = k;
        }
    }
    net.ff_d.assign(h + h[H_OFF_FF], h + h[H_OFF_FF] + h[H_FF]);
    net.po.assign(h + h[H_OFF_PO], h + h[H_OFF_PO] + h[H_PO]);
    const uint64_t nrp = (uint64_t)h[H_RAMS] * (h[H_ABITS] + 1 + h[H_WIDTH]);
    net.ram.assign(h + h[H_OFF_RAM], h + h[H_OFF_RAM] + nrp);
    for (const std::vector<uint32_t>* v : {&net.ff_d, &net.po, &net.ram})
        for (uint32_t x : *v)
            if (x >= g0 && net.def[x] == kNone) return false;
    // the clk = 1 evaluation: the cone's records must be the same gates in
    // level order and hold every gate an output depends on
    std::vector<uint32_t> at(net.nodes, 0);   // cone level of a node, from 1
    const uint32_t* cr = h + h[H_OFF_REC_CONE];
    const uint32_t* cl = h + h[H_OFF_LEV_CONE];
    for (uint32_t l = 0; l < h[H_LEV_CONE]; ++l)
        for (uint32_t k = cl[l]; k < cl[l + 1]; ++k) {
            const uint32_t* r = cr + 4 * k;
            const uint32_t d = r[0] & kDstMask;
            if (net.def[d] == kNone || at[d]) return false;
            const uint32_t* f = rec + 4 * net.def[d];
            if (r[0] != f[0] || r[1] != f[1] || r[2] != f[2] || (nin(r[0] >> 29) == 3 && r[3] != f[3])) return false;
            at[d] = l + 1;
        }
    std::vector<uint32_t> work;
    std::vector<char> seen(net.nodes, 0);
    for (uint32_t x : net.po)
        if (x >= g0 && !seen[x]) seen[x] = 1, work.push_back(x);
    while (!work.empty()) {
        const uint32_t x = work.back();
        work.pop_back();
        if (!at[x]) return false;
        const Gate& g = net.gates[net.def[x]];
        for (uint32_t j = 0; j < nin(g.type); ++j) {
            const uint32_t y = g.in[j];
            if (y < g0) continue;
            if (!at[y] || at[y] >= at[x]) return false;
            if (!seen[y]) seen[y] = 1, work.push_back(y);
        }
    }
    return true;
}

struct Plan {
    uint32_t nslots = 0;          // plane slots of a workgroup
    uint32_t nstate = 0;          // the first of them: inputs, RAM data, flip-flops (kept between launches)
    uint32_t nwaves = 0;
    uint32_t batch = 0;           // wavefront rows of a batch: kBatch, or 1 (small netlists)
    uint32_t n_ram_live = 0;
    uint32_t a0 = 0, b0 = 0;      // slots of input sets A and B (n_pi each)
    // device tables: words[4 * w] = {first batch word, batches (a
    // multiple of kUnroll), first line, 0} of wavefront w; words[off_po + k]: byte address of output k; words[off_ram + r * ram_words] = {RAM, byte address of its
    // read data, abits + 1 control addresses, width data addresses}
    std::vector<uint32_t> words;
    std::vector<uint64_t> rows;   // 64 per wavefront row, by lines
    uint32_t off_po = 0, off_ram = 0, ram_words = 0;
    uint32_t wave_rows = 0, levels = 0;   // of one cycle
};

// First-fit allocator of runs of slots.
class Slots {
public:
    explicit Slots(uint32_t base) : top_(base) {}
    uint32_t take(uint32_t n) {
        for (auto it = free_.begin(); it != free_.end(); ++it)
            if (it->second >= n) {
                const uint32_t at = it->first, left = it->second - n;
                free_.erase(it);
                if (left) free_[at + n] = left;
                return at;
            }
        const uint32_t at = top_;
        top_ += n;
        return at;
    }
    void give(uint32_t at, uint32_t n) {
        auto nx = free_.lower_bound(at);
        if (nx != free_.end() && at + n == nx->first) {
            n += nx->second;
            nx = free_.erase(nx);
        }
        if (nx != free_.begin()) {
            auto pv = std::prev(nx);
            if (pv->first + pv->second == at) {
                pv->second += n;
                return;
            }
        }
        free_[at] = n;
    }
    uint32_t top() const { return top_; }

private:
    std::map<uint32_t, uint32_t> free_;
    uint32_t top_;
};

class Planner {
public:
    Planner(const Net& net, uint32_t nwaves) : n_(net), nw_(nwaves) {}

    // Rows, levels and the slots they need (independent of the plane width).
    uint32_t schedule() {
        find_live();
        build_values();
        make_rows();
        set_levels();
        cut();
        place(0);
        return nslots_;
    }

    // The tables for planes of ``pb`` bytes: slots() * pb below 2^18.
    Plan emit(uint32_t pb) {
        place(pb);
        return tables(pb);
    }

private:
    struct Val {             // a gate version: NG (set A) or OG (set B)
        uint32_t type = 0, nin = 0;
        uint32_t in[3] = {0, 0, 0};   // value ids
        uint32_t fanout = 0;
        uint32_t ffs = kNone;         // flip-flops that take it: the first; next_ff_ links them
        bool keep = false;            // read by the lane work after the last level
        uint32_t mate = kNone;        // row: the value evaluated with this one
        bool inside = false;          // evaluated inside another value's row
    };
    struct Row {
        uint32_t cls, k1, k2, val, rd[3], nrd;   // a copy is the single AND a & a

        uint32_t level = 0, death = 0;
        bool inplace = false;
        uint32_t ff = kNone;          // in place (or commit): the flip-flop written
    };
    struct Batch {
        uint32_t first, n, cls, level, base;   // rows order_[first .. first + n)
        uint32_t death;
        bool inplace;
    };

    // Value ids: inputs of set A, of set B, flip-flops, RAM data, gate values.
    uint32_t src_b() const { return n_.n_pi; }
    uint32_t src_ff() const { return 2 * n_.n_pi; }
    uint32_t src_rd() const { return 2 * n_.n_pi + n_.n_ff; }
    uint32_t src_end() const { return src_rd() + n_.n_rams * n_.width; }
    uint32_t first_gate() const { return n_.n_pi + n_.n_ff + n_.n_rams * n_.width; }
    uint32_t nin(const Gate& g) const { return g.type == 4 ? 3u : 2u; }

    void find_live();
    void build_values();
    uint32_t value_of(uint32_t node, bool set_b) const {
        if (node < n_.n_pi) return set_b ? src_b() + node : node;
        if (node < first_gate()) return src_ff() + (node - n_.n_pi);
        return set_b && pi_dep_[node] ? og_[node] : ng_[node];
    }
    uint32_t add_value(uint32_t type, uint32_t nin, const uint32_t* in);
    uint32_t rooted(uint32_t v);
    void make_rows();
    void set_levels();
    void cut();
    void place(uint32_t pb);
    void spread_banks(const Batch* b, const Batch* e, uint32_t pb);
    Plan tables(uint32_t pb) const;
    const Net& n_;
    const uint32_t nw_;
    std::vector<char> live_, need_a_, need_b_, pi_dep_, ram_live_;
    std::vector<uint32_t> ng_, og_;
    std::vector<Val> vals_;
    std::vector<uint32_t> buf_of_;            // source value -> its copy
    std::vector<uint32_t> next_ff_;
    std::vector<uint32_t> po_val_, ram_val_;  // values the lane work reads
    std::vector<Row> rows_;
    std::vector<uint32_t> last_;              // per source value: last level that reads it
    uint32_t lmax_ = 0;
    std::vector<uint32_t> order_;             // rows in batch order
    std::vector<Batch> batches_;
    std::vector<uint32_t> slot_;              // per value
    uint32_t nslots_ = 0, nstate_ = 0, batch_ = kBatch;
};

inline void Planner::find_live() {
    const Net& n = n_;
    live_.assign(n.nodes, 0);
    ram_live_.assign(n.n_rams, 0);
    std::vector<uint32_t> work;
    auto mark = [&](uint32_t x) {
        if (!live_[x]) {
            live_[x] = 1;
            work.push_back(x);
        }
    };
    for (uint32_t p : n.po) mark(p);
    const uint32_t rd0 = n.n_pi + n.n_ff, pw = n.abits + 1 + n.width;
    while (!work.empty()) {
        const uint32_t x = work.back();
        work.pop_back();
        if (x < n.n_pi) continue;
        if (x < rd0) {
            mark(n.ff_d[x - n.n_pi]);
        } else if (x < first_gate()) {
            const uint32_t r = (x - rd0) / n.width;
            if (ram_live_[r]) continue;
            ram_live_[r] = 1;
            for (uint32_t k = 0; k < pw; ++k) mark(n.ram[r * pw + k]);
        } else {
            const Gate& g = n.gates[n.def[x]];
            for (uint32_t k = 0; k < nin(g); ++k) mark(g.in[k]);
        }
    }
}

inline uint32_t Planner::add_value(uint32_t type, uint32_t nin, const uint32_t* in) {
    Val v;
    v.type = type;
    v.nin = nin;
    for (uint32_t k = 0; k < nin; ++k) v.in[k] = in[k];
    vals_.push_back(v);
    return src_end() + (uint32_t)vals_.size() - 1;
}

// A value the edge or the lane work takes after the last level: a source is
// copied first (its slot may take the next state before).
inline uint32_t Planner::rooted(uint32_t v) {
    if (v >= src_end()) return v;
    if (buf_of_[v] == kNone) buf_of_[v] = add_value(kNone, 1, &v);
    return buf_of_[v];
}

inline void Planner::build_values() {
    const Net& n = n_;
    pi_dep_.assign(n.nodes, 0);
    need_a_.assign(n.nodes, 0);
    need_b_.assign(n.nodes, 0);
    for (uint32_t i = 0; i < n.n_pi; ++i) pi_dep_[i] = 1;
    // the gates in level order (gates is sorted by level)
    std::vector<uint32_t> node_of(n.gates.size());
    for (uint32_t x = first_gate(); x < n.nodes; ++x)
        if (n.def[x] != kNone) node_of[n.def[x]] = x;
    for (size_t k = 0; k < n.gates.size(); ++k) {
        const Gate& g = n.gates[k];
        char d = 0;
        for (uint32_t j = 0; j < nin(g); ++j) d |= pi_dep_[g.in[j]];
        pi_dep_[node_of[k]] = d;
    }
    // next-state cone (set A) and output cone (set B where inputs matter)
    for (uint32_t f = 0; f < n.n_ff; ++f)
        if (live_[n.n_pi + f]) need_a_[n.ff_d[f]] = 1;
    const uint32_t pw = n.abits + 1 + n.width;
    for (uint32_t r = 0; r < n.n_rams; ++r)
        if (ram_live_[r])
            for (uint32_t k = 0; k < pw; ++k) need_a_[n.ram[r * pw + k]] = 1;
    for (uint32_t p : n.po) need_b_[p] = 1;
    for (size_t k = n.gates.size(); k-- > 0;) {
        const uint32_t x = node_of[k];
        if (need_b_[x] && !pi_dep_[x]) need_a_[x] = 1;   // one version serves both
        const Gate& g = n.gates[k];
        for (uint32_t j = 0; j < nin(g); ++j) {
            if (need_a_[x]) need_a_[g.in[j]] = 1;
            if (need_b_[x] && pi_dep_[x]) need_b_[g.in[j]] = 1;
        }
    }
    ng_.assign(n.nodes, kNone);
    og_.assign(n.nodes, kNone);
    buf_of_.assign(src_end(), kNone);
    next_ff_.assign(n.n_ff, kNone);
    vals_.reserve(std::count(live_.begin(), live_.end(), 1));
    for (size_t k = 0; k < n.gates.size(); ++k) {
        const uint32_t x = node_of[k];
        const Gate& g = n.gates[k];
        uint32_t in[3];
        if (need_a_[x]) {
            for (uint32_t j = 0; j < nin(g); ++j) in[j] = value_of(g.in[j], false);
            ng_[x] = add_value(g.type, nin(g), in);
        }
        if (need_b_[x] && pi_dep_[x]) {
            for (uint32_t j = 0; j < nin(g); ++j) in[j] = value_of(g.in[j], true);
            og_[x] = add_value(g.type, nin(g), in);
        }
    }
    for (uint32_t f = 0; f < n.n_ff; ++f)
        if (live_[n.n_pi + f]) {
            const uint32_t v = rooted(value_of(n.ff_d[f], false));
            next_ff_[f] = vals_[v - src_end()].ffs;
            vals_[v - src_end()].ffs = f;
        }
    for (uint32_t p : n.po) {
        const uint32_t v = rooted(value_of(p, true));
        vals_[v - src_end()].keep = true;
        po_val_.push_back(v);
    }
    for (uint32_t r = 0; r < n.n_rams; ++r)
        for (uint32_t k = 0; k < pw; ++k) {
            if (!ram_live_[r]) {
                ram_val_.push_back(kNone);
                continue;
            }
            const uint32_t v = rooted(value_of(n.ram[r * pw + k], false));
            vals_[v - src_end()].keep = true;
            ram_val_.push_back(v);
        }
    for (const Val& v : vals_)
        for (uint32_t k = 0; k < v.nin; ++k)
            if (v.in[k] >= src_end()) vals_[v.in[k] - src_end()].fanout++;
}

// Pairs by a matching from the inputs up (optimal on the forest of values
// with one reader): a two-input gate takes in one unmatched two-input operand
// that it alone reads.
inline void Planner::make_rows() {
    const uint32_t g0 = src_end();
    for (Val& y : vals_) {
        if (y.nin != 2 || y.type > 3) continue;
        for (uint32_t k = 0; k < 2; ++k) {
            if (y.in[k] < g0) continue;
            Val& x = vals_[y.in[k] - g0];
            if (x.fanout != 1 || x.keep || x.ffs != kNone || x.nin != 2 || x.type > 3 || x.mate != kNone || x.inside)
                continue;
            y.mate = y.in[k];
            x.inside = true;
            break;
        }
    }
    rows_.reserve(vals_.size());
    for (uint32_t i = 0; i < vals_.size(); ++i) {
        const Val& y = vals_[i];
        if (y.inside) continue;
        Row r{};
        r.val = g0 + i;
        if (y.type == kNone) {
            r.cls = kSingle;
            r.nrd = 2;
            r.rd[0] = r.rd[1] = y.in[0];
        } else if (y.type == 4) {
            r.cls = kMux;
            r.nrd = 3;
            for (uint32_t k = 0; k < 3; ++k) r.rd[k] = y.in[k];
        } else if (y.mate != kNone) {
            const Val& x = vals_[y.mate - g0];
            r.cls = kPair;
            r.k1 = x.type;
            r.k2 = y.type;
            r.nrd = 3;
            r.rd[0] = x.in[0];
            r.rd[1] = x.in[1];
            r.rd[2] = y.in[0] == y.mate ? y.in[1] : y.in[0];
        } else {
            r.cls = kSingle;
            r.k1 = y.type;
            r.nrd = 2;
            r.rd[0] = y.in[0];
            r.rd[1] = y.in[1];
        }
        rows_.push_back(r);
    }
}

inline void Planner::set_levels() {
    const uint32_t g0 = src_end();
    // as soon as possible (rows are in a topological order: a value's row
    // comes after the rows of its operands)
    std::vector<uint32_t> readers(vals_.size(), 0), asap(vals_.size(), 0);
    for (Row& r : rows_) {
        uint32_t l = 0;
        for (uint32_t k = 0; k < r.nrd; ++k) {
            if (r.rd[k] < g0) {
                if (r.rd[k] >= src_rd()) l = std::max(l, kRamLevels);
                continue;
            }
            l = std::max(l, asap[r.rd[k] - g0]);
            readers[r.rd[k] - g0]++;
        }
        asap[r.val - g0] = r.level = l + 1;
        lmax_ = std::max(lmax_, r.level);
    }
    if (std::count(ram_live_.begin(), ram_live_.end(), 1)) lmax_ = std::max(lmax_, kRamLevels);
    auto scan = [&]() {
        last_.assign(g0, 0);
        for (const Row& r : rows_)
            for (uint32_t k = 0; k < r.nrd; ++k)
                if (r.rd[k] < g0) last_[r.rd[k]] = std::max(last_[r.rd[k]], r.level);
    };
    scan();
    // next-state values that nothing else reads move past the last reader of
    // their flip-flop, so that they can be written in place
    for (int it = 0; it < 2; ++it) {
        for (size_t i = 0; i < rows_.size(); ++i) {
            const Val& v = vals_[rows_[i].val - g0];
            if (v.keep || v.ffs == kNone || readers[rows_[i].val - g0]) continue;
            uint32_t want = kNone;
            for (uint32_t f = v.ffs; f != kNone; f = next_ff_[f]) want = std::min(want, last_[src_ff() + f] + 1);
            rows_[i].level = std::min(lmax_, std::max(asap[rows_[i].val - g0], want));
        }
        scan();
    }
    // in-place targets, commit copies, last uses
    const uint32_t lc = lmax_ + 1;
    std::vector<uint32_t> death(vals_.size(), 0);
    for (const Row& r : rows_)
        for (uint32_t k = 0; k < r.nrd; ++k)
            if (r.rd[k] >= g0) death[r.rd[k] - g0] = std::max(death[r.rd[k] - g0], r.level);
    const size_t nr = rows_.size();
    for (size_t i = 0; i < nr; ++i) {
        const Val& v = vals_[rows_[i].val - g0];
        uint32_t pick = kNone;
        for (uint32_t f = v.ffs; f != kNone; f = next_ff_[f])
            if (pick == kNone && last_[src_ff() + f] < rows_[i].level) pick = f;
        rows_[i].inplace = pick != kNone;
        rows_[i].ff = pick;
        uint32_t d = death[rows_[i].val - g0];
        if (v.keep) d = lc;
        for (uint32_t f = v.ffs; f != kNone; f = next_ff_[f]) {
            if (f == pick) continue;
            Row c{};
            c.cls = kCopy;
            c.val = kNone;
            c.nrd = 1;
            c.rd[0] = rows_[i].val;
            c.level = lc;
            c.inplace = true;
            c.ff = f;
            rows_.push_back(c);
            d = lc;
        }
        rows_[i].death = d;
    }
}

// Rows into batches: by level, class, destination kind and death.
inline void Planner::cut() {
    std::vector<uint32_t> ops((size_t)(lmax_ + 2) * 4, 0);
    for (const Row& r : rows_)
        if (r.cls == kSingle) ++ops[r.level * 4 + r.k1];
    for (Row& r : rows_)
        if (r.cls == kSingle && ops[r.level * 4 + r.k1] >= 64 * kBatch) r.cls = kOp + r.k1;
    // (two stable counting sorts, by death, then by level, class and in place:
    // their tables grow with the depth, not with its square, and hold any depth)
    const auto sort_by = [&](const std::vector<uint32_t>& in, size_t keys, const auto& key) {
        std::vector<uint32_t> start(keys + 1, 0), out(in.size());
        for (uint32_t i : in) ++start[key(rows_[i]) + 1];
        for (size_t k = 1; k < start.size(); ++k) start[k] += start[k - 1];
        for (uint32_t i : in) out[start[key(rows_[i])]++] = i;
        return out;
    };
    order_.resize(rows_.size());
    for (uint32_t i = 0; i < rows_.size(); ++i) order_[i] = i;
    order_ = sort_by(order_, lmax_ + 2, [](const Row& r) { return (size_t)r.death; });
    order_ = sort_by(order_, (size_t)(lmax_ + 2) * kClasses * 2, [](const Row& r) {
        return ((size_t)r.level * kClasses + r.cls) * 2 + (r.inplace ? 1u : 0u);
    });
    // batches of one wavefront row when the levels hold fewer than two per
    // wavefront on average: every wavefront gets some, and loads no more
    batch_ = rows_.size() < (size_t)(lmax_ + 1) * 128 * nw_ ? 1 : kBatch;
    for (size_t i = 0; i < order_.size();) {
        const uint32_t level = rows_[order_[i]].level;
        size_t e = i;
        while (e < order_.size() && rows_[order_[e]].level == level) ++e;
        // small levels take smaller batches likewise
        const uint32_t most = 64 * (uint32_t)std::min<size_t>(batch_, std::max<size_t>(1, (e - i) / (128 * nw_)));
        while (i < e) {
            const Row& r = rows_[order_[i]];
            Batch b{(uint32_t)i, 0, r.cls, level, 0, level, r.inplace};
            while (i < e && b.n < most && rows_[order_[i]].cls == r.cls && rows_[order_[i]].inplace == r.inplace) {
                b.death = std::max(b.death, rows_[order_[i]].death);
                ++b.n;
                ++i;
            }
            batches_.push_back(b);
        }
    }
}

// Slots for every value (``pb`` != 0: rows ordered for the LDS banks of
// planes of pb bytes; the slots needed do not depend on it).
inline void Planner::place(uint32_t pb) {
    const uint32_t g0 = src_end();
    // state slots: inputs of set A and B, RAM data, flip-flops
    slot_.assign(g0 + vals_.size(), kNone);
    uint32_t s = 0;
    for (uint32_t i = 0; i < 2 * n_.n_pi; ++i) slot_[i] = s++;
    for (uint32_t i = 0; i < n_.n_rams * n_.width; ++i) slot_[src_rd() + i] = s++;
    for (Batch& b : batches_) {
        if (!b.inplace) continue;
        b.base = s;
        for (uint32_t k = 0; k < b.n; ++k) {
            const Row& q = rows_[order_[b.first + k]];
            slot_[src_ff() + q.ff] = s;
            if (q.val != kNone) slot_[q.val] = s;
            ++s;
        }
    }
    nstate_ = s;
    // temporaries, level by level
    Slots pool(s);
    struct Block {
        uint32_t at, n;
    };
    std::vector<std::vector<Block>> ends(lmax_ + 3);
    for (uint32_t l = 1, w = 0; l <= lmax_ + 1; ++l) {
        for (const Block& b : ends[l - 1]) pool.give(b.at, b.n);
        for (; w < batches_.size() && batches_[w].level == l; ++w) {
            Batch& x = batches_[w];
            if (x.inplace && x.cls != kCopy) continue;
            if (pb) {
                const auto same = [&](const Batch& y) {
                    return y.level == l && y.cls == x.cls && y.inplace == x.inplace && y.death == x.death;
                };
                uint32_t e = w + 1;
                while (e < batches_.size() && same(batches_[e])) ++e;
                if (w == 0 || !same(batches_[w - 1])) spread_banks(&x, batches_.data() + e, pb);
            }
            if (x.inplace) continue;
            x.base = pool.take(x.n);
            for (uint32_t k = 0; k < x.n; ++k) slot_[rows_[order_[x.first + k]].val] = x.base + k;
            ends[x.death].push_back({x.base, x.n});
        }
    }
    nslots_ = pool.top();
}

// Dwords that 32 lanes' accesses of one operand name, by bank.
struct Banks {
    uint32_t dw[32][6];
    uint8_t n[32];
    uint8_t most;
    void clear() {
        std::fill(n, n + 32, 0);
        most = 0;
    }
    bool has(uint32_t d) const {
        for (uint32_t i = 0; i < n[d & 31]; ++i)
            if (dw[d & 31][i] == d) return true;
        return false;
    }
    // 256 for another pass, plus the dwords already in the bank
    uint32_t cost(uint32_t d) const {
        const uint32_t c = n[d & 31];
        return !c || has(d) ? (c || most ? 0u : 1u) : c + (c == most ? 256u : 0u);
    }
    void put(uint32_t d) {
        if (has(d)) return;
        if (n[d & 31] < 6) dw[d & 31][n[d & 31]++] = d;
        most = std::max(most, n[d & 31]);
    }
};

// Order the rows of batches [b, e) (consecutive in order_) greedily: each next
// row is the one of the first kWindow left whose operands need the fewest
// further passes of the current 32 lanes.
inline void Planner::spread_banks(const Batch* b, const Batch* e, uint32_t pb) {
    constexpr uint32_t kWindow = 128;
    std::vector<uint32_t> left;
    for (const Batch* x = b; x < e; ++x)
        left.insert(left.end(), order_.begin() + x->first, order_.begin() + x->first + x->n);
    Banks bk[3];
    size_t at = 0;   // left[at ..) are not placed
    for (const Batch* x = b; x < e; ++x)
        for (uint32_t k = 0; k < x->n; ++k) {
            if (k % 32 == 0)
                for (Banks& c : bk) c.clear();
            size_t best = at;
            uint32_t least = ~0u;
            const size_t end = k % 32 ? std::min(left.size(), at + kWindow) : at + 1;
            for (size_t i = at; i < end && least; ++i) {
                const Row& r = rows_[left[i]];
                uint32_t c = 0;
                for (uint32_t j = 0; j < r.nrd; ++j) c += bk[j].cost(slot_[r.rd[j]] * pb / 4);
                if (c < least) least = c, best = i;
            }
            const uint32_t row = left[best];
            left[best] = left[at];
            left[at++] = row;
            order_[x->first + k] = row;
            const Row& r = rows_[row];
            for (uint32_t j = 0; j < r.nrd; ++j) bk[j].put(slot_[r.rd[j]] * pb / 4);
        }
}

inline Plan Planner::tables(uint32_t pb) const {
    Plan p;
    p.nslots = nslots_;
    p.nstate = nstate_;
    p.nwaves = nw_;
    p.batch = batch_;
    const uint32_t per = batch_ == 1 ? 64 : 128;   // rows of a line
    p.a0 = 0;
    p.b0 = n_.n_pi;
    p.levels = lmax_ + 1;
    for (char x : ram_live_) p.n_ram_live += x ? 1 : 0;
    // batches to wavefronts, level by level, the costliest first to the least
    // loaded; the commit rows to the wavefronts without lane work
    std::vector<std::vector<uint32_t>> words(nw_), list(nw_);
    std::vector<uint32_t> ids;
    for (uint32_t l = 1, w = 0; l <= lmax_ + 1; ++l) {
        ids.clear();
        for (; w < batches_.size() && batches_[w].level == l; ++w) ids.push_back(w);
        const auto cost = [&](uint32_t i) { return (batches_[i].n + 63) / 64 * row_cost(batches_[i].cls); };
        std::stable_sort(ids.begin(), ids.end(), [&](uint32_t x, uint32_t y) { return cost(x) > cost(y); });
        const uint32_t w0 = l > lmax_ ? std::min(nw_ / 2, 2 + p.n_ram_live) : 0;
        std::vector<uint32_t> load(nw_, 0);
        // (the lane work beside the first levels)
        if (l == 1 && nw_ > 2) load[0] = kInputCost, load[1] = kHashCost;
        if (l == kRamLevels)
            for (uint32_t r = 0; r < p.n_ram_live && 2 + r < nw_; ++r) load[2 + r] = kRamCost;
        std::vector<std::vector<uint32_t>> mine(nw_);
        for (uint32_t i : ids) {
            const uint32_t k = (uint32_t)(std::min_element(load.begin() + w0, load.end()) - load.begin());
            load[k] += cost(i);
            mine[k].push_back(i);
        }
        for (uint32_t k = 0; k < nw_; ++k) {
            std::sort(mine[k].begin(), mine[k].end());
            for (uint32_t i : mine[k]) {
                const Batch& x = batches_[i];
                words[k].insert(words[k].end(), {x.cls | (x.n << 3), x.base * pb, 0u, 0u});
                list[k].push_back(i);
                p.wave_rows += (x.n + 63) / 64;
            }
            if (l > lmax_) continue;   // the cycle's last barrier follows the lane work
            if (mine[k].empty()) words[k].insert(words[k].end(), 4, 0u);
            words[k][words[k].size() - 4] |= 0x80000000u;
        }
    }
    p.words.assign(4 * nw_, 0);
    for (uint32_t k = 0; k < nw_; ++k) {
        while (words[k].empty() || words[k].size() % (4 * kUnroll)) words[k].insert(words[k].end(), 4, 0u);
        const uint32_t nb = (uint32_t)words[k].size() / 4;
        uint32_t line = 0;
        for (uint32_t j = 0; j < nb; ++j) {
            words[k][4 * j + 3] = line;
            words[k][4 * ((j + nb - kUnroll) % nb) + 2] = line;
            line += (((words[k][4 * j] >> 3) & 511u) + per - 1) / per;
        }
        p.words[4 * k] = (uint32_t)p.words.size();
        p.words[4 * k + 1] = nb;
        p.words.insert(p.words.end(), words[k].begin(), words[k].end());
        p.words[4 * k + 2] = (uint32_t)(p.rows.size() / per);
        for (uint32_t i : list[k]) {
            const Batch& x = batches_[i];
            const size_t at = p.rows.size();
            p.rows.resize(at + (x.n + per - 1) / per * per);
            for (uint32_t t = 0; t < p.rows.size() - at; ++t) {
                const Row& r = rows_[order_[x.first + std::min(t, x.n - 1)]];
                const uint32_t b = r.cls == kCopy ? slot_[src_ff() + r.ff] : slot_[r.rd[1]];
                const uint32_t c = r.nrd > 2 ? slot_[r.rd[2]] * pb : 0u;
                // row t of a line of two: lane t % 64, half t / 64
                const uint32_t in = t % per, to = per == 64 ? in : 2 * (in % 64) + in / 64;
                p.rows[at + t / per * per + to] = pack_row(slot_[r.rd[0]] * pb, b * pb, c, r.k1, r.k2);
            }
        }
    }
    // a batch's loads cover the most lines whatever it holds
    p.rows.resize(p.rows.size() + 64 * batch_, 0);
    p.off_po = (uint32_t)p.words.size();
    for (uint32_t v : po_val_) p.words.push_back(slot_[v] * pb);
    p.off_ram = (uint32_t)p.words.size();
    const uint32_t pw = n_.abits + 1 + n_.width;
    p.ram_words = 2 + pw;
    for (uint32_t r = 0; r < n_.n_rams; ++r) {
        if (!ram_live_[r]) continue;
        p.words.push_back(r);
        p.words.push_back(slot_[src_rd() + r * n_.width] * pb);
        for (uint32_t k = 0; k < pw; ++k) p.words.push_back(slot_[ram_val_[r * pw + k]] * pb);
    }
    p.words.resize(p.words.size() + 64, 0);   // 64 lanes load batch words at once
    return p;
}

// The plan of a checked program for workgroups of ``nwaves`` wavefronts and
// ``lds_bytes`` of LDS: its plane width in bytes, or 0 when the program runs
// level by level -- no outputs, not a plain levelised netlist, live planes
// beyond the LDS even at 8 stimuli, or no host memory to plan it in (the
// callers are C entry points, which no exception may leave).
inline uint32_t plan_program(const uint32_t* h, uint32_t nwaves, uint64_t lds_bytes, Plan* out) noexcept {
    try {
        Net net;
        if (!h[H_PO] || !read_net(h, net)) return 0;
        Planner pl(net, nwaves);
        const uint64_t slots = pl.schedule();
        // the widest planes that fit: a row costs the same for 8 stimuli as for 32
        for (uint32_t pb : {4u, 2u, 1u})
            if (slots * pb + 4 <= lds_bytes) {
                *out = pl.emit(pb);
                return pb;
            }
    } catch (const std::exception&) {
    }
    return 0;
}

}  // namespace gnplan
