// rf_gnlds.hip -- gate-level netlists in LDS: one workgroup of 16 wavefronts
// per 8, 16 or 32 stimuli runs whole cycles with every live node's plane (one
// bit per stimulus) in LDS, following the wavefront programs of rf_gnplan.h.
// No kernel boundary and no traffic to HBM but the RAM ports: a cycle is one
// pass over the program, a workgroup barrier per level.
//
// Bound (net5: 178,000 live gates, 155,000 rows, 124 KB of planes at 8 stimuli
// per workgroup, one workgroup per CU): LDS is busy 56 % of a cycle (half of
// that bank conflicts), VALU issue 39 %, the vector cache 42 %; the rest is the
// drain at 14 barriers: 26 us a cycle for 2,048 stimuli at once, against 122 us
// for 4,096 level by level through HBM, where the 31 dependent launches of a
// cycle bounded it whatever the number of stimuli. A workgroup's cycle costs
// the same for 8 stimuli as for 32, and the longest budget bounds the run, so
// small workgroups lose nothing. Batches of 2 or 6 wavefront rows instead of 4:
// 32 and 27 us. Rows loaded 8 instead of 16 bytes a lane: 35 us (the vector
// cache serves 4 lanes a cycle).
#include "rf_gnlds.h"

#include "rf_gnplan.h"
#include "rf_stim.h"
#include "rf_transpose.h"

namespace {

template <typename T>
using lds = __attribute__((address_space(3))) T;

// LDS byte address -> plane (the dynamic allocation is the only one, so it
// starts at LDS address 0).
template <typename T>
__device__ __forceinline__ uint32_t ld(uint32_t a) {
    return *reinterpret_cast<const lds<T>*>((size_t)a);
}
template <typename T>
__device__ __forceinline__ void st(uint32_t a, uint32_t v) {
    *reinterpret_cast<lds<T>*>((size_t)a) = (T)v;
}

constexpr uint32_t kMask = (1u << gnplan::kAddrBits) - 1u;

// All ones when bit ``at`` of v is set, else 0.
__device__ __forceinline__ uint32_t mask_bit(uint32_t v, int at) {
    return (uint32_t)((int32_t)(v << (31 - at)) >> 31);
}
// Three-input bit operation; the truth table has a = 0xf0, b = 0xcc, c = 0xaa.
template <uint32_t TT>
__device__ __forceinline__ uint32_t bitop3(uint32_t a, uint32_t b, uint32_t c) {
    return (uint32_t)__builtin_amdgcn_bitop3_b32((int)a, (int)b, (int)c, TT);
}
// a k b with the operator's masks at bit ``at`` of y (pack_row); bits above
// the plane are not kept.
__device__ __forceinline__ uint32_t row_op(uint32_t a, uint32_t b, uint32_t y, int at) {
    const uint32_t p = mask_bit(y, at), q = mask_bit(y, at + 1), n = mask_bit(y, at + 2);
    const uint32_t t = bitop3<0x70>(a, b, p);   // a & ~(b & p)
    return bitop3<0x68>(t, b, q) ^ n;           // q ? t ^ b : t & b
}

// The values of N wavefront rows of a class, all operand reads first.
template <uint32_t CLS, int N, typename T, int B>
__device__ __forceinline__ void row_values(const uint2 (&R)[B], uint32_t (&v)[N]) {
    uint32_t a[N], b[N], c[N];
#pragma unroll
    for (int u = 0; u < N; ++u) {
        a[u] = ld<T>(R[u].x & kMask);
        if constexpr (CLS != gnplan::kCopy) b[u] = ld<T>(R[u].y >> 14);
        if constexpr (CLS == gnplan::kPair || CLS == gnplan::kMux)
            c[u] = ld<T>(__builtin_amdgcn_alignbit(R[u].y, R[u].x, 18) & kMask);
    }
    __builtin_amdgcn_sched_barrier(0);   // (the scheduler would wait for a row before the next one's reads)
#pragma unroll
    for (int u = 0; u < N; ++u) {
        if constexpr (CLS == gnplan::kMux) v[u] = bitop3<0xca>(a[u], b[u], c[u]);
        else if constexpr (CLS == gnplan::kSingle) v[u] = row_op(a[u], b[u], R[u].y, 4);
        else if constexpr (CLS == gnplan::kPair) v[u] = row_op(row_op(a[u], b[u], R[u].y, 4), c[u], R[u].y, 7);
        else if constexpr (CLS == gnplan::kOp) v[u] = a[u] & b[u];
        else if constexpr (CLS == gnplan::kOp + 1) v[u] = a[u] | b[u];
        else if constexpr (CLS == gnplan::kOp + 2) v[u] = a[u] ^ b[u];
        else if constexpr (CLS == gnplan::kOp + 3) v[u] = ~(a[u] & b[u]);
        else v[u] = a[u];
    }
}

// A batch of n rows of one class (at most kBatch wavefront rows, all their
// operand reads before the first write: rows of a level read nothing that the
// level writes). Rows past n read what their addresses name and are dropped.
template <uint32_t CLS, typename T, int B>
__device__ __forceinline__ void batch_rows(const uint2 (&R)[B], uint32_t n, uint32_t dst, uint32_t t) {
    const uint32_t d = dst + t * (uint32_t)sizeof(T);
    const auto put = [&](int u, uint32_t v) {   // (a copy's destination is its own, in the b field)
        st<T>(CLS == gnplan::kCopy ? R[u].y >> 14 : d + u * 64 * (uint32_t)sizeof(T), v);
    };
    if constexpr (B > 1) {
        if (n > 64) {
            uint32_t v[B];
            row_values<CLS, B, T, B>(R, v);
            put(0, v[0]);
            if (n == 64 * B) {
#pragma unroll
                for (int u = 1; u < B; ++u) put(u, v[u]);
            } else {
#pragma unroll
                for (int u = 1; u < B; ++u)
                    if (t + u * 64 < n) put(u, v[u]);
            }
            return;
        }
    }
    uint32_t v[1];
    row_values<CLS, 1, T, B>(R, v);
    if (t < n) put(0, v[0]);
}

template <typename T, int B>
__device__ __forceinline__ void batch_run(const uint2 (&R)[B], uint32_t w, uint32_t dst, uint32_t t) {
    const uint32_t n = (w >> 3) & 511u, cls = w & 7u;
    if (n) {
        if (cls < gnplan::kOp) {
            if (cls == gnplan::kSingle) batch_rows<gnplan::kSingle, T, B>(R, n, dst, t);
            else if (cls == gnplan::kPair) batch_rows<gnplan::kPair, T, B>(R, n, dst, t);
            else batch_rows<gnplan::kMux, T, B>(R, n, dst, t);
        } else if (cls < gnplan::kOp + 2) {
            if (cls == gnplan::kOp) batch_rows<gnplan::kOp, T, B>(R, n, dst, t);
            else batch_rows<gnplan::kOp + 1, T, B>(R, n, dst, t);
        } else {
            if (cls == gnplan::kOp + 2) batch_rows<gnplan::kOp + 2, T, B>(R, n, dst, t);
            else if (cls == gnplan::kOp + 3) batch_rows<gnplan::kOp + 3, T, B>(R, n, dst, t);
            else batch_rows<gnplan::kCopy, T, B>(R, n, dst, t);
        }
    }
}

// The input words of cycle ``cyc`` for the workgroup's W lanes (one
// wavefront): thread t builds word t / W of lane t % W, so one 64 x 64
// transpose turns up to 64 / W words (at least the two an engine takes) into
// planes: thread t's bits [k W, (k + 1) W) are the plane of input 64 k + t.
template <typename T>
__device__ __forceinline__ uint64_t input_words(const rf_gnl_params& p, uint64_t stim, uint32_t cyc, uint32_t t) {
    constexpr uint32_t W = 8 * sizeof(T);
    const uint32_t j = t / W;
    return bp_transpose64(64u * j < p.n_pi ? rf_stim(p.seed, stim, cyc, j) : 0ull, t);
}
template <typename T>
__device__ __forceinline__ void put_inputs(const rf_gnl_params& p, uint64_t col, uint32_t t) {
#pragma unroll
    for (uint32_t k = 0; k < 2; ++k)
        if (64 * k + t < p.n_pi) st<T>(p.a0 + (64 * k + t) * sizeof(T), (uint32_t)(col >> (k * 8 * sizeof(T))));
}

// B: wavefront rows of the plan's batches.
template <typename T, int B>
__global__ void __launch_bounds__(RF_GNL_THREADS) rf_gnl_kernel(rf_gnl_params p) {
    constexpr uint32_t W = 8 * sizeof(T);          // lanes of the workgroup
    constexpr uint32_t NW = RF_GNL_THREADS / 64;
    extern __shared__ uint32_t L[];
    const uint32_t tid = threadIdx.x, t = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t lane0 = blockIdx.x * W;
    // lanes are sorted by budget, so the first one runs longest
    const uint32_t N = p.budget[lane0];
    const uint32_t kend = min(p.k1, N + 1u);
    if (N == 0 || p.k0 >= kend) return;
    const uint32_t lane = lane0 + t % W;
    const bool inb = lane < p.nlanes;
    const uint64_t stim = inb ? p.sid[lane] : 0u;
    uint32_t* img = p.image + (size_t)blockIdx.x * (p.state_bytes / 4);
    for (uint32_t i = tid; i < p.state_bytes / 4; i += RF_GNL_THREADS) L[i] = p.k0 ? img[i] : 0u;
    __syncthreads();
    if (wave == 0 && p.k0 == 0) put_inputs<T>(p, input_words<T>(p, stim, 0, t), t);
    uint64_t h = 0;
    uint32_t bud = 0;
    if (wave == 1 && t < W && inb) {
        h = p.hash[lane];
        bud = p.budget[lane];
    }
    const uint32_t po = wave == 1 && t < p.n_po ? p.words[p.off_po + t] : 0u;
    // this wavefront's program: batch words and row stream. A batch's rows are
    // loaded three batches ahead (an L2 read takes about as long as two
    // batches), always the plan's B wavefront rows, so that the loads in flight
    // are known without branches and complete in order (scalar loads would
    // make every LDS wait a wait for them too). The words of kChunk batches
    // come with one load, four lanes a batch: a load of one address by all
    // lanes would cost the vector cache as much as 16 bytes for each.
    constexpr uint32_t kLine = B > 1 ? 1024 : 512, kChunk = 15;
    const uint32_t nb = __builtin_amdgcn_readfirstlane(p.words[4 * wave + 1]);
    const uint32_t* prog = p.words + __builtin_amdgcn_readfirstlane(p.words[4 * wave]);
    const char* rows = reinterpret_cast<const char*>(p.rows) +
                       (size_t)__builtin_amdgcn_readfirstlane(p.words[4 * wave + 2]) * kLine;
    const uint32_t tl = t * (kLine / 64);
    uint2 R0[B], R1[B], R2[B];
    const auto fetch = [&](uint2(&Q)[B], uint32_t line) {
        const char* base = rows + (size_t)line * kLine;
        if constexpr (B == 1) {
            Q[0] = *reinterpret_cast<const uint2*>(base + tl);
        } else {
#pragma unroll
            for (int u = 0; u < B; u += 2) {
                const uint4 q = *reinterpret_cast<const uint4*>(base + u / 2 * kLine + tl);
                Q[u] = make_uint2(q.x, q.y);
                Q[u + 1] = make_uint2(q.z, q.w);
            }
        }
    };
    uint32_t ahead = prog[t];             // the next chunk's words
    const auto word_of = [&](uint32_t v, uint32_t j) {
        return (uint32_t)__builtin_amdgcn_readlane((int)v, (int)j);
    };
    fetch(R0, word_of(ahead, 3));
    fetch(R1, word_of(ahead, 7));
    fetch(R2, word_of(ahead, 11));
    // The lane work that waits for memory or for long chains runs beside the
    // first levels of the next cycle: wavefront 0 builds the next inputs,
    // wavefront 1 folds the last outputs into the hash, a RAM's wavefront
    // waits for the word it read and writes its planes.
    uint64_t col = 0, outs = 0, word = 0;
    uint32_t rd = ~0u;                    // planes that ``word`` is for
    const int nbytes = p.n_po <= 8 ? 1 : p.n_po <= 16 ? 2 : p.n_po <= 32 ? 4 : 8;
    const auto put_word = [&]() {
        const uint64_t c = bp_transpose64(word, t);
        if (t < p.width) st<T>(rd + t * sizeof(T), (uint32_t)c);
        rd = ~0u;
    };
    const auto fold = [&](uint32_t cyc) {
        const uint64_t v = bp_transpose64(outs, t);
        if (cyc < bud) h = rf_fnv_bytes(h, v, nbytes);
    };
    __syncthreads();
    for (uint32_t k = p.k0; k < kend; ++k) {
        uint32_t level = 0;
        if (wave == 0) col = input_words<T>(p, stim, k + 1, t);
        else if (wave == 1 && k > p.k0 && k > 1) fold(k - 2);
        for (uint32_t c = 0; c < nb; c += kChunk) {
            const uint32_t now = ahead;
            ahead = prog[4 * (c + kChunk < nb ? c + kChunk : 0u) + t];
            const uint32_t m = min(kChunk, nb - c);
            for (uint32_t j = 0; j < m; j += 3) {
                const auto step = [&](uint2(&Q)[B], uint32_t i) {
                    const uint32_t w = word_of(now, 4 * i), line = word_of(now, 4 * i + 2);
                    batch_run<T, B>(Q, w, word_of(now, 4 * i + 1), t);
                    fetch(Q, line);
                    if (w >> 31) {
                        if (++level == gnplan::kRamLevels && rd != ~0u) put_word();
                        __syncthreads();
                    }
                };
                step(R0, j);
                step(R1, j + 1);
                step(R2, j + 2);
            }
        }
        // lane work after the last level, beside the other wavefronts' commit
        // rows (their destinations are flip-flops, which nothing here touches)
        if (wave == 0) {
            for (uint32_t i = t; i < p.n_pi; i += 64) st<T>(p.b0 + i * sizeof(T), ld<T>(p.a0 + i * sizeof(T)));
            put_inputs<T>(p, col, t);
        } else if (wave == 1) {
            outs = t < p.n_po ? (uint64_t)ld<T>(po) : 0ull;
        } else {
            for (uint32_t r = wave - 2; r < p.n_ram; r += NW - 2) {
                if (rd != ~0u) put_word();     // more RAMs than wavefronts: all but the last at once
                const uint32_t* rw = p.words + p.off_ram + r * p.ram_words;
                const uint32_t ctl = t <= p.abits ? rw[2 + t] : 0u;
                const uint32_t dat = t < p.width ? rw[2 + p.abits + 1 + t] : 0u;
                const uint64_t aw = bp_transpose64(t <= p.abits ? (uint64_t)ld<T>(ctl) : 0ull, t);
                const uint64_t wd = bp_transpose64(t < p.width ? (uint64_t)ld<T>(dat) : 0ull, t);
                const uint32_t addr = (uint32_t)(aw & ((1ull << p.abits) - 1ull));
                const bool on = t < W && inb && addr < p.depth;
                uint64_t* mem = p.M + ((size_t)lane * p.n_rams + rw[0]) * p.depth;
                word = on ? mem[addr] : 0ull;
                const uint64_t wmask = p.width >= 64 ? ~0ull : ((1ull << p.width) - 1ull);
                if (on && ((aw >> p.abits) & 1ull)) mem[addr] = wd & wmask;
                rd = __builtin_amdgcn_readfirstlane(rw[1]);
            }
        }
        __syncthreads();
    }
    if (wave == 1 && kend > 1) fold(kend - 2);
    if (rd != ~0u) put_word();
    __syncthreads();
    if (wave == 1 && t < W && inb) p.hash[lane] = h;
    if (kend <= N)     // more iterations to come in the next launch
        for (uint32_t i = tid; i < p.state_bytes / 4; i += RF_GNL_THREADS) img[i] = L[i];
}

template <typename T, int B>
hipError_t launch_b(const rf_gnl_params& p, uint32_t groups, hipStream_t stream) {
    const void* fn = reinterpret_cast<const void*>(&rf_gnl_kernel<T, B>);
    hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)RF_GNL_LDS);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((rf_gnl_kernel<T, B>), dim3(groups), dim3(RF_GNL_THREADS), p.lds_bytes, stream, p);
    return hipGetLastError();
}

template <typename T>
hipError_t launch(const rf_gnl_params& p, uint32_t groups, hipStream_t stream) {
    return p.batch == 1 ? launch_b<T, 1>(p, groups, stream) : launch_b<T, gnplan::kBatch>(p, groups, stream);
}

}  // namespace

hipError_t rf_gnl_launch(const rf_gnl_params& p, uint32_t pb, uint32_t groups, hipStream_t stream) {
    if (!groups || p.lds_bytes > RF_GNL_LDS || (p.state_bytes & 3u) || p.state_bytes > p.lds_bytes)
        return hipErrorInvalidValue;
    switch (pb) {
        case 1: return launch<uint8_t>(p, groups, stream);
        case 2: return launch<uint16_t>(p, groups, stream);
        case 4: return launch<uint32_t>(p, groups, stream);
        default: return hipErrorInvalidValue;
    }
}
