// tau selection on the device (the reference tunes tau on the host inside the
// timed loop: tuneValidRate, tool.cu:438-490, over managed-memory norm maps).
//
//  - select: exact order statistic.  The fp32 norm products are non-negative,
//    so their bit patterns order like the values; a 3-pass radix select
//    (11 + 11 + 10 bits, most significant first) over the nbM*nbN*nbK products,
//    recomputed from the norm maps in every pass, finds the want-th largest.
//  - count:  number of products >= a threshold and their sum.
//  - bisect: the reference's bisection, ten of its rounds per launch: the
//    thresholds that ten rounds can visit form a binary tree of 1023 nodes, one
//    walk over the products counts all of them, and the path actually taken is
//    followed afterwards.
//
// What bounds these: a selection at 2048^3 / tile 32 is 2.6e5 products, at N = 16384
// / tile 64 1.7e7 -- a few microseconds of arithmetic -- so the time is launches,
// round trips to memory that all CUs share, and the host's wait.  Every pass
// therefore ends in the launch that counted: the workgroup that finishes last
// combines the others' results and takes the pass's decision (a separate one-thread
// walk over the 2048 bins took 30-160 us of dependent loads per pass, and
// double-precision atomics on one address are compare-and-swap loops: 15 us of 256
// workgroups' time at 2.6e5 products).  The decision is written straight to pinned
// host memory, where the host looks for it, and every launch leaves the counters
// at zero.  Few products (k_tau_small_*) are held by one workgroup, and all passes
// are one launch.
// Whole calls, norm maps and the multiply behind them included: 5024 x 4128 x 3168 at
// tile 32 to a kept fraction 667 -> 133 us, the reference's tuned 2048^3 (8 of at most
// 20 rounds) 381 -> 75 us.
// What is left in a launch of 2.6e5 products, 6.3 us for a count: five round trips past the L2 (arguments, norms, parts, ticket, parts
// again), the result's way to the host, and some 500 instructions.  (Divisions of a step's number, 64-bit addresses of its rows, wave sums by
// LDS shuffles, the tree's state read word by word and its decisions taken one after the other by one thread: count 7.35 -> 6.3 us, a bisection
// of one tree 18.75 -> 16.4, a selection 22.4 -> 21.7; 2.1e6 products 7.7 -> 6.9, 24.3 -> 21.9, 24.6 -> 23.5.)
#include "gemm_device.h"
#include "reduce_device.h"

namespace spamm {

constexpr int TAU_NTH = 1024;               // threads per workgroup
constexpr int TAU_NW = TAU_NTH / 64;
constexpr int TAU_MAXB = 256;               // one workgroup per CU at most: every one of them adds its part to the same few words
constexpr int TAU_JB_COUNT = 16;            // output columns whose products share one load of nA
constexpr int TAU_JB_TREE = 4;              // (where a product is much work: more waves, and code that is fetched sooner)
constexpr int TAU_COPIES = 2;               // global copies of a histogram: workgroups that add to one copy queue on its busy bins
constexpr int TREE_LEAVES = 1 << TREE_ROUNDS;
constexpr int TREE_COPIES = 4;              // global copies of the leaves' counts
constexpr int64_t TAU_SMALL_MAX = 24 * TAU_NTH;   // products that one workgroup holds

struct TauTune {
    double norm, up, down, rate;
    int done;
    unsigned int call;                      // whose bisection this is
    int rounds, pad_;
};

struct TauWorkspace {
    TauState st;
    TauTune tune;
    Tickets tickets;                        // workgroups of the running pass that have finished
    unsigned long long hist[3][TAU_COPIES][2048];   // one per pass: cleared together, beforehand
    unsigned long long leaf[TREE_COPIES][TREE_LEAVES];
    unsigned long long part[TAU_MAXB][2];   // per workgroup: {count, bits of the sum}
};

size_t tau_workspace_bytes() { return sizeof(TauWorkspace); }

// Every product once: a wave takes one tile row i, TAU_JB tile columns and 64 k, lane = k.  f(product,
// live) runs in all lanes; `live` is false in lanes beyond the last k.  A wave's step is one round trip
// of TAU_JB + 1 loads and some hundred instructions, so the steps are kept small and spread over as many
// waves as there are (whole rows of k per wave: 22 us instead of 15 for the last pass over 1.7e7 products).
// In two parts, as most waves have one step or a few: the first step's norms are asked for by the constructor, ahead of what a
// kernel prepares for its products.  Rows lie at a buffer's scalar offset, a step's place comes by reciprocals (TauGrid).
struct TauGrid {
    uint32_t kb, jb;             // words of 64 k, groups of TAU_JB columns
    uint32_t rec_kb, rec_jb;     // floor((2^32 - 1) / kb), (.. / jb); rec_kb = 0: steps * kb or rows * jb * jb leaves 32 bits, divide
};

template <int TAU_JB>
struct Products {
    const float *nA, *nBt;
    int nbM, nbK, nbN;
    TauGrid g;
    int64_t units, u;
    int lane, rows;              // rows: of TAU_JB, those that exist
    bool live;
    float a, b[TAU_JB];

    __device__ __forceinline__ void load() {
        uint32_t ij, i, j;
        int k0;
        if (g.rec_kb) {
            ij = __umulhi((uint32_t)u + 1u, g.rec_kb);
            k0 = (int)((uint32_t)u - ij * g.kb) * 64;
            i = __umulhi(ij + 1u, g.rec_jb);
            j = ij - i * g.jb;
        } else {
            ij = (uint32_t)(u / g.kb);
            k0 = (int)(u - (int64_t)ij * g.kb) * 64;
            i = ij / g.jb;
            j = ij % g.jb;
        }
        const int j0 = (int)j * TAU_JB, stride = nbK * 4;
        rows = nbN - j0 < TAU_JB ? nbN - j0 : TAU_JB;
        live = k0 + lane < nbK;
        const int voff = (live ? k0 + lane : nbK - 1) * 4;
        const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((void *)(nA + (int64_t)i * nbK), 0, stride, 0x00020000);
        const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc((void *)(nBt + (int64_t)j0 * nbK), 0, rows * stride, 0x00020000);
        a = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(ra, voff, 0, 0));
#pragma unroll
        for (int jj = 0; jj < TAU_JB; jj++)
            b[jj] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rb, voff, (jj < rows ? jj : rows - 1) * stride, 0));
    }
    __device__ __forceinline__ Products(const float *nA_, const float *nBt_, int nbM_, int nbK_, int nbN_, const TauGrid &g_)
        : nA(nA_), nBt(nBt_), nbM(nbM_), nbK(nbK_), nbN(nbN_), g(g_) {
        lane = threadIdx.x & 63;
        const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        units = (int64_t)nbM * g.jb * g.kb;
        u = (int64_t)blockIdx.x * TAU_NW + wave;
        if (u < units) load();
    }
    template <typename F>
    __device__ __forceinline__ void each(F &&f) {
        while (u < units) {
#pragma unroll
            for (int jj = 0; jj < TAU_JB; jj++)
                if (jj < rows) f(a * b[jj], live);
            u += (int64_t)gridDim.x * TAU_NW;
            if (u < units) load();
        }
    }
};

// One digit of the select: histogram of the PASS-th digit over the products whose higher bits equal
// the prefix found so far, then (last workgroup) the bin that holds the wanted rank.  Zero products
// never enter the histogram: sparse data would otherwise queue on one bin.  (What the first pass counted is the
// positive ones; the others counted too, an add per wave to one address, made a selection of 2.1e6 products
// with zeros among them 22 us longer: 58.4 -> 35.9, 1.6e7 81.7 -> 56.5.)
// Neighbouring k have neighbouring exponents, so the lanes of a wave meet on few bins: four copies of
// every bin, side by side, quarter the queue (one copy: 28 us for the first digit of 1.7e7 products).
// Where all products fit 32 bits, two neighbouring bins are one 64-bit word of the global histogram: half the adds of 256
// workgroups that meet some 400 bins each where the products span many exponents, and half the loads behind the ticket
// (2.6e5 products 35.3 -> 34.4 us, 1.6e7 84.1 -> 81.7).
template <int PASS>
__global__ __launch_bounds__(TAU_NTH) void k_tau_hist(const float *__restrict__ nA, const float *__restrict__ nBt, int nbM,
                                                      int nbK, int nbN, TauGrid grid, unsigned long long total, unsigned long long want0,
                                                      TauWorkspace *__restrict__ ws, TauState *__restrict__ host_out,
                                                      unsigned long long *__restrict__ host_seq, unsigned long long seq) {
    constexpr int BITS = PASS == 2 ? 10 : 11, SHIFT = PASS == 0 ? 21 : (PASS == 1 ? 10 : 0);
    constexpr int NB = 1 << BITS, COPIES = 4, PER = NB / TAU_NTH;
    __shared__ __attribute__((aligned(16))) unsigned int lh[NB * COPIES];
    __shared__ unsigned long long s_sum[TAU_NW];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    Products<TAU_JB_COUNT> products(nA, nBt, nbM, nbK, nbN, grid);
    TauState prev = {};
    if (PASS) prev = ws->st;
    for (int b = threadIdx.x; b < NB * COPIES / 4; b += TAU_NTH) reinterpret_cast<uint4 *>(lh)[b] = make_uint4(0u, 0u, 0u, 0u);
    __syncthreads();
    const uint32_t prefix = prev.prefix;
    const bool packed = total >> 32 == 0;                         // no count leaves 32 bits: two bins a word
    products.each([&](float p, bool live) {
        const bool pos = live && p > 0.0f;                        // NaN counts as 0
        const uint32_t key = __builtin_bit_cast(uint32_t, p);
        bool in = pos;
        if constexpr (PASS > 0) in = pos && (key >> (SHIFT + BITS)) == prefix;
        if (in) atomicAdd(&lh[((key >> SHIFT) & (NB - 1)) * COPIES + (lane & (COPIES - 1))], 1u);
    });
    __syncthreads();
    for (int w = threadIdx.x; w < NB / 2; w += TAU_NTH) {
        unsigned long long c[2] = {0, 0};
#pragma unroll
        for (int r = 0; r < 2 * COPIES; r++) c[r / COPIES] += lh[w * 2 * COPIES + r];
        unsigned long long *hist = ws->hist[PASS][blockIdx.x % TAU_COPIES];
        if (packed) {
            const unsigned long long both = c[0] | c[1] << 32;
            if (both) atomicAdd(&hist[w], both);
        } else {
            if (c[0]) atomicAdd(&hist[2 * w], c[0]);
            if (c[1]) atomicAdd(&hist[2 * w + 1], c[1]);
        }
    }
    if (!last_workgroup(&ws->tickets)) return;

    // thread t takes bins NB - 1 - t * PER downwards; `above` = products in the bins over its own.
    // (The loads of this step are independent and go out together: a round trip that bypasses the L2
    // is over a microsecond, and five of them one after the other were half of this kernel's time.)
    unsigned long long h[PER], mine = 0, part[PER][TAU_COPIES];
    const int top = NB - 1 - (int)threadIdx.x * PER;
    // (what this pass counted in is zero again for the next selection)
    if (packed) {                                                 // the thread's two bins are one word, or its one bin half of one
        unsigned long long both[TAU_COPIES];
#pragma unroll
        for (int r = 0; r < TAU_COPIES; r++) both[r] = agent_load(&ws->hist[PASS][r][top >> 1]);
#pragma unroll
        for (int r = 0; r < TAU_COPIES; r++) {
            if (both[r]) agent_store(&ws->hist[PASS][r][top >> 1], 0ull);
#pragma unroll
            for (int e = 0; e < PER; e++) part[e][r] = both[r] >> ((top - e) & 1 ? 32 : 0) & 0xffffffffull;
        }
    } else {
#pragma unroll
        for (int e = 0; e < PER; e++)
#pragma unroll
            for (int r = 0; r < TAU_COPIES; r++) part[e][r] = agent_load(&ws->hist[PASS][r][top - e]);
#pragma unroll
        for (int e = 0; e < PER; e++)
#pragma unroll
            for (int r = 0; r < TAU_COPIES; r++)
                if (part[e][r]) agent_store(&ws->hist[PASS][r][top - e], 0ull);
    }
#pragma unroll
    for (int e = 0; e < PER; e++) {
        h[e] = 0;
#pragma unroll
        for (int r = 0; r < TAU_COPIES; r++) h[e] += part[e][r];
        mine += h[e];
    }
    const unsigned long long incl = wave_scan(mine);
    if (lane == 63) s_sum[wave] = incl;
    // The host goes on when it sees the last pass's result, on another stream if it likes: by then nothing of this
    // launch is still on its way to the workspace (and the state in it, which no launch after this reads, stays as it is)
    if constexpr (PASS == 2) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    unsigned long long above = incl - mine;
    for (int w = 0; w < wave; w++) above += s_sum[w];
    unsigned long long want = prev.want;
    if (PASS == 0) {
        unsigned long long positive = 0;                          // (this pass counts every positive product)
        for (int w = 0; w < TAU_NW; w++) positive += s_sum[w];
        want = want0 < positive ? want0 : positive;               // zero tail: settle for the smallest positive product
        if (positive == 0 && threadIdx.x == 0) {                  // nothing but zeros: only tau = 0 keeps anything
            TauState z = {};
            z.kept = total;
            ws->st = z;
        }
    }
    if (want == 0) {                                              // (the passes after such a first one)
        if (PASS == 2 && threadIdx.x == 0) publish_result(host_out, prev, host_seq, seq);
        return;
    }
    if (above < want && want <= above + mine) {
#pragma unroll
        for (int e = 0; e < PER; e++) {
            if (above < want && want <= above + h[e]) {
                TauState st;
                st.want = want - above;                           // rank inside the bin
                st.greater = prev.greater + above;
                st.prefix = (prefix << (PASS ? BITS : 0)) | (uint32_t)(NB - 1 - (int)threadIdx.x * PER - e);
                st.tau_bits = st.prefix;
                st.kept = st.greater + h[e];
                if (PASS == 2) publish_result(host_out, st, host_seq, seq);
                else ws->st = st;
            }
            above += h[e];
        }
    }
}

// Round 0 of the bisection measures at tau = 0 and moves to the mean product (tool.cu:445-468).
__device__ __forceinline__ TauTune first_round(unsigned long long cnt, double sum, unsigned long long total, double expected, double tol,
                                               int max_rounds) {
    TauTune t = {};
    t.rate = (double)((float)cnt / (float)total);
    t.norm = t.up = t.down = 0.0;
    t.done = fabs(t.rate - expected) < tol;
    if (!t.done) t.norm = t.up = sum / (double)total;
    t.rounds = 1;
    if (t.rounds >= max_rounds) t.done = 1;
    return t;
}

// The state of the bisection passes from launch to launch, and from call to call on whatever stream: stored where every
// XCD sees it, so that nothing of it is written back after the result has been published.
__device__ __forceinline__ void store_tune(TauWorkspace *ws, const TauTune &t) {
    static_assert(sizeof(TauTune) % 8 == 0, "the state is whole 64-bit words");
    struct Words {
        unsigned long long w[sizeof(TauTune) / 8];
    };
    const Words words = __builtin_bit_cast(Words, t);
#pragma unroll
    for (unsigned i = 0; i < sizeof(TauTune) / 8; i++) agent_store(reinterpret_cast<unsigned long long *>(&ws->tune) + i, words.w[i]);
}

// (double)p >= thr over fp32 p is p >= the smallest fp32 value that is not below thr.  (Mean and thresholds are
// negative where uploaded norm maps hold negative values.)
__device__ __forceinline__ float fp32_threshold(double thr) {
    const float f = (float)thr;
    if (!((double)f < thr)) return f;
    return __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, f) + (f < 0.0f ? -1 : 1));
}

// The two numbers that a round of the bisection starts from (tool.cu:448-463), and with `tune` its
// first round: products with (double)p >= thr and the double sum of all products.  Sums of a
// workgroup and of the whole are added in a fixed order: the same norm maps give the same sum.
__global__ __launch_bounds__(TAU_NTH) void k_tau_count(const float *__restrict__ nA, const float *__restrict__ nBt, int nbM,
                                                       int nbK, int nbN, TauGrid grid, double thr, unsigned long long total, int tune,
                                                       double expected, double tol, int max_rounds, unsigned int call, int last,
                                                       TauWorkspace *__restrict__ ws, TauCounts *__restrict__ host_out,
                                                       TauResult *__restrict__ host_tune, unsigned long long *__restrict__ host_seq,
                                                       unsigned long long seq) {
    __shared__ unsigned long long s_cnt[TAU_NW];
    __shared__ double s_sum[TAU_NW];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    Products<TAU_JB_COUNT> products(nA, nBt, nbM, nbK, nbN, grid);
    const float thr32 = fp32_threshold(thr);
    unsigned long long cnt = 0;
    double sum = 0.0;
    products.each([&](float p, bool live) {
        cnt += __builtin_popcountll(__ballot(live && p >= thr32));
        sum += live ? (double)p : 0.0;
    });
    auto block_sum = [&]() {                                      // of sum and the waves' cnt, in thread 0
        sum = wave_sum(sum);
        if (lane == 0) { s_cnt[wave] = cnt; s_sum[wave] = sum; }
        __syncthreads();
        cnt = 0;
        sum = 0.0;
        for (int w = 0; w < TAU_NW; w++) { cnt += s_cnt[w]; sum += s_sum[w]; }
    };
    block_sum();
    if (threadIdx.x == 0) {
        agent_store(&ws->part[blockIdx.x][0], cnt);
        agent_store(&ws->part[blockIdx.x][1], __builtin_bit_cast(unsigned long long, sum));
    }
    if (!last_workgroup(&ws->tickets)) return;
    const bool have = threadIdx.x < gridDim.x;                    // gridDim.x <= TAU_MAXB <= TAU_NTH
    cnt = have ? agent_load(&ws->part[threadIdx.x][0]) : 0ull;
    sum = have ? __builtin_bit_cast(double, agent_load(&ws->part[threadIdx.x][1])) : 0.0;
    cnt = wave_sum(cnt);
    block_sum();
    if (threadIdx.x != 0) return;
    TauCounts tc;
    tc.count = cnt;
    tc.sum = sum;
    if (!tune) publish_result(host_out, tc, host_seq, seq);
    if (tune) {
        TauTune t = first_round(cnt, sum, total, expected, tol, max_rounds);
        t.call = call;
        store_tune(ws, t);
        const TauResult r = {t.norm, t.rate, t.done};
        if (t.done || last) publish_result(host_tune, r, host_seq, seq);
    }
}

// One step of the bisection away from a measured rate (tool.cu:469-486).  False where it leaves everything as it
// was, bit for bit: every later round then measures the same threshold and ends here again.  (Doubles run out of
// thresholds within some 5e4 rounds of any target, so no kernel runs longer whatever the caller's limit.)
__device__ __forceinline__ bool bisect_step(TauTune &t, bool above) {
    const TauTune was = t;
    const double up = was.up == was.norm ? was.up * 2 : was.up;
    t.norm = (was.norm + (above ? up : was.down)) / 2;
    t.up = above ? up : was.norm;
    t.down = above ? was.norm : was.down;
    const auto same = [](double a, double b) { return __builtin_bit_cast(unsigned long long, a) == __builtin_bit_cast(unsigned long long, b); };
    return !(same(t.norm, was.norm) && same(t.up, was.up) && same(t.down, was.down));
}

// What a lane without a product holds: no threshold keeps it.
constexpr float NO_PRODUCT = __builtin_nanf("");

// TREE_ROUNDS rounds of the bisection.  Node n of the tree (heap order, node 1 = the round to come) is the
// threshold after the answers that n's bits below the leading one spell, most significant first:
// 1 = the kept rate was above the target.  A product is looked up among the thresholds as in a search tree, one
// level per round, and counted in the leaf where it ends: node by node the products that it keeps are then those of
// the leaves from its rank up.  The thresholds of a tree are in order by themselves unless the mean is negative or
// no number (uploaded norm maps), and are ranked one by one then.
// What bounds it: round trips past the L2 -- the state, the norms, the counts, the ticket, the counts again -- and, from
// 1e7 products on, the look-up's ten LDS reads.  Whole calls, four rounds a launch, each product compared with all of 15
// thresholds, and a wait for the stream -> this (rounds 9 | 20): 64000 products 40 | 60 -> 32 | 42, 2.6e5 41 | 63 -> 32 | 43,
// 2.0e6 57 | 100 -> 40 | 56, 1.7e7 (10 rounds) 165 | 252 -> 71 | 113.
__global__ __launch_bounds__(TAU_NTH) void k_tau_tree(const float *__restrict__ nA, const float *__restrict__ nBt, int nbM,
                                                      int nbK, int nbN, TauGrid grid, unsigned long long total, double expected, double tol,
                                                      int max_rounds, unsigned int call, int last, TauWorkspace *__restrict__ ws,
                                                      TauResult *__restrict__ host_tune, unsigned long long *__restrict__ host_seq,
                                                      unsigned long long seq) {
    // a launch behind the one that ended the bisection has nothing to do, and by now the workspace may be another
    // call's, on another stream: what tells is one word, read with the others, which are used only if it says so
    TauTune start;
    {
        struct Words {
            unsigned long long w[sizeof(TauTune) / 8];
        } words;
#pragma unroll
        for (unsigned i = 0; i < sizeof(TauTune) / 8; i++) words.w[i] = agent_load(reinterpret_cast<const unsigned long long *>(&ws->tune) + i);
        start = __builtin_bit_cast(TauTune, words);
    }
    if (start.done != 0 || start.call != call) return;
    constexpr int COPIES = 4;
    __shared__ float s_heap[TREE_LEAVES];
    __shared__ float s_sorted[TREE_LEAVES];
    __shared__ unsigned int s_leaf[TREE_LEAVES * COPIES];
    __shared__ unsigned long long s_kept[TREE_LEAVES];
    __shared__ unsigned long long s_sum[TAU_NW];
    __shared__ uint16_t s_next[TREE_LEAVES];
    __shared__ int s_unsorted;
    Products<TAU_JB_TREE> products(nA, nBt, nbM, nbK, nbN, grid);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // thread n: node n and its rank among the thresholds, 1 to TREE_LEAVES - 1
    static_assert(TREE_LEAVES == TAU_NTH, "a thread per node");
    const int n = threadIdx.x;
    TauTune at_node = start;
    for (int bit = 30 - __builtin_clz(n ? n : 1); bit >= 0; bit--) bisect_step(at_node, (n >> bit) & 1);
    const float own = n ? fp32_threshold(at_node.norm) : -__builtin_inff();
    const int depth = 31 - __builtin_clz(n ? n : 1);
    int rank = n ? (2 * (n - (1 << depth)) + 1) << (TREE_ROUNDS - 1 - depth) : 0;
    if (n == 0) s_unsorted = 0;
    s_sorted[rank] = own;
    s_heap[n] = own;
#pragma unroll
    for (int c = 0; c < COPIES; c++) s_leaf[n * COPIES + c] = 0;
    __syncthreads();
    if (n && !(s_sorted[n - 1] <= s_sorted[n])) s_unsorted = 1;
    __syncthreads();
    if (s_unsorted) {                                             // (a threshold that is no number keeps nothing: last)
        const bool nan = own != own;
        int r = 0;
        for (int m = 1; m < TREE_LEAVES; m++) {
            const int at = 31 - __builtin_clz(m);
            const float o = s_sorted[(2 * (m - (1 << at)) + 1) << (TREE_ROUNDS - 1 - at)];
            r += nan ? (o == o || m <= n) : (o < own || (o == own && m <= n));
        }
        const int place = rank;
        if (n) rank = r;
        __syncthreads();
        s_sorted[rank] = own;
        __syncthreads();
        if (n) s_heap[n] = s_sorted[place];
        __syncthreads();
    }
    products.each([&](float p, bool live) {
        int at = 1;
#pragma unroll
        for (int level = 0; level < TREE_ROUNDS; level++) at = 2 * at + (p >= s_heap[at] ? 1 : 0);
        if (live && at != TREE_LEAVES) atomicAdd(&s_leaf[(at - TREE_LEAVES) * COPIES + (lane & (COPIES - 1))], 1u);
    });
    __syncthreads();
    {
        unsigned long long c = 0;
#pragma unroll
        for (int r = 0; r < COPIES; r++) c += s_leaf[n * COPIES + r];
        if (c) atomicAdd(&ws->leaf[blockIdx.x % TREE_COPIES][n], c);
    }
    if (!last_workgroup(&ws->tickets)) return;
    // products in the leaves from each thread's own up
    unsigned long long part[TREE_COPIES], incl = 0;
#pragma unroll
    for (int r = 0; r < TREE_COPIES; r++) part[r] = agent_load(&ws->leaf[r][TREE_LEAVES - 1 - n]);
#pragma unroll
    for (int r = 0; r < TREE_COPIES; r++) {
        if (part[r]) agent_store(&ws->leaf[r][TREE_LEAVES - 1 - n], 0ull);
        incl += part[r];
    }
    incl = wave_scan(incl);
    if (lane == 63) s_sum[wave] = incl;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");              // (the leaves are zero again before the result is published)
    __syncthreads();
    for (int w = 0; w < wave; w++) incl += s_sum[w];
    s_kept[TREE_LEAVES - 1 - n] = incl;
    __syncthreads();
    // every thread takes its node's decision; the path from the root then is a look-up per round, and the thread of the node where it
    // ends has the result (one thread that took the decisions in turn: 2 us)
    TauTune t = at_node;
    t.rate = (double)((float)s_kept[rank] / (float)total);
    t.rounds = start.rounds + depth;
    t.done = fabs(t.rate - expected) < tol;
    const bool above = t.rate > expected;
    if (!t.done) {
        const bool moved = bisect_step(t, above);
        t.done = ++t.rounds >= max_rounds || !moved;
    }
    s_next[n] = (uint16_t)(t.done || depth == TREE_ROUNDS - 1 ? n : 2 * n + (above ? 1 : 0));
    __syncthreads();
    int node = 1;
#pragma unroll
    for (int level = 0; level < TREE_ROUNDS - 1; level++) node = s_next[node];
    if (n != node) return;
    store_tune(ws, t);
    const TauResult res = {t.norm, t.rate, t.done};
    if (t.done || last) publish_result(host_tune, res, host_seq, seq);
}

// Small problems by one workgroup that holds every product in registers: E per thread, 1024 threads.  All
// passes of a selection and all rounds of a bisection are then one launch, with a barrier between them.
// Whole calls, launches of their own -> this: 528 products to a kept fraction 66 -> 42 us, tuned 69 -> 50; 21952
// products 49 and 59.  At 64 per thread the one CU is the slower: 32768 products tuned 83 against 75 us, 64000 to a
// kept fraction 72.5 against 71, hence TAU_SMALL_MAX.
// What bounds it: the chain of three histograms, each two barriers and a scan.  Scans by LDS shuffles, divisions -> by lane moves and
// reciprocals: a selection of 512 or 4096 products 7.45 -> 6.35 us.
template <int E>
__device__ __forceinline__ void load_products(const float *__restrict__ nA, const float *__restrict__ nBt, int nbK, int nbN, uint32_t rec_k,
                                              uint32_t rec_n, int total, float (&p)[E]) {
    // product idx = (i * nbN + j) * nbK + k; thread t has t, t + 1024, ...; quotients by rec_ = floor((2^32 - 1) / nb_), exact
    // for divisors up to TAU_SMALL_MAX
    static_assert((TAU_NTH + 1) * TAU_SMALL_MAX < 1ll << 32, "exact quotients");
    int idx = threadIdx.x;
    const int row = (int)__umulhi((uint32_t)idx + 1u, rec_k), drow = (int)__umulhi(TAU_NTH + 1u, rec_k);
    int i = (int)__umulhi((uint32_t)row + 1u, rec_n), j = row - i * nbN, k = idx - row * nbK;
    const int di = (int)__umulhi((uint32_t)drow + 1u, rec_n), dj = drow - di * nbN, dk = TAU_NTH - drow * nbK;
#pragma unroll
    for (int e = 0; e < E; e++) {
        const bool live = idx < total;
        const float a = nA[live ? i * nbK + k : 0], b = nBt[live ? j * nbK + k : 0];
        p[e] = live ? a * b : NO_PRODUCT;
        idx += TAU_NTH;
        k += dk;
        if (k >= nbK) { k -= nbK; j++; }
        j += dj;
        if (j >= nbN) { j -= nbN; i++; }
        i += di;
    }
}

template <int E>
__global__ __launch_bounds__(TAU_NTH) void k_tau_small_select(const float *__restrict__ nA, const float *__restrict__ nBt, int nbK, int nbN,
                                                              uint32_t rec_k, uint32_t rec_n, int total, unsigned int want0, TauState *__restrict__ host_out,
                                                              unsigned long long *__restrict__ host_seq, unsigned long long seq) {
    constexpr int COPIES = 4;
    __shared__ __attribute__((aligned(16))) unsigned int lh[2048 * COPIES];
    __shared__ unsigned int s_sum[TAU_NW], s_found[3];            // prefix, rank inside the bin, products above it
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    float p[E];
    load_products<E>(nA, nBt, nbK, nbN, rec_k, rec_n, total, p);
    for (int b = threadIdx.x; b < 2048 * COPIES; b += TAU_NTH) lh[b] = 0;
    unsigned int positive = 0;
#pragma unroll
    for (int e = 0; e < E; e++) positive += (unsigned int)__builtin_popcountll(__ballot(p[e] > 0.0f));    // NaN counts as 0
    if (lane == 0) s_sum[wave] = positive;
    __syncthreads();
    positive = 0;
#pragma unroll
    for (int w = 0; w < TAU_NW; w++) positive += s_sum[w];
    unsigned int want = want0 < positive ? want0 : positive, prefix = 0, greater = 0;     // zero tail: settle for the smallest positive product
    TauState st = {};
    if (want == 0) {                                              // nothing but zeros: only tau = 0 keeps anything
        st.kept = (unsigned long long)total;
        if (threadIdx.x == 0) publish_result(host_out, st, host_seq, seq);
        return;
    }
    static_for<3>([&](auto pass) {
        constexpr int PASS = decltype(pass)::value, BITS = PASS == 2 ? 10 : 11, SHIFT = PASS == 0 ? 21 : (PASS == 1 ? 10 : 0);
        constexpr int NB = 1 << BITS, PER = NB / TAU_NTH;
#pragma unroll
        for (int e = 0; e < E; e++) {
            const uint32_t key = __builtin_bit_cast(uint32_t, p[e]);
            bool in = p[e] > 0.0f;
            if constexpr (PASS > 0) in = in && (key >> (SHIFT + BITS)) == prefix;
            if (in) atomicAdd(&lh[((key >> SHIFT) & (NB - 1)) * COPIES + (lane & (COPIES - 1))], 1u);
        }
        __syncthreads();
        // thread t takes bins NB - 1 - t * PER downwards; `above` = products in the bins over its own
        unsigned int h[PER], mine = 0;
#pragma unroll
        for (int e = 0; e < PER; e++) {
            uint4 *bin = reinterpret_cast<uint4 *>(&lh[(NB - 1 - (int)threadIdx.x * PER - e) * COPIES]);
            const uint4 c = *bin;
            *bin = make_uint4(0u, 0u, 0u, 0u);
            h[e] = c.x + c.y + c.z + c.w;
            mine += h[e];
        }
        const unsigned int incl = wave_scan(mine);
        if (lane == 63) s_sum[wave] = incl;
        __syncthreads();
        unsigned int above = incl - mine;
#pragma unroll
        for (int w = 0; w < TAU_NW; w++) above += w < wave ? s_sum[w] : 0u;
#pragma unroll
        for (int e = 0; e < PER; e++) {
            if (above < want && want <= above + h[e]) {           // exactly one thread and bin
                s_found[0] = (prefix << (PASS ? BITS : 0)) | (uint32_t)(NB - 1 - (int)threadIdx.x * PER - e);
                s_found[1] = want - above;
                s_found[2] = greater + above;
                if constexpr (PASS == 2) {
                    st.want = want - above;
                    st.greater = greater + above;
                    st.prefix = st.tau_bits = s_found[0];
                    st.kept = st.greater + h[e];
                    publish_result(host_out, st, host_seq, seq);
                }
            }
            above += h[e];
        }
        if constexpr (PASS < 2) {
            __syncthreads();
            prefix = s_found[0];
            want = s_found[1];
            greater = s_found[2];
        }
    });
}

template <int E>
__global__ __launch_bounds__(TAU_NTH) void k_tau_small_tune(const float *__restrict__ nA, const float *__restrict__ nBt, int nbK, int nbN,
                                                            uint32_t rec_k, uint32_t rec_n, int total, double expected, double tol, int max_rounds,
                                                            TauResult *__restrict__ host_out, unsigned long long *__restrict__ host_seq,
                                                            unsigned long long seq) {
    __shared__ unsigned int s_cnt[2][TAU_NW];
    __shared__ double s_sum[TAU_NW];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    float p[E];
    load_products<E>(nA, nBt, nbK, nbN, rec_k, rec_n, total, p);
    double sum = 0.0;
#pragma unroll
    for (int e = 0; e < E; e++) sum += (int)threadIdx.x + e * TAU_NTH < total ? (double)p[e] : 0.0;
    sum = wave_sum(sum);
    if (lane == 0) s_sum[wave] = sum;
    int turn = 0;
    // products >= thr, of all waves
    auto count = [&](double thr) -> unsigned int {
        const float f = fp32_threshold(thr);
        unsigned int c = 0;
#pragma unroll
        for (int e = 0; e < E; e++) c += (unsigned int)__builtin_popcountll(__ballot(p[e] >= f));
        if (lane == 0) s_cnt[turn][wave] = c;
        __syncthreads();
        c = 0;
#pragma unroll
        for (int w = 0; w < TAU_NW; w++) c += s_cnt[turn][w];
        turn ^= 1;             // (the next count writes the other half: no wave is two counts ahead of another)
        return c;
    };
    // every thread follows the bisection by itself
    const unsigned int positive = count(0.0);
    sum = 0.0;
#pragma unroll
    for (int w = 0; w < TAU_NW; w++) sum += s_sum[w];
    TauTune t = first_round(positive, sum, (unsigned long long)total, expected, tol, max_rounds);
    while (!t.done) {
        t.rate = (double)((float)count(t.norm) / (float)total);
        if (fabs(t.rate - expected) < tol) break;
        const bool moved = bisect_step(t, t.rate > expected);
        if (++t.rounds >= max_rounds || !moved) break;
    }
    if (threadIdx.x == 0) {
        const TauResult res = {t.norm, t.rate, 1};
        publish_result(host_out, res, host_seq, seq);
    }
}

// once after allocation: every launch leaves the tickets and the histograms as it found them
__global__ __launch_bounds__(256) void k_tau_clear(TauWorkspace *ws) {
    const int b = blockIdx.x * 256 + threadIdx.x;                 // 8 workgroups per histogram copy
    (&ws->hist[0][0][0])[b] = 0;
    if (b < TREE_COPIES * TREE_LEAVES) (&ws->leaf[0][0])[b] = 0;
    if (b <= (int)TICKET_GROUPS) ws->tickets.t[b].n = 0;
}

hipError_t launch_tau_clear(void *workspace, hipStream_t s) {
    k_tau_clear<<<3 * TAU_COPIES * 2048 / 256, 256, 0, s>>>((TauWorkspace *)workspace);
    return hipGetLastError();
}

static int64_t tau_products(int64_t nbM, int64_t nbK, int64_t nbN) { return nbM * nbK * nbN; }

bool tau_tune_small(int64_t nbM, int64_t nbK, int64_t nbN) { return tau_products(nbM, nbK, nbN) <= TAU_SMALL_MAX; }

static TauGrid tau_steps(int64_t nbM, int64_t nbK, int64_t nbN, int jb) {
    const uint64_t kb = (uint64_t)(nbK + 63) / 64, groups = (uint64_t)(nbN + jb - 1) / jb, rows = (uint64_t)nbM * groups;
    const bool short_ = rows * kb * kb < 0xffffffffull && rows * groups < 0xffffffffull;
    return {(uint32_t)kb, (uint32_t)groups, short_ ? 0xffffffffu / (uint32_t)kb : 0u, short_ ? 0xffffffffu / (uint32_t)groups : 0u};
}

static unsigned tau_grid(int64_t nbM, int64_t nbK, int64_t nbN, int jb = TAU_JB_COUNT) {
    const int64_t units = nbM * ((nbN + jb - 1) / jb) * ((nbK + 63) / 64);
    const int64_t blocks = (units + TAU_NW - 1) / TAU_NW;
    return (unsigned)(blocks < TAU_MAXB ? blocks : TAU_MAXB);
}

// For passes whose workgroups count in 32 bits and leave no part of their own (k_tau_hist, k_tau_tree): as many workgroups
// that none has much over 2^30 products.  (A multiply that fits the card's memory stays below it; norm maps alone,
// 65535 tiles a side, hold up to 2^48 products.)
static unsigned tau_count_grid(int64_t nbM, int64_t nbK, int64_t nbN, int jb) {
    const unsigned grid = tau_grid(nbM, nbK, nbN, jb);
    const int64_t total = tau_products(nbM, nbK, nbN);
    return total >> 31 > grid / 2 ? (unsigned)(total >> 30) : grid;
}

hipError_t launch_tau_select(const float *nA, const float *nBt, int64_t nbM, int64_t nbK, int64_t nbN,
                             unsigned long long want, void *workspace, TauState *host_out, unsigned long long *host_seq,
                             unsigned long long seq, hipStream_t s) {
    TauWorkspace *ws = (TauWorkspace *)workspace;
    const int64_t n = tau_products(nbM, nbK, nbN);
    if (n <= TAU_SMALL_MAX) {
#define SPAMM_SELECT(E) k_tau_small_select<E><<<1, TAU_NTH, 0, s>>>(nA, nBt, (int)nbK, (int)nbN, 0xffffffffu / (uint32_t)nbK, 0xffffffffu / (uint32_t)nbN, (int)n, (unsigned int)want, host_out, host_seq, seq)
        if (n <= 8 * TAU_NTH) SPAMM_SELECT(8);
        else SPAMM_SELECT(24);
#undef SPAMM_SELECT
        return hipGetLastError();
    }
    const unsigned grid = tau_count_grid(nbM, nbK, nbN, TAU_JB_COUNT);
    const unsigned long long total = (unsigned long long)n;
    const TauGrid steps = tau_steps(nbM, nbK, nbN, TAU_JB_COUNT);
    k_tau_hist<0><<<grid, TAU_NTH, 0, s>>>(nA, nBt, (int)nbM, (int)nbK, (int)nbN, steps, total, want, ws, host_out, host_seq, seq);
    k_tau_hist<1><<<grid, TAU_NTH, 0, s>>>(nA, nBt, (int)nbM, (int)nbK, (int)nbN, steps, total, want, ws, host_out, host_seq, seq);
    k_tau_hist<2><<<grid, TAU_NTH, 0, s>>>(nA, nBt, (int)nbM, (int)nbK, (int)nbN, steps, total, want, ws, host_out, host_seq, seq);
    return hipGetLastError();
}

hipError_t launch_tau_count(const float *nA, const float *nBt, int64_t nbM, int64_t nbK, int64_t nbN, double thr,
                            void *workspace, TauCounts *host_out, unsigned long long *host_seq, unsigned long long seq, hipStream_t s) {
    TauWorkspace *ws = (TauWorkspace *)workspace;
    k_tau_count<<<tau_grid(nbM, nbK, nbN), TAU_NTH, 0, s>>>(nA, nBt, (int)nbM, (int)nbK, (int)nbN, tau_steps(nbM, nbK, nbN, TAU_JB_COUNT), thr,
                                                       (unsigned long long)nbM * nbK * nbN, 0, 0.0, 0.0, 0, 0u, 0, ws, host_out, nullptr,
                                                       host_seq, seq);
    return hipGetLastError();
}

hipError_t launch_tau_tune_small(const float *nA, const float *nBt, int64_t nbM, int64_t nbK, int64_t nbN, double expected, double tol,
                                 int max_rounds, TauResult *host_out, unsigned long long *host_seq, unsigned long long seq, hipStream_t s) {
    const int64_t n = tau_products(nbM, nbK, nbN);
#define SPAMM_TUNE(E) k_tau_small_tune<E><<<1, TAU_NTH, 0, s>>>(nA, nBt, (int)nbK, (int)nbN, 0xffffffffu / (uint32_t)nbK, 0xffffffffu / (uint32_t)nbN, (int)n, expected, tol, max_rounds, host_out, host_seq, seq)
    if (n <= 8 * TAU_NTH) SPAMM_TUNE(8);
    else SPAMM_TUNE(24);
#undef SPAMM_TUNE
    return hipGetLastError();
}

hipError_t launch_tau_tune(const float *nA, const float *nBt, int64_t nbM, int64_t nbK, int64_t nbN, double expected, double tol,
                           int max_rounds, bool first, int passes, unsigned int call, void *workspace, TauResult *host_out,
                           unsigned long long *host_seq, unsigned long long seq, hipStream_t s) {
    TauWorkspace *ws = (TauWorkspace *)workspace;
    const unsigned long long total = (unsigned long long)nbM * nbK * nbN;
    if (first)
        k_tau_count<<<tau_grid(nbM, nbK, nbN), TAU_NTH, 0, s>>>(nA, nBt, (int)nbM, (int)nbK, (int)nbN, tau_steps(nbM, nbK, nbN, TAU_JB_COUNT), 0.0, total, 1, expected, tol,
                                                           max_rounds, call, passes == 0, ws, nullptr, host_out, host_seq, seq);
    for (int p = 0; p < passes; p++)
        k_tau_tree<<<tau_count_grid(nbM, nbK, nbN, TAU_JB_TREE), TAU_NTH, 0, s>>>(nA, nBt, (int)nbM, (int)nbK, (int)nbN, tau_steps(nbM, nbK, nbN, TAU_JB_TREE), total, expected, tol,
                                                                             max_rounds, call, p == passes - 1, ws, host_out, host_seq, seq);
    return hipGetLastError();
}

}  // namespace spamm
