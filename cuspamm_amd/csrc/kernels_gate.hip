// Stage 2: the tau gate.
//
// Replaces the gating prologue that the reference re-runs inside every
// multiply block (cuSpAMM.cu:302-334): bitmap of nA[i,k]*nB[k,j] >= tau
// (fp32 multiply, fp32 compare, :305-306), serial O(n^2) compaction
// (:315-325) and a shared-memory tree count (:328-334).  Here one workgroup
// owns one macro tile (256 x 256 elements of C = MT x MT output tiles):
//   gate     a wave takes 64 k at a time, lane = k: the comparisons of the macro
//            tile's norm pairs are the lane's bits, the set of tiles that keep its
//            k; transposed across the wave they are the tiles' bitmaps, which go
//            to memory with the per-tile counts;
//   list     each k with a bit set is an entry of the macro tile's union list,
//            those kept by every tile first; a scan of the words' entry counts
//            places them.  The union list is what the gated GEMM walks; its
//            length and the kept-product total are the work counts used to order
//            macro tiles for load balance.
// The reference's compacted per-tile list (offset[], :315-325) is the bitmap's
// set bits in ascending order; nothing downstream reads it, so it is produced
// from the bitmap only when asked for (k_klist).
#include "gemm_device.h"

namespace spamm {

// lo[lane idx] = low word, hi[lane idx] = high word of a wave-uniform 64-bit m; idx must fold to
// a constant (unrolled loops).  On gfx90a and later a VALU instruction that reads an SGPR needs
// two wait states after the VALU instruction that wrote it (here: the compare behind the ballot).
// The compiler inserts them only around instructions it can see, not around inline assembly, so
// the s_nop is part of it.
__device__ __forceinline__ void set_lane2(int &lo, int &hi, uint64_t m, int idx) {
    // (readfirstlane: under register pressure the compiler may hold the uniform words in VGPRs)
    const int mlo = __builtin_amdgcn_readfirstlane((int)(uint32_t)m);
    const int mhi = __builtin_amdgcn_readfirstlane((int)(uint32_t)(m >> 32));
    asm("s_nop 1\n\tv_writelane_b32 %0, %2, %4\n\tv_writelane_b32 %1, %3, %4"
        : "+v"(lo), "+v"(hi)
        : "s"(mlo), "s"(mhi), "n"(idx));
}

template <int CTRL>
__device__ __forceinline__ int dpp(int v) {
    return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xf, 0xf, true);
}

// 64 x 64 bit-matrix transpose across a wave: lane t holds row t; on return lane b holds column b (bit t of the result = bit b
// of lane t's input).  Six butterfly steps, each swapping the off-diagonal j x j blocks of lane pairs (l, l ^ j), without LDS: the
// blocks of 32 and of 16 are swapped by instructions of their own, bytes picked by a permute, and what stays is a rotate and a
// bitwise select.
__device__ __forceinline__ uint64_t transpose64(uint64_t x, int lane) {
    const auto h = __builtin_amdgcn_permlane32_swap((uint32_t)x, (uint32_t)(x >> 32), false, false);
    uint32_t v[2] = {h[0], h[1]};
    const uint32_t sel16 = lane & 16 ? 0x07060302u : 0x05040100u, sel8 = lane & 8 ? 0x03070105u : 0x06020400u;
    const uint32_t keep4 = lane & 4 ? 0xf0f0f0f0u : 0x0f0f0f0fu, keep2 = lane & 2 ? 0xccccccccu : 0x33333333u, keep1 = lane & 1 ? 0xaaaaaaaau : 0x55555555u;
    const uint32_t turn4 = lane & 4 ? 4u : 28u, turn2 = lane & 2 ? 2u : 30u, turn1 = lane & 1 ? 1u : 31u;
    auto part = [](uint32_t w, uint32_t other, uint32_t keep, uint32_t turn) {
        return (w & keep) | (__builtin_amdgcn_alignbit(other, other, turn) & ~keep);
    };
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const auto r = __builtin_amdgcn_permlane16_swap(v[i], v[i], false, false);       // the pair's even row's, its odd row's
        uint32_t w = __builtin_amdgcn_perm(r[1], r[0], sel16);
        w = __builtin_amdgcn_perm((uint32_t)dpp<0x128>((int)w), w, sel8);                // lane ^ 8
        w = part(w, (uint32_t)dpp<0x1B>(dpp<0x141>((int)w)), keep4, turn4);              // 7 - lane, ^ 3: lane ^ 4
        w = part(w, (uint32_t)dpp<0x4E>((int)w), keep2, turn2);                          // lane ^ 2
        v[i] = part(w, (uint32_t)dpp<0xB1>((int)w), keep1, turn1);                       // lane ^ 1
    }
    return (uint64_t)v[1] << 32 | v[0];
}

template <int MT>
struct GateCfg {
    static constexpr int NT = MT * MT;             // output tiles per macro tile
    static constexpr int NTP = NT < 8 ? 8 : NT;    // bitmap rows per 64-k word in LDS (a transposed word needs 64 * NTP bits)
    static constexpr int BT = MT < 4 ? MT : 4;     // a wave's block of tiles per dimension
    static constexpr int QD = MT / BT;
    static constexpr int NQ = QD * QD;
    static constexpr uint64_t FULL = NT == 64 ? ~0ull : ((1ull << NT) - 1ull);
};

// A macro tile whose bitmaps exceed a CU's LDS (K / tile beyond ~19 400 at tile 32): the k range is walked in chunks of `cw` 64-k
// words, twice -- once to count, once to place the list entries -- and the bitmaps of a chunk are recomputed for the second walk;
// the per-word summaries cover all words.
template <int MT, int NTH = (MT == 2 ? 64 : 256)>
__global__ __launch_bounds__(NTH) void k_gate_chunks(GateBuffers g, int nbM, int nbK, int nbN, int nMacN, float tau, int cw) {
    using G = GateCfg<MT>;
    constexpr int NW = NTH / 64;
    constexpr int NT = G::NT, NTP = G::NTP, BT = G::BT;
    extern __shared__ uint64_t smem[];
    const int words = (nbK + 63) >> 6;
    uint64_t *lmask = smem;                                  // [cw][NTP]: tile bitmaps, later transposed in place
    uint64_t *luf = smem + (size_t)cw * NTP;                 // [words][2]: union word, kept-by-all word
    int *wfull = reinterpret_cast<int *>(luf + 2 * (size_t)words);   // [words + 1] prefix of full entries
    int *wpart = wfull + (words + 1);                        // [words + 1] prefix of partial entries

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int macro = blockIdx.x;
    const int mi = macro / nMacN, mj = macro % nMacN;

    // ---- phase 1: bitmaps.  Item = (64-k word, block of BT x BT tiles); two items per step so
    // that their norm loads are in flight together (each is a cache round trip).  Loads are
    // unconditional from clamped addresses; what lies outside the matrix is masked after the
    // ballot (k per lane, tile rows / columns per wave).
    struct Item {
        float pa[BT], pb[BT];
    };
    auto load_item = [&](int w0, int item, Item &it) {
        const int q = item % G::NQ, w = w0 + item / G::NQ;
        const int k = w * 64 + lane;
        const int kc = k < nbK ? k : nbK - 1;
#pragma unroll
        for (int a = 0; a < BT; a++) {
            const int i = mi * MT + (q / G::QD) * BT + a;
            it.pa[a] = g.nA[(int64_t)(i < nbM ? i : nbM - 1) * nbK + kc];
        }
#pragma unroll
        for (int b = 0; b < BT; b++) {
            const int j = mj * MT + (q % G::QD) * BT + b;
            it.pb[b] = g.nBt[(int64_t)(j < nbN ? j : nbN - 1) * nbK + kc];
        }
    };
    // whole macro tile inside the matrix: only the last k word may need masking
    const bool interior = (mi + 1) * MT <= nbM && (mj + 1) * MT <= nbN;
    auto gate_item = [&](int w0, int item, const Item &it) {
        const int q = item % G::NQ, wl = item / G::NQ, w = w0 + wl;
        const int ti0 = (q / G::QD) * BT, tj0 = (q % G::QD) * BT;
        int mlo = 0, mhi = 0;                 // lane a*BT+b collects the word of tile (a, b)
        if (interior && (w + 1) * 64 <= nbK) {
#pragma unroll
            for (int a = 0; a < BT; a++)
#pragma unroll
                for (int b = 0; b < BT; b++) {
                    const uint64_t m = __ballot(it.pa[a] * it.pb[b] >= tau);
                    set_lane2(mlo, mhi, m, a * BT + b);
                }
        } else {
            const uint64_t kmask = __ballot(w * 64 + lane < nbK);
#pragma unroll
            for (int a = 0; a < BT; a++)
#pragma unroll
                for (int b = 0; b < BT; b++) {
                    // wave-uniform all-ones / zero: is tile (a, b) of the block inside the matrix
                    const uint64_t inside =
                        0ull - (uint64_t)((mi * MT + ti0 + a < nbM) & (mj * MT + tj0 + b < nbN));
                    const uint64_t m = __ballot(it.pa[a] * it.pb[b] >= tau) & kmask & inside;
                    set_lane2(mlo, mhi, m, a * BT + b);
                }
        }
        if (lane < BT * BT)
            lmask[(size_t)wl * NTP + (ti0 + lane / BT) * MT + tj0 + lane % BT] =
                ((uint64_t)(uint32_t)mhi << 32) | (uint32_t)mlo;
    };
    auto build_bitmaps = [&](int w0, int cwn) {
        const int n_items = G::NQ * cwn;
        for (int it0 = wave; it0 < n_items; it0 += 2 * NW) {
            const int it1 = it0 + NW;
            Item i0, i1;
            load_item(w0, it0, i0);
            if (it1 < n_items) load_item(w0, it1, i1);
            gate_item(w0, it0, i0);
            if (it1 < n_items) gate_item(w0, it1, i1);
        }
    };
    // ---- phase 2b: transpose every word in place: entry b of word w becomes the set of tiles
    // (bit t = tile t of the macro tile) that keep k = 64 w + b, NTP bits wide
    auto tile_bits = [&](int wl, int b) -> uint64_t {
        if constexpr (NTP == 64) return lmask[(size_t)wl * 64 + b];
        else if constexpr (NTP == 16) return reinterpret_cast<const uint16_t *>(lmask + (size_t)wl * 16)[b];
        else return reinterpret_cast<const uint8_t *>(lmask + (size_t)wl * 8)[b];
    };
    auto transpose_words = [&](int w0, int cwn, bool record) {
        for (int wl = wave; wl < cwn; wl += NW) {
            const uint64_t row = lane < NT ? lmask[(size_t)wl * NTP + lane] : 0ull;
            const uint64_t bits = transpose64(row, lane);
            const uint64_t u = __ballot(bits != 0ull), f = __ballot(bits == G::FULL);
            // the wave has read all rows of the word before any lane writes its column
            if constexpr (NTP == 64) lmask[(size_t)wl * 64 + lane] = bits;
            else if constexpr (NTP == 16) reinterpret_cast<uint16_t *>(lmask + (size_t)wl * 16)[lane] = (uint16_t)bits;
            else reinterpret_cast<uint8_t *>(lmask + (size_t)wl * 8)[lane] = (uint8_t)bits;
            if (record && lane == 0) {
                const int w = w0 + wl;
                luf[2 * w] = u;
                luf[2 * w + 1] = f;
                wfull[w + 1] = __builtin_popcountll(f);
                wpart[w + 1] = __builtin_popcountll(u & ~f);
            }
        }
    };

    int cnt = 0;                               // wave 0, lane < NT: kept k of tile `lane`
    int n_full = 0, n_part = 0, rot_f = 0, rot_p = 0;
    // One walk over the k chunks; `pass` is a compile-time tag: 0 counts, 1 places.
    auto walk = [&](auto pass_tag) {
        constexpr int pass = decltype(pass_tag)::value;
        int w0 = 0;
        do {
            const int cwn = words - w0 < cw ? words - w0 : cw;
            build_bitmaps(w0, cwn);
            __syncthreads();
            if constexpr (pass == 0) {
                // ---- phase 2a: per-tile counts and the bitmaps to memory
                if (wave == 0 && lane < NT)
                    for (int wl = 0; wl < cwn; wl++) cnt += __builtin_popcountll(lmask[(size_t)wl * NTP + lane]);
                const float inv_words = 1.0f / (float)cwn;     // e < 2^16, cwn <= 1024: the quotient below is exact
                for (int e = threadIdx.x; e < NT * cwn; e += NTH) {
                    const int t = (int)(((float)e + 0.5f) * inv_words), wl = e - t * cwn;
                    const int i = mi * MT + t / MT, j = mj * MT + t % MT;
                    if (i < nbM && j < nbN) g.mask[((int64_t)i * nbN + j) * words + w0 + wl] = lmask[(size_t)wl * NTP + t];
                }
                __syncthreads();
            }
            transpose_words(w0, cwn, pass == 0);
            __syncthreads();
            if constexpr (pass == 1) {
                // ---- phase 2c: union list with per-tile bits.  Entries whose k is kept by every
                // tile of the macro tile ("full") come first, then the partial ones, each group
                // in ascending k rotated to the anchor: the GEMM runs a branch-free loop over the
                // first group.  (k_small lists its units' k in the same order; C's bits depend on it.)
                const int k1 = (w0 + cwn) * 64 < nbK ? (w0 + cwn) * 64 : nbK;
                for (int k = w0 * 64 + threadIdx.x; k < k1; k += NTH) {
                    const int w = k >> 6, b = k & 63;
                    const uint64_t bits = tile_bits(w - w0, b);
                    if (bits != 0ull) {
                        const uint64_t u = luf[2 * w], f = luf[2 * w + 1];
                        const uint64_t below = (1ull << b) - 1ull;
                        int pos;
                        if (bits == G::FULL) {
                            pos = wfull[w] + __builtin_popcountll(f & below) - rot_f;
                            if (pos < 0) pos += n_full;
                        } else {
                            pos = wpart[w] + __builtin_popcountll(u & ~f & below) - rot_p;
                            if (pos < 0) pos += n_part;
                            pos += n_full;
                        }
                        uint32_t need = 0;
#pragma unroll
                        for (int a = 0; a < MT; a++) {
                            const uint32_t rowbits = (uint32_t)(bits >> (a * MT)) & ((1u << MT) - 1u);
                            if (rowbits) need |= 1u << a;
                            need |= rowbits << 8;
                        }
                        MacroEntry en;
                        en.k = (uint32_t)k;
                        en.need = need;
                        en.mask_lo = (uint32_t)bits;
                        en.mask_hi = (uint32_t)(bits >> 32);
                        g.macro_list[(int64_t)macro * nbK + pos] = en;
                    }
                }
                __syncthreads();     // the next chunk's bitmaps overwrite these
            }
            w0 += cw;
        } while (w0 < words);
    };
    walk(std::integral_constant<int, 0>{});
    // ---- between the walks: inclusive scans over the words give each word's offset in its group
    if (threadIdx.x == 0) { wfull[0] = 0; wpart[0] = 0; }
    __syncthreads();
    if (words < 64) {
        if (wave == 0) {
            int vf = lane <= words ? wfull[lane] : 0, vp = lane <= words ? wpart[lane] : 0;
#pragma unroll
            for (int off = 1; off < 64; off <<= 1) {
                const int tf = __shfl_up(vf, off, 64), tp = __shfl_up(vp, off, 64);
                if (lane >= off) { vf += tf; vp += tp; }
            }
            if (lane <= words) { wfull[lane] = vf; wpart[lane] = vp; }
        }
        __syncthreads();
    } else {
        // Hillis-Steele in LDS
        for (int off = 1; off <= words; off <<= 1) {
            int addf[1024 / NTH + 1], addp[1024 / NTH + 1];        // words <= 1024
            int n = 0;
            for (int w = threadIdx.x; w <= words; w += NTH) {
                addf[n] = w >= off ? wfull[w - off] : 0;
                addp[n] = w >= off ? wpart[w - off] : 0;
                n++;
            }
            __syncthreads();
            n = 0;
            for (int w = threadIdx.x; w <= words; w += NTH) {
                wfull[w] += addf[n];
                wpart[w] += addp[n];
                n++;
            }
            __syncthreads();
        }
    }
    n_full = wfull[words];
    n_part = wpart[words];
    // Each group is rotated to start at an anchor k shared by the whole super
    // tile (the k where its diagonal would sit): the workgroups of a super
    // tile run together on one XCD, and walking k from a common start keeps
    // them on the same A row panels and B column panels at the same time.
    {
        const int anchor = list_anchor(mi, mj, MT, nbM, nbK, nbN);
        const int wa = anchor >> 6, ba = anchor & 63;
        const uint64_t u = luf[2 * wa], f = luf[2 * wa + 1];
        const uint64_t below = (1ull << ba) - 1ull;
        rot_f = wfull[wa] + __builtin_popcountll(f & below);     // entries of each group below the anchor
        rot_p = wpart[wa] + __builtin_popcountll(u & ~f & below);
    }
    walk(std::integral_constant<int, 1>{});
    // per-tile counts and the macro tile's kept-product total
    int work = 0;
    if (wave == 0) {
        if (lane < NT) {
            const int i = mi * MT + lane / MT, j = mj * MT + lane % MT;
            if (i < nbM && j < nbN) g.counts[(int64_t)i * nbN + j] = cnt;
        }
        work = cnt;
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) work += __shfl_xor(work, off, 64);
    }
    if (threadIdx.x == 0) {
        g.macro_count[2 * macro] = n_full + n_part;
        g.macro_count[2 * macro + 1] = n_full;
        g.macro_work[macro] = work;
    }
}

// The gate of one macro tile.  A wave takes whole 64-k words, lane = k: the MT + MT norms of its k come in at once, and the MT * MT
// comparisons are the lane's own bits -- the set of tiles that keep its k, which is what the list needs.  Norms are neither negative nor NaN
// as a rule, so that their products order like their bit patterns: a comparison is a product, a subtraction, and a shift
// that takes the sign in.  (A word with others in it, or a tau that is NaN, is compared as floats.)  A word in which not even
// the largest norms' product is kept is done with there.  The tiles' bitmaps are the words' transposes.
// One barrier: behind it every wave has all words' unions, places them by a scan of its own, and lists the words it gated.
// NTH threads: 256, or 64 for macro tiles of 2 x 2 output tiles (tile 128), whose few comparisons give three of four waves
// nothing to do.
// What bounds it: instructions, and for few macro tiles their chain.  A wave per 4 x 4 tiles with a ballot and two lane writes a
// comparison, bitmaps in LDS and their transposes by LDS shuffles, against this; gate and schedule together (the schedule's part is 4 to
// 5 us up to 64 super tiles, 12 at 128, 24 at 512): tile 32 5024^3 10.1 -> 7.1 us, 12032^3 31.6 -> 22.3; tile 64 8192^3 9.6 -> 8.1,
// 10048^3 15.7 -> 12.3, 16384^3 (band) 26.4 -> 20.0; tile 128 32768^3 (band) 49.5 -> 34.4.
template <int MT, int NTH = (MT == 2 ? 64 : 256)>
__global__ __launch_bounds__(NTH) void k_gate(GateBuffers g, int nbM, int nbK, int nbN, float tau) {
    using G = GateCfg<MT>;
    constexpr int NW = NTH / 64, NT = G::NT;
    constexpr int STEP = MT == 8 ? 1 : (MT == 4 ? 2 : 4);     // words whose norms a wave has in flight
    asm volatile("" : "+s"(g.nA), "+s"(g.nBt), "+s"(g.counts), "+s"(g.mask), "+s"(g.macro_list), "+s"(g.macro_count), "+s"(g.macro_work),
                 "+s"(nbM), "+s"(nbK), "+s"(nbN), "+s"(tau));
    extern __shared__ __attribute__((aligned(16))) uint64_t smem[];
    __shared__ int s_cnt[NW][64];
    const int words = (nbK + 63) >> 6;
    ulonglong2 *s_uf = reinterpret_cast<ulonglong2 *>(smem);                   // [words] union, kept by all
    uint32_t *s_pre = reinterpret_cast<uint32_t *>(s_uf + words);              // [words, even] entries before the word: kept by all | others << 16
    typedef typename std::conditional<MT == 8, uint64_t, typename std::conditional<MT == 4, uint16_t, uint8_t>::type>::type Bits;
    Bits *s_bits = reinterpret_cast<Bits *>(s_pre + ((words + 1) & ~1));       // [words][64]

    const int lane = threadIdx.x & 63, wave = NW == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int mi = blockIdx.y, mj = blockIdx.x;
    const int64_t macro = (int64_t)mi * gridDim.x + mj;
    const int rows = nbM - mi * MT < MT ? nbM - mi * MT : MT, cols = nbN - mj * MT < MT ? nbN - mj * MT : MT;
    const bool interior = rows == MT && cols == MT;
    uint64_t inside = 0;                                                       // tiles of the macro tile that exist
#pragma unroll
    for (int a = 0; a < MT; a++) inside |= a < rows ? ((1ull << cols) - 1ull) << (a * MT) : 0ull;
    const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((void *)(g.nA + (int64_t)mi * MT * nbK), 0, rows * nbK * 4, 0x00020000);
    const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc((void *)(g.nBt + (int64_t)mj * MT * nbK), 0, cols * nbK * 4, 0x00020000);
    const uint32_t tau_bits = tau > 0.0f ? __float_as_uint(tau) : 0u;
    const int ti = lane / MT, tj = lane % MT;
    const bool tile_lane = lane < NT && ti < rows && tj < cols;                // lane = tile
    const int64_t tile = (int64_t)(mi * MT + ti) * nbN + mj * MT + tj;
    auto below = [](uint64_t m) { return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u)); };

    int cnt = 0;                               // lane < NT: kept k of tile `lane` in the wave's words
    const bool in_regs = words <= NW * STEP;
    uint64_t bits_[STEP];
    for (int w0 = wave; w0 < words; w0 += NW * STEP) {
        uint32_t a[STEP][MT], b[STEP][MT];
#pragma unroll
        for (int n = 0; n < STEP; n++) {
            const int w = w0 + n * NW, k = w * 64 + lane;
            if (w >= words) break;
            const int voff = k < nbK ? k * 4 : 0x40000000;
#pragma unroll
            for (int x = 0; x < MT; x++) {
                a[n][x] = __builtin_amdgcn_raw_buffer_load_b32(ra, voff, (x < rows ? x : rows - 1) * (nbK * 4), 0);
                b[n][x] = __builtin_amdgcn_raw_buffer_load_b32(rb, voff, (x < cols ? x : cols - 1) * (nbK * 4), 0);
            }
        }
#pragma unroll
        for (int n = 0; n < STEP; n++) {
            const int w = w0 + n * NW;
            if (w >= words) break;
            const bool live = w * 64 + lane < nbK;
            uint32_t amax = a[n][0], bmax = b[n][0];
#pragma unroll
            for (int x = 1; x < MT; x++) {
                amax = a[n][x] > amax ? a[n][x] : amax;
                bmax = b[n][x] > bmax ? b[n][x] : bmax;
            }
            uint64_t bits = 0, row = 0, u = 0, f = 0;
            const bool plain = __ballot((amax > bmax ? amax : bmax) >= 0x7f800000u) == 0ull && tau == tau;
            if (!plain || __ballot(live && __uint_as_float(amax) * __uint_as_float(bmax) >= tau) != 0ull) {
                if (plain) {
                    uint32_t half[2] = {0u, 0u};
#pragma unroll
                    for (int t = NT - 1; t >= 0; t--) {
                        const uint32_t p = __float_as_uint(__uint_as_float(a[n][t / MT]) * __uint_as_float(b[n][t % MT]));
                        half[t / 32] = __builtin_amdgcn_alignbit(half[t / 32], p - tau_bits, 31);
                    }
                    bits = ~((uint64_t)half[1] << 32 | half[0]) & G::FULL;
                } else {
#pragma unroll
                    for (int t = 0; t < NT; t++)
                        bits |= __uint_as_float(a[n][t / MT]) * __uint_as_float(b[n][t % MT]) >= tau ? 1ull << t : 0ull;
                }
                if (!interior) bits &= inside;
                bits = live ? bits : 0ull;
                u = __ballot(bits != 0ull);
                f = __ballot(bits == G::FULL);
                row = transpose64(bits, lane);
                cnt += __builtin_popcountll(row);
                if (!in_regs) s_bits[w * 64 + lane] = (Bits)bits;
            }
            bits_[n] = bits;
            if (tile_lane) g.mask[tile * words + w] = row;
            if (lane == 0) s_uf[w] = ulonglong2{u, f};
        }
    }
    s_cnt[wave][lane] = cnt;
    __syncthreads();

    // Where each word's entries lie: those kept by every tile of the macro tile ("full") first, then the partial ones.  (Where
    // several waves are, all write the same.)
    uint32_t before = 0;
    for (int v0 = 0; v0 < words; v0 += 64) {
        const int v = v0 + lane;
        const ulonglong2 uf = s_uf[v < words ? v : 0];
        const uint32_t own = v < words ? (uint32_t)__builtin_popcountll(uf.y) | (uint32_t)__builtin_popcountll(uf.x & ~uf.y) << 16 : 0u;
        const uint32_t incl = wave_scan(own);
        if (v < words) s_pre[v] = before + incl - own;
        before += (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
    }
    __builtin_amdgcn_wave_barrier();
    const int n_full = (int)(before & 0xffffu), n_part = (int)(before >> 16);
    if (wave == 0) {                           // per-tile counts and the macro tile's kept-product total
        int sum = 0;
#pragma unroll
        for (int v = 0; v < NW; v++) sum += s_cnt[v][lane];
        if (tile_lane) g.counts[tile] = sum;
        const int work = wave_sum(sum);
        if (lane == 0) {
            g.macro_count[2 * macro] = n_full + n_part;
            g.macro_count[2 * macro + 1] = n_full;
            g.macro_work[macro] = work;
        }
    }
    if (before == 0u) return;
    // Each group in ascending k, rotated to start at an anchor k shared by the whole super tile (the k where its diagonal would
    // sit): the workgroups of a super tile run together on one XCD, and walking k from a common start keeps them on the same A row
    // panels and B column panels at the same time.  (k_small lists its units' k in the same order; C's bits depend on it.)
    const int anchor = list_anchor(mi, mj, MT, nbM, nbK, nbN), wa = anchor >> 6;
    const ulonglong2 anchor_uf = s_uf[wa];
    const uint64_t below_a = (1ull << (anchor & 63)) - 1ull;
    const uint32_t at_a = s_pre[wa];
    const int rot_f = (int)(at_a & 0xffffu) + __builtin_popcountll(anchor_uf.y & below_a);         // entries of each group below the anchor
    const int rot_p = (int)(at_a >> 16) + __builtin_popcountll(anchor_uf.x & ~anchor_uf.y & below_a);
    const __amdgpu_buffer_rsrc_t rl = __builtin_amdgcn_make_buffer_rsrc((void *)(g.macro_list + macro * nbK), 0, nbK * (int)sizeof(MacroEntry), 0x00020000);
    auto list_word = [&](int w, uint64_t bits) {
        const ulonglong2 uf = s_uf[w];
        const uint32_t pre = s_pre[w];
        int pf = (int)(pre & 0xffffu) + below(uf.y) - rot_f, pp = (int)(pre >> 16) + below(uf.x & ~uf.y) - rot_p;
        pf = pf < 0 ? pf + n_full : pf;
        pp = pp < 0 ? pp + n_full + n_part : pp + n_full;
        const int pos = bits == G::FULL ? pf : pp;
        uint32_t need = 0;                     // rows, columns of the macro tile that keep this k
        if constexpr (MT == 8) {
            uint32_t c = (uint32_t)bits | (uint32_t)(bits >> 32);
            c |= c >> 16;
            need = ((c | c >> 8) & 0xffu) << 8;
#pragma unroll
            for (int h = 0; h < 2; h++) {
                uint32_t x = (uint32_t)(bits >> (32 * h));
                x |= x >> 4;
                x |= x >> 2;
                x = (x | x >> 1) & 0x01010101u;
                need |= ((x * 0x10204080u) >> 28) << (4 * h);
            }
        } else {
#pragma unroll
            for (int x = 0; x < MT; x++) {
                const uint32_t rowbits = (uint32_t)bits >> (x * MT) & ((1u << MT) - 1u);
                need |= (rowbits ? 1u << x : 0u) | rowbits << 8;
            }
        }
        const u32x4 en = {(uint32_t)(w * 64 + lane), need, (uint32_t)bits, (uint32_t)(bits >> 32)};
        __builtin_amdgcn_raw_buffer_store_b128(en, rl, bits != 0ull ? pos * (int)sizeof(MacroEntry) : 0x40000000, 0, 0);
    };
    if (in_regs) {
#pragma unroll
        for (int n = 0; n < STEP; n++)
            if (wave + n * NW < words && __ballot(bits_[n] != 0ull) != 0ull) list_word(wave + n * NW, bits_[n]);
    } else {
        for (int w = wave; w < words; w += NW)
            if (__builtin_amdgcn_readfirstlane((int)(s_uf[w].x != 0ull))) list_word(w, (uint64_t)s_bits[w * 64 + lane]);
    }
}

// Schedule for the GEMM.  Macro tiles are grouped into super tiles of
// SUPER_M x SUPER_N (= 32, one per CU of an XCD); workgroups are dispatched
// round-robin over the n_xcd XCDs of the device, so workgroup b runs on XCD
// b % n_xcd and is the (b / n_xcd)-th workgroup that XCD starts (n_xcd = 1: one
// flat sequence, for devices that are not whole XCDs of 32 CUs).
//   1. Super tiles are ranked by descending length (entries of their macro
//      tiles' union lists: that, not the kept-product count, is the time a
//      workgroup takes) and dealt to the XCDs: every XCD owns whole super
//      tiles, so the workgroups sharing one L2 share A row panels and B column
//      panels.  Up to LPT_MAX_SUPER super tiles are dealt greedily, each to the
//      XCD with the least length so far (at most `rounds` per XCD, the size
//      the grid and the order buffer are laid out for); a plain snake deal by
//      rank leaves XCDs up to 18 % apart when a problem has only a few super
//      tiles per XCD, and the slowest XCD sets the kernel's time.  Beyond that
//      size the deal is the snake (the serial greedy loop would take longer
//      than it saves, and many super tiles per XCD even out by themselves).
//   2. Inside an XCD the computing macro tiles run super tile by super tile
//      (measured on banded inputs, heaviest-first classes inside an XCD did
//      not shorten the tail but pulled neighbours apart: 10 % more L2 misses).
//   3. Macro tiles with nothing kept come last in each XCD's sequence: their
//      workgroups only write zeros and start when CUs fall idle at the end.
// Output: order[x * P + q] = macro tile id of XCD x's q-th workgroup for
// q < sched[8 + x] (entries beyond are not written), sched[x] = number of
// computing items, sched[8 + x] = number of all items.
// What bounds it: one workgroup on an idle chip, so its time is latencies one after the other.
// The macro tiles' results are read once, by all threads, along C's rows; what the later steps need of them
// -- a length and a set of computing macro tiles per super tile -- stays in LDS, ranks come from
// prefix sums where the key is only "holds work", the serial deals run in one wave on lane
// moves inside a row (DPP) instead of trips through LDS, and every thread writes its own part of
// the sequences, the tables of four super tiles in flight.  By the kernel trace, first form -> before: 16384^2 of C (128 super
// tiles, band) 16.6 -> 12.1 us, 32768^2 (512, band) 52.9 -> 24.3.  Then reads along the rows, the band's groups dealt by two
// sorts of eight lanes, divisions by reciprocals and sequences four at a time, gate and schedule together: 16384^2 20.0 -> 17.6 us,
// 32768^2 34.4 -> 27.1.  Up to 64 super tiles are k_order_few's.
// Super tiles along C's rows, and floor((2^32 - 1) / them): exact quotients, there are at most ORDER_MAX_SUPER super tiles
struct SuperGrid {
    int n;
    uint32_t rec;
    __device__ __forceinline__ int origin(int sid) const {               // first macro tile row, column
        const int si = (int)__umulhi((uint32_t)sid + 1u, rec);
        return si * SUPER_M << 16 | (sid - si * n) * SUPER_N;
    }
};

// Offset of a macro tile beyond C in the buffer of kept products, and, doubled (which leaves 31 bits, so it is unsigned), in that of the
// lists' lengths: neither holds it, and zero comes back.
constexpr uint32_t NO_MACRO = 0x40000000u;

struct Super {
    uint32_t len, comp, work;       // entries of its macro tiles' lists, computing macro tiles (bit: slot), kept products
};
// Sums over every eight lanes, in all of them
__device__ __forceinline__ Super super_of_eight(Super s) {
    auto eight = [&](auto ctrl) {
        s.len += (uint32_t)dpp<decltype(ctrl)::value>((int)s.len);
        s.work += (uint32_t)dpp<decltype(ctrl)::value>((int)s.work);
        s.comp |= (uint32_t)dpp<decltype(ctrl)::value>((int)s.comp);
    };
    eight(std::integral_constant<int, 0xB1>{});          // lane ^ 1
    eight(std::integral_constant<int, 0x4E>{});          // lane ^ 2
    eight(std::integral_constant<int, 0x141>{});         // 7 - lane: the other four
    return s;
}

// Every eight lanes' keys in order, the least (DOWN: the greatest) in the first
template <bool DOWN>
__device__ __forceinline__ uint32_t sort8(uint32_t k, int lane) {
    auto step = [&](auto ctrl, int upper) {
        const uint32_t o = (uint32_t)dpp<decltype(ctrl)::value>((int)k), lo = k < o ? k : o, hi = k < o ? o : k;
        k = (upper != 0) != DOWN ? hi : lo;
    };
    constexpr std::integral_constant<int, 0xB1> x1{};
    constexpr std::integral_constant<int, 0x4E> x2{};
    step(x1, lane & 1);
    step(std::integral_constant<int, 0x1B>{}, lane & 2);         // 3 - lane of the four
    step(x1, lane & 1);
    step(std::integral_constant<int, 0x141>{}, lane & 4);        // 7 - lane of the eight
    step(x2, lane & 2);
    step(x1, lane & 1);
    return k;
}

__global__ __launch_bounds__(1024) void k_order(GateBuffers g, int nMacM, int nMacN, SuperGrid sup,
                                                int n_super, int rounds, int n_xcd) {
    extern __shared__ __attribute__((aligned(16))) int swork[];               // [n_super + 8] length; at the end, computing macro tiles before an XCD's r-th super tile
    int *sempty = swork + n_super + MAX_XCD;                                  // [n_super + 8] at the end: empty macro tiles before it
    uint32_t *scomp = reinterpret_cast<uint32_t *>(sempty + n_super + MAX_XCD);  // [n_super] computing macro tiles (bit: slot)
    int *srank_id = reinterpret_cast<int *>(scomp + n_super);                 // [n_super] super tile origin by rank,
    uint16_t *sdeal = reinterpret_cast<uint16_t *>(srank_id + n_super);      // then (dealt by table) [n_xcd][rounds] rank of each XCD's r-th super tile
    __shared__ unsigned long long total;
    __shared__ int s_with_work, s_count[16], s_len[64], s_orig[64];
    __shared__ int s_cnt[MAX_XCD], s_before[MAX_XCD], s_nall[MAX_XCD];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, wave_u = __builtin_amdgcn_readfirstlane(wave);
    const uint64_t below = (1ull << lane) - 1ull;
    const int P = rounds * SUPER_M * SUPER_N;
    if (threadIdx.x == 0) { total = 0; s_with_work = 0; }
    __syncthreads();
    {
        const __amdgpu_buffer_rsrc_t work_of = __builtin_amdgcn_make_buffer_rsrc((void *)g.macro_work, 0, nMacM * nMacN * 4, 0x00020000);
        const __amdgpu_buffer_rsrc_t count_of = __builtin_amdgcn_make_buffer_rsrc((void *)g.macro_count, 0, nMacM * nMacN * 8, 0x00020000);
        unsigned long long mine = 0;
        int with_work = 0;
        // A wave reads 64 macro tiles of each of a super tile row's rows, a column a lane: eight super tiles.  (By super tiles, four macro
        // tiles a thread, an instruction touched 32 lines: 512 super tiles 19000 clocks.)
        static_assert(SUPER_N == 8, "eight lanes a super tile");
        const int across = (sup.n + 7) / 8, strips = (nMacM + SUPER_M - 1) / SUPER_M * across;
        const uint32_t across_rec = 0xffffffffu / (uint32_t)across;
#pragma unroll 2
        for (int strip = wave_u; strip < strips; strip += 16) {
            const int si = (int)__umulhi((uint32_t)strip + 1u, across_rec), sj = (strip - si * across) * 8 + (lane >> 3);
            const int mj = sj * SUPER_N + (lane & 7), mi0 = si * SUPER_M;
            uint32_t w[SUPER_M], l[SUPER_M];
#pragma unroll
            for (int a = 0; a < SUPER_M; a++) {
                const uint32_t off = mi0 + a < nMacM && mj < nMacN ? (uint32_t)((mi0 + a) * nMacN + mj) * 4u : NO_MACRO;
                w[a] = __builtin_amdgcn_raw_buffer_load_b32(work_of, (int)off, 0, 0);
                l[a] = __builtin_amdgcn_raw_buffer_load_b32(count_of, (int)(off * 2u), 0, 0);
            }
            Super sp = {0, 0, 0};
#pragma unroll
            for (int a = 0; a < SUPER_M; a++) {
                sp.len += l[a];
                sp.work += w[a];
                sp.comp |= (l[a] ? 1u << (a * SUPER_N) : 0u);
            }
            sp.comp <<= lane & 7;
            sp = super_of_eight(sp);
            const bool leads = (lane & 7) == 0 && sj < sup.n;
            if (leads) { swork[si * sup.n + sj] = (int)sp.len; scomp[si * sup.n + sj] = sp.comp; }
            mine += leads ? sp.work : 0u;
            with_work += __builtin_popcountll(__ballot(leads && sp.len > 0));
        }
        mine = wave_sum(mine);
        if (lane == 0 && mine) { atomicAdd(&total, mine); atomicAdd(&s_with_work, with_work); }
    }
    __syncthreads();
    // How the super tiles are dealt to the XCDs (sdeal, or the snake formula in dealt):
    //   DEAL_LPT    few super tiles hold work: ranked by length, each goes to the XCD with the
    //               least length so far (pure balance);
    //   DEAL_BAND   at most BAND_DEAL_MAX super tiles hold work and they are at most
    //               60 % of all (a narrow band): ranked in
    //               row-major order, those with work first; every group of n_xcd consecutive
    //               ones -- neighbours along the band that read the same operand panels -- runs
    //               at the same time, one per XCD, and inside a group the heaviest goes to the
    //               XCD with the least length so far.  Measured against the snake: -4 to -6 %
    //               GEMM time on exponential-decay bands that keep 10 % (N = 16384), -2 % at
    //               N = 32768, but +1 to +3 % when most super tiles hold work (algebraic decay,
    //               30 % kept), hence the condition;
    //   DEAL_SNAKE  ranked by length, dealt in snake order (no table: any number of super tiles).
    enum { DEAL_LPT, DEAL_BAND, DEAL_SNAKE };
    const int n_ne = s_with_work;               // super tiles with work
    const int deal = n_super > LPT_MAX_SUPER ? DEAL_SNAKE
                     : (n_ne <= LPT_GREEDY_MAX ? DEAL_LPT
                        : (n_ne <= BAND_DEAL_MAX && 5 * n_ne <= 3 * n_super ? DEAL_BAND : DEAL_SNAKE));
    // Ranking: super tiles with work before those without; in the snake and the greedy deal by
    // descending length, equal lengths by index, in the band deal by index.  srank_id[rank] becomes
    // the super tile's origin.
    constexpr int RANK_SORT_MIN = 512;
    if (deal != DEAL_SNAKE) {
        // by index first: prefix sums of "holds work" (the lengths move to their ranks)
        constexpr int STEPS = LPT_MAX_SUPER / 1024;
        int len_[STEPS], rank_[STEPS], ne = 0;
#pragma unroll
        for (int n = 0; n < STEPS; n++) {
            if (n * 1024 >= n_super) break;
            const int sid = n * 1024 + threadIdx.x;
            const int len = sid < n_super ? swork[sid] : 0;
            const uint64_t m = __ballot(len > 0);
            if (lane == 0) s_count[wave] = __builtin_popcountll(m);
            __syncthreads();
            int before = ne, here = ne;
#pragma unroll
            for (int v = 0; v < 16; v++) {
                before += v < wave ? s_count[v] : 0;
                here += s_count[v];
            }
            before += __builtin_popcountll(m & below);
            len_[n] = len;
            rank_[n] = len > 0 ? before : n_ne + (sid - before);
            ne = here;
            __syncthreads();
        }
#pragma unroll
        for (int n = 0; n < STEPS; n++) {
            const int sid = n * 1024 + threadIdx.x;
            if (sid >= n_super) break;
            const int rank = rank_[n], origin = sup.origin(sid);
            swork[rank] = len_[n];
            srank_id[rank] = origin;
            if (deal == DEAL_LPT && rank < n_ne) { s_len[rank] = len_[n]; s_orig[rank] = origin; }
        }
        __syncthreads();
        if (wave == 0 && deal == DEAL_LPT) {
            // the (at most 64) super tiles with work by length: lane = one of them
            int len = lane < n_ne ? s_len[lane] : 0, rank = 0;
            const int origin = lane < n_ne ? s_orig[lane] : 0;
            for (int j = 0; j < n_ne; j++) {
                const int lj = __builtin_amdgcn_readlane(len, j);
                rank += lj > len || (lj == len && j < lane);
            }
            if (lane < n_ne) { s_len[rank] = len; srank_id[rank] = origin; }
            __builtin_amdgcn_wave_barrier();
            len = lane < n_ne ? *const_cast<volatile int *>(&s_len[lane]) : 0;
            // lane x < n_xcd keeps XCD x's length so far and its number of super tiles; the
            // least-loaded XCD with room is the minimum of (length, lane) over eight lanes
            // (lengths stay far below 2^28: at most LPT_GREEDY_MAX super tiles of 32 lists)
            const int x = lane;
            uint32_t load = 0;
            int cnt = 0;
            for (int r = 0; r < n_ne; r++) {
                uint32_t key = (x < n_xcd && cnt < rounds) ? (load << 3) | (uint32_t)x : ~0u, o;
                o = (uint32_t)dpp<0xB1>((int)key); key = o < key ? o : key;        // lane ^ 1
                o = (uint32_t)dpp<0x4E>((int)key); key = o < key ? o : key;        // lane ^ 2
                o = (uint32_t)dpp<0x141>((int)key); key = o < key ? o : key;       // 7 - lane: the other four
                if ((int)(key & 7u) == x) {
                    sdeal[x * rounds + cnt] = (uint16_t)r;
                    cnt++;
                    load += (uint32_t)__builtin_amdgcn_readlane(len, r);
                }
            }
            if (x < MAX_XCD) s_cnt[x] = cnt;
        }
        if (wave == 0 && deal == DEAL_BAND) {
            // every eight lanes: the XCDs by their length so far and the group's super tiles by theirs, both sorted with
            // the number in the key; the n-th shortest XCD takes the n-th heaviest super tile.  (One XCD may be dealt all super
            // tiles: its key needs the 32nd bit.)
            static_assert((uint64_t)BAND_DEAL_MAX * SUPER_M * SUPER_N * 65535 * 8 + MAX_XCD < 0xfffffff0u, "an XCD's key stays below the absent ones'");
            const int x = lane & 7;
            const int ngroups = (n_ne + n_xcd - 1) / n_xcd;
            auto weight = [&](int g2) -> int { const int r = g2 * n_xcd + x; return x < n_xcd && r < n_ne ? swork[r] : -1; };     // -1: no super tile
            uint32_t load = x < n_xcd ? (uint32_t)x : 0xfffffff0u + (uint32_t)x;      // length << 3 | XCD; absent ones stay behind all others
            int w = weight(0);
            for (int g2 = 0; g2 < ngroups; g2++) {
                const int wn = weight(g2 + 1);
                load = sort8<false>(load, lane);
                const uint32_t heavy = sort8<true>((uint32_t)(w + 1) << 3 | (uint32_t)(7 - x), lane);
                const int wm = (int)(heavy >> 3) - 1;
                if (wm > 0) {                    // (the last group may have fewer super tiles than XCDs)
                    if (lane < MAX_XCD) sdeal[(load & 7u) * rounds + g2] = (uint16_t)(g2 * n_xcd + 7 - (int)(heavy & 7u));
                    load += (uint32_t)wm << 3;
                }
                if (g2 == ngroups - 1 && lane < n_xcd) s_cnt[load & 7u] = g2 + (wm > 0);
                w = wn;
            }
        }
        __syncthreads();
        // super tiles with nothing kept (ranks n_ne ..) fill the XCDs' remaining slots in order
        if (threadIdx.x < n_xcd) {
            int before = 0;
            for (int v = 0; v < (int)threadIdx.x; v++) before += rounds - s_cnt[v];
            s_before[threadIdx.x] = before;
        }
    } else if (n_super <= RANK_SORT_MIN) {
        // rank = number of super tiles that come first, n_super^2 comparisons with the j range cut
        // into `parts` pieces so that all 1024 threads take part
        int parts = 2;
        while (parts < 32 && n_super * parts * 2 <= (int)blockDim.x) parts *= 2;
        for (int sid = threadIdx.x; sid < n_super; sid += blockDim.x) srank_id[sid] = 0;
        __syncthreads();
        const int chunk = (n_super + parts - 1) / parts;
        for (int e = threadIdx.x; e < n_super * parts; e += blockDim.x) {
            const int sid = e % n_super, part = e / n_super;
            const int w = swork[sid];
            const int j1 = (part + 1) * chunk < n_super ? (part + 1) * chunk : n_super;
            int rank = 0;
            for (int j = part * chunk; j < j1; j++) {
                const int kj = swork[j];
                rank += (kj > w) || (kj == w && j < sid);
            }
            if (rank) atomicAdd(&srank_id[sid], rank);
        }
        __syncthreads();
        const int sid = threadIdx.x;              // n_super <= RANK_SORT_MIN < blockDim.x: one super tile per thread
        const int rank = sid < n_super ? srank_id[sid] : 0;
        __syncthreads();
        if (sid < n_super) srank_id[rank] = sup.origin(sid);
    } else {
        // a bitonic sort of the indices in LDS (padded to a power of two with indices >= n_super,
        // which sort last): log^2 steps of one compare-exchange per thread instead of n_super
        // comparisons per super tile on this one CU (150 us at 2048 super tiles)
        int np2 = 2 * RANK_SORT_MIN;
        while (np2 < n_super) np2 <<= 1;
        int *sidx = srank_id;                     // [np2]
        for (int i = threadIdx.x; i < np2; i += blockDim.x) sidx[i] = i;
        __syncthreads();
        for (int k = 2; k <= np2; k <<= 1)
            for (int j = k >> 1; j > 0; j >>= 1) {
                for (int t = threadIdx.x; t < np2 / 2; t += blockDim.x) {
                    const int i = ((t & ~(j - 1)) << 1) | (t & (j - 1)), l = i | j;
                    const int a = sidx[i], b = sidx[l];
                    const int ka = a < n_super ? swork[a] : -1, kb = b < n_super ? swork[b] : -1;
                    const bool a_first = ka > kb || (ka == kb && a < b);
                    if (a_first != ((i & k) == 0)) { sidx[i] = b; sidx[l] = a; }
                }
                __syncthreads();
            }
        // sidx[rank] = super tile; every thread turns its own slots into origins
        for (int r = threadIdx.x; r < n_super; r += blockDim.x) srank_id[r] = sup.origin(sidx[r]);
    }
    __syncthreads();

    // rank of XCD x's r-th super tile; n_super and beyond: none
    auto dealt = [&](int x, int r) -> int {
        if (deal == DEAL_SNAKE) return r * n_xcd + ((r & 1) ? n_xcd - 1 - x : x);
        return r < s_cnt[x] ? (int)sdeal[x * rounds + r] : n_ne + s_before[x] + r - s_cnt[x];
    };
    auto sid_of = [&](int origin) -> int { return (origin >> 16) / SUPER_M * sup.n + (origin & 0xffff) / SUPER_N; };
    // computing macro tiles go to the front of the XCD's sequence in order, empty ones to the back: one wave
    // per XCD adds up how many of each come before its r-th super tile
    if (wave < n_xcd) {
        const int x = wave;
        int nc = 0, ne = 0;
        for (int r0 = 0; r0 < rounds; r0 += 64) {
            const int r = r0 + lane, sr = r < rounds ? dealt(x, r) : n_super;
            int c = 0, e = 0;
            if (sr < n_super) {
                const int origin = srank_id[sr], hm = nMacM - (origin >> 16), wn = nMacN - (origin & 0xffff);
                c = __builtin_popcount(scomp[sid_of(origin)]);
                e = (hm < SUPER_M ? hm : SUPER_M) * (wn < SUPER_N ? wn : SUPER_N) - c;
            }
            uint32_t incl = (uint32_t)c | (uint32_t)e << 16;              // (64 super tiles: at most 2048 of each)
            const uint32_t own = incl;
#pragma unroll
            for (int off = 1; off < 64; off <<= 1) {
                const uint32_t o = __shfl_up(incl, off, 64);
                if (lane >= off) incl += o;
            }
            const uint32_t last = __builtin_amdgcn_readlane(incl, 63), first = incl - own;
            if (r < rounds) {
                swork[x * rounds + r] = nc + (int)(first & 0xffffu);
                sempty[x * rounds + r] = ne + (int)(first >> 16);
            }
            nc += (int)(last & 0xffffu);
            ne += (int)(last >> 16);
        }
        if (lane == 0) {
            s_nall[x] = nc + ne;
            g.sched[x] = nc;
            g.sched[MAX_XCD + x] = nc + ne;
            g.sched[2 * MAX_XCD + x] = 0;      // ticket counter of the persistent GEMM
        }
    }
    if (threadIdx.x == 0) g.kept->total = (int64_t)total;
    __syncthreads();
    // the sequences, all waves: XCD x by 16 / n_xcd of them, half a wave per super tile, lane = macro tile
    {
        const int x = wave % n_xcd, per = 2 * 16 / n_xcd, slot = lane % (SUPER_M * SUPER_N);
        const int nall = s_nall[x], cnt = deal == DEAL_SNAKE ? 0 : s_cnt[x], rest = deal == DEAL_SNAKE ? 0 : n_ne + s_before[x] - cnt;
        const uint32_t before = (1u << slot) - 1u;
        constexpr int UNROLL = 4;                // super tiles whose tables a half wave has in flight
        for (int r0 = wave / n_xcd * 2 + lane / (SUPER_M * SUPER_N); r0 < rounds; r0 += UNROLL * per) {
            int at[UNROLL], origin[UNROLL], first[UNROLL], empty[UNROLL];
            uint32_t comp[UNROLL];
#pragma unroll
            for (int u = 0; u < UNROLL; u++) {
                const int r = r0 + u * per;
                at[u] = n_super;                 // its rank; n_super: none
                if (r < rounds) at[u] = deal == DEAL_SNAKE ? r * n_xcd + ((r & 1) ? n_xcd - 1 - x : x) : (r < cnt ? (int)sdeal[x * rounds + r] : rest + r);
            }
#pragma unroll
            for (int u = 0; u < UNROLL; u++) {
                const int r = r0 + u * per < rounds ? r0 + u * per : 0;
                origin[u] = srank_id[at[u] < n_super ? at[u] : 0];
                first[u] = swork[x * rounds + r];
                empty[u] = sempty[x * rounds + r];
            }
#pragma unroll
            for (int u = 0; u < UNROLL; u++) comp[u] = scomp[sid_of(origin[u])];
#pragma unroll
            for (int u = 0; u < UNROLL; u++) {
                const int oi = origin[u] >> 16, oj = origin[u] & 0xffff;
                const int mi = oi + slot / SUPER_N, mj = oj + slot % SUPER_N;
                const int c = __builtin_popcount(comp[u] & before);
                const int wn = nMacN - oj < SUPER_N ? nMacN - oj : SUPER_N;       // (slots before this one that exist, less the computing ones)
                const int q = (comp[u] >> slot) & 1u ? first[u] + c : nall - 1 - (empty[u] + (slot / SUPER_N) * wn + slot % SUPER_N - c);
                if (at[u] < n_super && mi < nMacM && mj < nMacN) g.order[x * P + q] = mi * nMacN + mj;
            }
        }
    }
}

// The schedule of at most 64 super tiles, a super tile a lane: every wave ranks and deals all of them for itself, in registers, and
// then lays out the sequence of one XCD (fewer XCDs: several waves share one).  Dealt as by k_order, which
// with so few always deals greedily; fewer super tiles than XCDs (C of at most 7 x 32 macro tiles) are not dealt whole, which would
// leave XCDs empty -- 2048^3 at tile 32 is two of them, 64 workgroups on a quarter of the chip -- but the macro
// tiles themselves, consecutive ones in row-major order (neighbours along a row share the A panel) in equal chunks, one per XCD,
// unranked.
// What bounds it: its chain of instructions, alone on the chip: a load, a barrier, a readlane and a compare per rank, a deal of 14
// instructions per super tile.  Against k_order, which has ranks and deals go through LDS with some twenty barriers
// among 16 waves, gate and schedule together: 5120^2 of C (15 super tiles) 12.3 -> 8.0 us, 8192^2 (32, 10 % kept) 13.9 -> 9.6,
// 10048^2 (50) 21.4 -> 15.7.  The line is the wave's 64 lanes.
constexpr int ORDER_FEW = 64;
constexpr int ORDER_FEW_WAVES = 8;
static_assert(ORDER_FEW <= LPT_GREEDY_MAX && MAX_XCD <= ORDER_FEW_WAVES, "always the greedy deal; a wave for every XCD");
__global__ __launch_bounds__(ORDER_FEW_WAVES * 64) void k_order_few(const int32_t *macro_work, const int32_t *macro_count, int32_t *order, int32_t *sched,
                                                                  KeptProducts *kept, int nMacM, int nMacN, SuperGrid sup,
                                                                  int n_super, int rounds, int xcd_shift) {
    asm volatile("" : "+s"(macro_work), "+s"(macro_count), "+s"(order), "+s"(sched), "+s"(kept), "+s"(nMacM), "+s"(nMacN), "+s"(sup.n),
                 "+s"(sup.rec), "+s"(n_super), "+s"(rounds), "+s"(xcd_shift));
    __shared__ Super s_super[ORDER_FEW];
    __shared__ u32x4 s_seq[ORDER_FEW + MAX_XCD];     // [n_xcd][rounds] origin, computing macro tiles, of the XCD's ones before it computing | empty << 16
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n_xcd = 1 << xcd_shift, n_macro = nMacM * nMacN, P = rounds * SUPER_M * SUPER_N;
    auto below = [](uint64_t m) { return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u)); };
    {
        const __amdgpu_buffer_rsrc_t work_of = __builtin_amdgcn_make_buffer_rsrc((void *)macro_work, 0, n_macro * 4, 0x00020000);
        const __amdgpu_buffer_rsrc_t count_of = __builtin_amdgcn_make_buffer_rsrc((void *)macro_count, 0, n_macro * 8, 0x00020000);
        const int sid = threadIdx.x >> 3, at = threadIdx.x & 7;
        const int origin = sup.origin(sid), mi = (origin >> 16) + (at >> 1), mj = (origin & 0xffff) + (at & 1) * 4;
        const uint32_t first = (uint32_t)(mi * nMacN + mj) * 4u;
        const int room = sid < n_super && mi < nMacM ? nMacN - mj : 0;
        uint32_t w[4], l[4];
#pragma unroll
        for (int b = 0; b < 4; b++) {
            const uint32_t off = b < room ? first + b * 4u : NO_MACRO;
            w[b] = __builtin_amdgcn_raw_buffer_load_b32(work_of, (int)off, 0, 0);
            l[b] = __builtin_amdgcn_raw_buffer_load_b32(count_of, (int)(off * 2u), 0, 0);
        }
        Super sp = {l[0] + l[1] + l[2] + l[3], 0, w[0] + w[1] + w[2] + w[3]};
#pragma unroll
        for (int b = 0; b < 4; b++) sp.comp |= l[b] ? 1u << (at * 4 + b) : 0u;
        sp = super_of_eight(sp);
        if (at == 0) s_super[sid] = sp;
    }
    __syncthreads();
    if (wave == ORDER_FEW_WAVES - 1) {
        const unsigned long long total = wave_sum((unsigned long long)s_super[lane].work);
        if (lane == 0) kept->total = (int64_t)total;
    }
    if (n_super < n_xcd) {                      // one round of at most 28 macro tiles per XCD
        if (wave < n_xcd) {
            const int chunk = (n_macro + n_xcd - 1) >> xcd_shift, m = wave * chunk + lane;
            const bool in = lane < chunk && m < n_macro;
            const bool comp = in && macro_work[in ? m : 0] > 0;
            const uint64_t bi = __ballot(in), bc = __ballot(comp), be = bi & ~bc;
            const int nall = __builtin_popcountll(bi);
            if (comp) order[wave * P + below(bc)] = m;
            else if (in) order[wave * P + nall - 1 - below(be)] = m;
            if (lane == 0) {
                sched[wave] = __builtin_popcountll(bc);
                sched[MAX_XCD + wave] = nall;
                sched[2 * MAX_XCD + wave] = 0;
            }
        }
        return;
    }
    // Ranked by descending length, equal lengths by index: no two keys are equal, and those of lanes without a super tile are the least
    static_assert((uint64_t)SUPER_M * SUPER_N * 65535 * 64 < 1ull << 32, "a key's length");
    const uint32_t key = s_super[lane].len << 6 | (uint32_t)(63 - lane);
    int rank = 0;
    for (int j = 0; j < n_super; j += 8)
#pragma unroll
        for (int d = 0; d < 8; d++) rank += (uint32_t)__builtin_amdgcn_readlane((int)key, j + d) > key ? 1 : 0;
    const uint32_t ranked = (uint32_t)__builtin_amdgcn_ds_permute(rank * 4, (int)key);      // (lanes from n_super on: anything)
    const int len = lane < n_super ? (int)(ranked >> 6) : 0, sid = 63 - (int)(ranked & 63u);
    const uint32_t comp = lane < n_super ? s_super[sid].comp : 0u;
    const int n_ne = __builtin_popcountll(__ballot(len > 0));     // super tiles with work: the first ranks
    // Each to the XCD with the least length so far that has room: the least of (length, XCD) over eight lanes, of which every eight
    // hold the same.  The first ones go to the XCDs in turn.
    int dealt = lane;
    if (n_ne > n_xcd) {
        const int x = lane & 7;
        uint32_t load = x < n_xcd ? (uint32_t)__builtin_amdgcn_ds_bpermute(x * 4, len) << 3 | (uint32_t)x : ~0u;
        int room = rounds - 1;
        for (int r = n_xcd; r < n_ne; r++) {
            uint32_t least = load, o;
            o = (uint32_t)dpp<0xB1>((int)least); least = o < least ? o : least;
            o = (uint32_t)dpp<0x4E>((int)least); least = o < least ? o : least;
            o = (uint32_t)dpp<0x141>((int)least); least = o < least ? o : least;
            const uint32_t more = load + ((uint32_t)__builtin_amdgcn_readlane(len, r) << 3);
            const bool mine = load == least;
            room -= mine ? 1 : 0;
            load = mine ? (room > 0 ? more : ~0u) : load;
            dealt = lane == r ? (int)least : dealt;
        }
    }
    dealt &= 7;
    // The XCD's super tiles: those dealt to it, then of the ones without work, which fill the XCDs' remaining slots in order
    const int x = wave & (n_xcd - 1), part = wave >> xcd_shift, parts = ORDER_FEW_WAVES >> xcd_shift;
    const bool work = lane < n_ne;
    const int n_dealt = __builtin_popcountll(__ballot(work && dealt == x)), n_less = __builtin_popcountll(__ballot(work && dealt < x));
    const int fill = n_ne + x * rounds - n_less, fill_end = fill + rounds - n_dealt;
    const bool member = work ? dealt == x : lane < n_super && lane >= fill && lane < fill_end;
    const uint64_t members = __ballot(member);
    const int origin = sup.origin(sid), hm = nMacM - (origin >> 16), wn = nMacN - (origin & 0xffff);
    const int n_comp = member ? __builtin_popcount(comp) : 0;
    const int n_empty = member ? (hm < SUPER_M ? hm : SUPER_M) * (wn < SUPER_N ? wn : SUPER_N) - n_comp : 0;
    const uint32_t own = (uint32_t)n_comp | (uint32_t)n_empty << 16, incl = wave_scan(own);      // (at most 2048 of each)
    const uint32_t last = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
    const int nc = (int)(last & 0xffffu), nall = nc + (int)(last >> 16);
    if (member) s_seq[x * rounds + below(members)] = u32x4{(uint32_t)origin, comp, incl - own, 0u};    // (where waves share an XCD all write the same)
    if (lane == 0 && part == 0) {
        sched[x] = nc;
        sched[MAX_XCD + x] = nall;
        sched[2 * MAX_XCD + x] = 0;             // ticket counter of the persistent GEMM
    }
    __builtin_amdgcn_wave_barrier();
    // Half a wave per super tile, lane = macro tile: computing ones to the front of the sequence in order, the others to its back
    const int slot = lane & 31, n_members = __builtin_popcountll(members);
    const uint32_t before = (1u << slot) - 1u;
    for (int r = part * 2 + (lane >> 5); r < n_members; r += parts * 2) {
        const u32x4 e = s_seq[x * rounds + r];
        const int oi = (int)(e.x >> 16), oj = (int)(e.x & 0xffffu), mi = oi + slot / SUPER_N, mj = oj + slot % SUPER_N;
        const int width = nMacN - oj < SUPER_N ? nMacN - oj : SUPER_N;       // (slots before this one that exist, less the computing ones)
        const int c = __builtin_popcount(e.y & before);
        const int q = (e.y >> slot) & 1u ? (int)(e.z & 0xffffu) + c
                                         : nall - 1 - ((int)(e.z >> 16) + (slot / SUPER_N) * width + slot % SUPER_N - c);
        if (mi < nMacM && mj < nMacN) order[x * P + q] = mi * nMacN + mj;
    }
}

// Per-tile ascending list of kept k (the reference's offset[], cuSpAMM.cu:315-325)
// from the gate's bitmaps: one wave per output tile, popcount below the lane's
// bit gives every kept k its slot.
__global__ __launch_bounds__(256) void k_klist(const uint64_t *__restrict__ mask, uint16_t *__restrict__ klist,
                                               int64_t n_tiles, int nbK, int words) {
    const int lane = threadIdx.x & 63;
    const int64_t tid = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (tid >= n_tiles) return;
    int base = 0;
    for (int w = 0; w < words; w++) {
        const uint64_t m = mask[tid * words + w];
        if ((m >> lane) & 1ull)
            klist[tid * nbK + base + __builtin_popcountll(m & ((1ull << lane) - 1ull))] = (uint16_t)(w * 64 + lane);
        base += __builtin_popcountll(m);
    }
}

hipError_t launch_klist(const uint64_t *mask, uint16_t *klist, int64_t n_tiles, int64_t nbK, hipStream_t s) {
    k_klist<<<(unsigned)((n_tiles + 3) / 4), 256, 0, s>>>(mask, klist, n_tiles, (int)nbK, (int)((nbK + 63) / 64));
    return hipGetLastError();
}

// A macro tile's bitmaps take words * NTP * 8 bytes of LDS (tile 32: 512 bytes per 64 k tiles)
// beside 24 bytes of summaries per word; what does not fit a CU's LDS is walked in chunks of
// gate_chunk_words() words; `cap` > 0 (a context's developer knob) forces smaller chunks so that
// ordinary shapes take the chunked path.
static size_t gate_fixed_bytes(size_t words) { return words * 16 + 2 * (words + 1) * 4; }

int gate_chunk_words(int tile, int64_t nbK, int cap) {
    const int MT = macro_dim(tile);
    const size_t ntp = MT * MT < 8 ? 8 : MT * MT;
    const size_t words = (size_t)((nbK + 63) / 64);
    size_t cw = (gate_lds_limit() - gate_fixed_bytes(words)) / (ntp * 8);
    if (cap > 0 && cw > (size_t)cap) cw = (size_t)cap;
    return (int)(cw < words ? cw : words);
}

size_t gate_lds_bytes(int tile, int64_t nbK, int cap) {
    const int MT = macro_dim(tile);
    const size_t ntp = MT * MT < 8 ? 8 : MT * MT;
    const size_t words = (size_t)((nbK + 63) / 64);
    return ntp * (size_t)gate_chunk_words(tile, nbK, cap) * 8 + gate_fixed_bytes(words);
}

// k_gate may use all of a CU's LDS for the macro tile's bitmaps (its workgroups are short)
hipError_t gate_init() {
    hipError_t e;
    const void *gates[6] = {reinterpret_cast<const void *>(&k_gate<8>), reinterpret_cast<const void *>(&k_gate_chunks<8>),
                            reinterpret_cast<const void *>(&k_gate<4>), reinterpret_cast<const void *>(&k_gate_chunks<4>),
                            reinterpret_cast<const void *>(&k_gate<2>), reinterpret_cast<const void *>(&k_gate_chunks<2>)};
    for (const void *f : gates)
        if ((e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)gate_lds_limit())) != hipSuccess) return e;
    // k_order: its tables may take order_lds_limit() on top of a few static bytes
    return hipFuncSetAttribute(reinterpret_cast<const void *>(&k_order), hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int)order_lds_limit());
}

hipError_t launch_gate(const GateBuffers &g, int64_t nbM, int64_t nbK, int64_t nbN, int tile,
                       float tau, int n_xcd, int chunk_cap, hipStream_t s) {
    const int MT = macro_dim(tile);
    const int nMacM = (int)((nbM + MT - 1) / MT), nMacN = (int)((nbN + MT - 1) / MT);
    const int n_macro = nMacM * nMacN;
    const size_t lds = gate_lds_bytes(tile, nbK, chunk_cap);
    const int cw = gate_chunk_words(tile, nbK, chunk_cap);
    const bool one = cw >= (int)((nbK + 63) / 64);
#define SPAMM_GATE(MTV)                                                                                          \
    if (one) k_gate<MTV><<<dim3((unsigned)nMacN, (unsigned)nMacM), MTV == 2 ? 64 : 256, lds, s>>>(g, (int)nbM, (int)nbK, (int)nbN, tau);      \
    else k_gate_chunks<MTV><<<n_macro, MTV == 2 ? 64 : 256, lds, s>>>(g, (int)nbM, (int)nbK, (int)nbN, nMacN, tau, cw)
    switch (MT) {
        case 8: SPAMM_GATE(8); break;
        case 4: SPAMM_GATE(4); break;
        case 2: SPAMM_GATE(2); break;
        default: return hipErrorInvalidValue;
    }
#undef SPAMM_GATE
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const int nSupM = (nMacM + SUPER_M - 1) / SUPER_M, nSupN = (nMacN + SUPER_N - 1) / SUPER_N;
    const int n_super = nSupM * nSupN;
    const int rounds = (n_super + n_xcd - 1) / n_xcd;
    const SuperGrid sup = {nSupN, 0xffffffffu / (uint32_t)nSupN};
    if (n_super <= ORDER_FEW)
        k_order_few<<<1, ORDER_FEW_WAVES * 64, 0, s>>>(g.macro_work, g.macro_count, g.order, g.sched, g.kept, nMacM, nMacN, sup, n_super, rounds,
                                                       __builtin_ctz((unsigned)n_xcd));
    else
        k_order<<<1, 1024, order_lds_bytes(tile, nbM, nbN), s>>>(g, nMacM, nMacN, sup, n_super, rounds, n_xcd);
    return hipGetLastError();
}

}  // namespace spamm
