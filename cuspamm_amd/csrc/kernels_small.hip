// Stages 2 and 3 in one launch, for small and middling outputs.
//
// Where C has few macro tiles (up to some 1.5 per CU) the gate (k_gate), the schedule (k_order) and the
// gated GEMM are each a few microseconds of latency on a mostly idle chip, and the
// GEMM's 256-wide work units leave most CUs without any.  Here one workgroup owns a
// unit of U x U elements of C (U = 128 or 64) and does all three for it: it forms the
// tau mask of its output tiles from the norm maps, lists the k tiles they keep in
// LDS, and multiplies along that list.  What the gate leaves for the caller -- mask,
// counts, kept total -- is written on the way out; the macro tiles' work lists, which
// nothing reads after this kernel, are built by k_gate if somebody asks for them.
//
// Two forms: K / tile up to 64 (small_word_body, the list in a register) and beyond (small_unit_body, the list in LDS).
//
// A unit's life with its list in LDS, measured on fp16 2048^3 at tile 32, 5 % kept (which has its list in a register since), us: gate 2.0 (most
// of it the norms' round trip), list 0.3, first stages 0.8, 9 to 14 stages 3.4 to 6, C 1.5.
//
// Of the k loop's 0.285 us per stage on 256 CUs (2048^3 dense) the loads alone take 0.2 (a bare copy of the same panels into
// LDS, 21 TB/s over the chip), all else without them 0.18; without the MFMAs 0.27, without the LDS reads 0.285.  Two stages
// per sync, rings of 6 and 8 and square blocks of units per XCD changed it by 1 % or cost workgroups per CU.
//
// The order of the sum is k_gemm's: entries that every tile of the unit's MACRO tile
// keeps come first, then the others, each group in ascending k rotated to the
// macro tile's anchor.  So a unit looks at the norms of its whole macro tile, and C is
// the same bit for bit whichever kernel runs.
//
// What bounds it: a chain of latencies -- norms in, first stages in, one sync per 32 k,
// results out -- of which units of 128 (16 KiB a stage, two workgroups per CU, or three) make
// the k loop shortest and units of 64 spread a small C over more CUs.  Gate, schedule
// and GEMM as launches of their own -> this kernel, whole multiplies, when it took their place: 256^3 24.6 -> 14.7 us, 1056 x 1568 x
// 1312 38.2 -> 22.8, fp16 2048^3 at tile 32, 5 % kept, 38.5 -> 26.3, 2048^3 dense 63 -> 38, 1024 rows against a resident 8192^2
// 50.3 -> 36.5.  With both norm-map passes in one launch, the copies in the memory-side cache and the list in a register they take
// 8.1, 12.4, 14.4, 33 and 30.5.
#include "gemm_device.h"

namespace spamm {

template <int B, int U, int RING>
struct SmallCfg {
    static constexpr int MT = 256 / B;                       // tiles per macro tile per dimension
    static constexpr int PD = 256 / U;                       // units per macro tile per dimension
    static constexpr int TU = U / B > 0 ? U / B : 1;         // tiles (slots) per unit per dimension
    static constexpr int TT = TU * TU;
    static constexpr int RS = B < U ? B : U;                 // rows of a slot
    static constexpr int NSPE = B / 32;                      // stages of 32 k per list entry
    static constexpr int TILE_BYTES = B * B * 2;
    static constexpr int OP_BYTES = U * 64;                  // one operand's part of a stage
    static constexpr int STAGE_BYTES = 2 * OP_BYTES;         // 16 or 8 KiB
    static constexpr int NBUF = RING;
    static constexpr int CPS = RS / 16;                      // 1 KiB chunks per slot
    static constexpr int CHW = U / 64;                       // chunks per wave per operand per stage (in one slot)
    static constexpr int LPW = 2 * CHW;
    static constexpr int NB = U / 32;                        // 16-wide MFMA blocks per wave per dimension
    static constexpr int NP = TU > 1 ? TU / 2 : 1;           // tiles per wave per dimension
    static constexpr int RB = NB / NP;                       // MFMA blocks per tile and wave per dimension
    static constexpr uint32_t ROW_BITS = (1u << TU) - 1u;
    static constexpr uint32_t COL_BITS = TU == 4 ? 0x1111u : (TU == 2 ? 0x5u : 0x1u);
    static_assert(CHW == 1 || CPS >= 2, "a wave's two chunks lie in one slot, one after the other");
};

// LDS behind the ring: list entries, {full, partial} words, tile bits per k
size_t small_lds_bytes_(int stage_bytes, int nbuf, int64_t nbK) {
    const size_t words = (size_t)((nbK + 63) / 64);
    return (size_t)stage_bytes * nbuf + words * 64 * 4 + words * 16 + words * 64 * 2;
}

// Offsets are 32-bit: C has SMALL_MAX_UNITS units of 128 x 128 at most and K / B is at most SMALL_MAX_NBK, so that C, the norm
// maps and the masks stay below 2^31 bytes (the packed operands need not).
struct SmallGrid {
    int nMacN;
    uint32_t mac_rec;        // floor((2^32 - 1) / nMacN): the macro row of macro tile m is the upper half of (m + 1) * mac_rec
    int n_units, chunk;      // units, and per XCD
    int xcd_shift, mode;     // log2 of the XCDs
};

// What a unit needs of GateBuffers, within the second line of arguments
struct UnitGate {
    const float *nA, *nBt;
    KeptProducts *kept;
    int32_t *counts;
    uint64_t *mask;
};

// Two (or one) dma_loads of neighbouring chunks
template <int N>
__device__ __forceinline__ void dma_chunks(const unsigned char *sbase, uint32_t voff, uint32_t lds_addr) {
    if constexpr (N == 2)
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\n\tglobal_load_lds_dwordx4 %1, %2 offset:1024"
                     :
                     : "s"(lds_addr), "v"(voff), "s"(sbase)
                     : "memory", "m0");
    else
        dma_load<0>(sbase, voff, lds_addr);
}

// (Norms by buffers' scalar offsets, smallest and largest norm as integers, the first entries by one read of LDS, loads of full stages without a
// look at the entry's bits, masks and counts formed at the end: 1024 rows against a resident 8192^2 23.6 -> 22.4 us alone, its gate 3.3 -> 2.8,
// 5024 x 4128 x 3168 at tile 32, 10 % kept 41.3 -> 39.8, its gate 7.2 -> 6.0.)
template <int B, int U, int RING>
__device__ __forceinline__ void small_unit_body(const unsigned char *pA, const unsigned char *pB, int nbM, int nbK, int nbN, SmallGrid sg,
                                                float tau, float *C, UnitGate g) {
    using H = SmallCfg<B, U, RING>;
    constexpr int NBUF = H::NBUF, MT = H::MT, TU = H::TU, TT = H::TT, NB = H::NB, BLK = MT / TU;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    // all arguments at once: a line of them asked for later is another 0.3 us
    asm volatile("" : "+s"(pA), "+s"(pB), "+s"(nbM), "+s"(nbK), "+s"(nbN), "+s"(tau), "+s"(C), "+s"(g.nA), "+s"(g.nBt), "+s"(g.kept),
                 "+s"(g.counts), "+s"(g.mask));
    const int words = (nbK + 63) >> 6, mode = sg.mode;
    uint32_t *s_list = reinterpret_cast<uint32_t *>(smem + NBUF * H::STAGE_BYTES);   // k | tile bits << 16
    uint64_t *s_fp = reinterpret_cast<uint64_t *>(s_list + words * 64);              // [words][2]
    uint16_t *s_bits = reinterpret_cast<uint16_t *>(s_fp + 2 * words);               // [words * 64]

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wr = wave >> 1, wc = wave & 1;
    // consecutive units (neighbours share operand panels) in equal chunks, one per XCD
    const uint32_t unit = (blockIdx.x & ((1u << sg.xcd_shift) - 1u)) * (uint32_t)sg.chunk + (blockIdx.x >> sg.xcd_shift);
    if (unit >= (uint32_t)sg.n_units) return;
    const uint32_t macro = unit / (H::PD * H::PD), part = unit % (H::PD * H::PD), ui = part / H::PD, uj = part % H::PD;
    const int mi = (int)__umulhi(macro + 1u, sg.mac_rec), mj = (int)macro - mi * sg.nMacN;
    const int M = nbM * B, N = nbN * B;
    const int urow = mi * 256 + (int)ui * U, ucol = mj * 256 + (int)uj * U;
    if (urow >= M || ucol >= N) return;
    const int ti0 = urow / B, tj0 = ucol / B;                          // first tile of the unit

    // ---- gate: a wave takes 64 k at a time, lane = k, and holds the norms of the macro tile's rows and columns, the unit's own first (rows
    // clamped; a lane beyond the last k reads what follows, or nothing behind the map's end), the next 64's on their way
    const bool multiply = (mode & SMALL_MULTIPLY) != 0;        // (the gate alone needs no list, and the unit's norms only)
    const bool interior = (mi + 1) * MT <= nbM && (mj + 1) * MT <= nbN;
    const int rows_in = nbM - ti0, cols_in = nbN - tj0;                // of the unit's tile rows and columns, those below exist
    const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((void *)g.nA, 0, nbM * nbK * 4, 0x00020000);
    const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc((void *)g.nBt, 0, nbN * nbK * 4, 0x00020000);
    uint32_t a[MT] = {}, b[MT] = {};
    auto load_norms = [&](int w) {
        const int voff = (w * 64 + lane) * 4, stride = nbK * 4;
        auto load = [&](int blk) {
            const int i0 = mi * MT + ((ti0 + blk * TU) & (MT - 1)), j0 = mj * MT + ((tj0 + blk * TU) & (MT - 1));
#pragma unroll
            for (int x = 0; x < TU; x++) {
                const int i = i0 + x < nbM ? i0 + x : nbM - 1, j = j0 + x < nbN ? j0 + x : nbN - 1;
                a[blk * TU + x] = __builtin_amdgcn_raw_buffer_load_b32(ra, voff, i * stride, 0);
                b[blk * TU + x] = __builtin_amdgcn_raw_buffer_load_b32(rb, voff, j * stride, 0);
            }
        };
        load(0);
        if (multiply) {
#pragma unroll
            for (int blk = 1; blk < BLK; blk++) load(blk);
        }
    };
    if (wave < words) load_norms(wave);
    const int anchor = multiply ? list_anchor(mi, mj, MT, nbM, nbK, nbN) : 0;
    for (int w = wave; w < words; w += 4) {
        const int k = w * 64 + lane;
        const bool live = k < nbK;
        float au[TU], bu[TU];
#pragma unroll
        for (int x = 0; x < TU; x++) {                                 // (what does not exist is kept at no threshold: NaN)
            au[x] = live && x < rows_in ? __uint_as_float(a[x]) : __builtin_nanf("");
            bu[x] = x < cols_in ? __uint_as_float(b[x]) : __builtin_nanf("");
        }
        uint32_t ub = 0;                                               // the unit's tiles that keep this lane's k
#pragma unroll
        for (int t = TT - 1; t >= 0; t--) ub = ub + ub + (au[t / TU] * bu[t % TU] >= tau ? 1u : 0u);
        // kept by every tile of the macro tile: rounding is monotone, so the product of the smallest norms decides -- unless one
        // is not finite (inf * 0 and NaN are never kept), or below zero: then all products are looked at
        uint32_t amin = a[0], bmin = b[0], big = a[0] > b[0] ? a[0] : b[0];
#pragma unroll
        for (int x = 1; x < MT; x++) {
            amin = a[x] < amin ? a[x] : amin;
            bmin = b[x] < bmin ? b[x] : bmin;
            const uint32_t m = a[x] > b[x] ? a[x] : b[x];
            big = m > big ? m : big;
        }
        bool full = __uint_as_float(amin) * __uint_as_float(bmin) >= tau;
        if (__ballot(big >= 0x7f800000u) != 0ull) {
            full = true;
#pragma unroll
            for (int x = 0; x < MT; x++)
#pragma unroll
                for (int y = 0; y < MT; y++) full = full && __uint_as_float(a[x]) * __uint_as_float(b[y]) >= tau;
        }
        full = full && live && interior;
        const uint64_t F = __ballot(full), P = __ballot(ub != 0u && !full);
        if (w + 4 < words) load_norms(w + 4);
        if (lane == 0) {
            s_fp[2 * w] = F;
            s_fp[2 * w + 1] = P;
        }
        s_bits[k] = (uint16_t)ub;
    }
    __syncthreads();
    // What the gate leaves behind, out of s_bits: wave x has row x of the unit's tiles (a tile shared by several units is written by the
    // first).  A unit's kept products are a word of its own: added to one total by atomics they queued up at the kernel's end, where 200
    // to 1000 units finish together (1024^3 10 % 15.4 -> 13.7 us whole, 2048^3 dense 33.8 -> 31.5, 1056 x 1568 x 1312 18.6 -> 17.7).  The total is
    // minus their number then: what the last gate was is known on the device, also behind a replayed graph.
    auto store_gate = [&]() {
        if (!(mode & SMALL_GATE)) return;
        const bool owner = (ui * U) % B == 0 && (uj * U) % B == 0;
        if (wave < TU && wave < rows_in && owner) {
            const bool mine = lane < TU && lane < cols_in;
            const uint32_t tile = (uint32_t)((ti0 + wave) * nbN + tj0 + lane);
            int count = 0;
            for (int w = 0; w < words; w++) {
                const uint32_t ub = (uint32_t)s_bits[w * 64 + lane] >> (wave * TU);
                uint64_t word = 0;
#pragma unroll
                for (int y = 0; y < TU; y++) {
                    const uint64_t m = __ballot((ub >> y) & 1u);
                    word = lane == y ? m : word;
                }
                if (mine) g.mask[tile * (uint32_t)words + w] = word;
                count += __builtin_popcountll(word);
            }
            if (mine) g.counts[tile] = count;
        }
        if (wave == 3) {
            const int units_n = (N + U - 1) / U;
            int total = 0;
            if (owner)
                for (int w = 0; w < words; w++) total += __builtin_popcount((uint32_t)s_bits[w * 64 + lane]);
#pragma unroll
            for (int off = 1; off < 64; off <<= 1) total += __shfl_xor(total, off, 64);
            if (lane == 0) {
                g.kept->units[urow / U * units_n + ucol / U] = (uint32_t)total;
                if (unit == 0) g.kept->total = -((M + U - 1) / U * units_n);
            }
        }
    };

    int S = 0, Sfull = 0;
    if (multiply) {
        // ---- list: every wave scans the words' counts (at most 64 words), then places its own words' entries
        const uint64_t below_a = (1ull << (anchor & 63)) - 1ull;
        int n_full, n_part;
        auto place = [&](int w, uint64_t F, uint64_t P, int base_f, int base_p, int rot_f, int rot_p) {
            const uint64_t below = (1ull << lane) - 1ull;
            int pos = -1;
            if ((F >> lane) & 1ull) {
                pos = base_f + __builtin_popcountll(F & below) - rot_f;
                if (pos < 0) pos += n_full;
            } else if ((P >> lane) & 1ull) {
                pos = base_p + __builtin_popcountll(P & below) - rot_p;
                if (pos < 0) pos += n_part;
                pos += n_full;
            }
            if (pos >= 0) s_list[pos] = (uint32_t)(w * 64 + lane) | (uint32_t)s_bits[w * 64 + lane] << 16;
        };
        {
            const uint64_t Fl = lane < words ? s_fp[2 * lane] : 0ull, Pl = lane < words ? s_fp[2 * lane + 1] : 0ull;
            int bf = __builtin_popcountll(Fl), bp = __builtin_popcountll(Pl);
            const int own_f = bf, own_p = bp;
            for (int off = 1; off < words; off <<= 1) {
                const int tf = __shfl_up(bf, off, 64), tp = __shfl_up(bp, off, 64);
                if (lane >= off) { bf += tf; bp += tp; }
            }
            n_full = __builtin_amdgcn_readlane(bf, words - 1);
            n_part = __builtin_amdgcn_readlane(bp, words - 1);
            bf -= own_f;
            bp -= own_p;
            const int rot_f = __builtin_amdgcn_readlane(bf + __builtin_popcountll(Fl & below_a), anchor >> 6);
            const int rot_p = __builtin_amdgcn_readlane(bp + __builtin_popcountll(Pl & below_a), anchor >> 6);
            for (int w = wave; w < words; w += 4)
                place(w, s_fp[2 * w], s_fp[2 * w + 1], __builtin_amdgcn_readlane(bf, w), __builtin_amdgcn_readlane(bp, w), rot_f, rot_p);
        }
        __syncthreads();
        S = (n_full + n_part) * H::NSPE;
        Sfull = n_full * H::NSPE;
    }

    if (multiply && S == 0) {
        constexpr int LPR = U / 4;                                     // lanes per row
        const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
        const int c0 = ucol + (lane % LPR) * 4;
        if (c0 < N)
            for (int r = wave * (64 / LPR) + lane / LPR; r < U && urow + r < M; r += 4 * (64 / LPR))
                __builtin_nontemporal_store(zero, reinterpret_cast<f32x4 *>(C + (uint32_t)((urow + r) * N + c0)));
    }
    f32x4 acc[NB][NB];
#pragma unroll
    for (int r = 0; r < NB; r++)
#pragma unroll
        for (int c = 0; c < NB; c++) acc[r][c] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    if (S > 0) {
        // ---- staging: a wave copies CHW consecutive 1 KiB chunks of the A part and of the B part of a stage
        // (the ring protocol and its hand-counted waits are k_gemm's)
        const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)smem;
        const int chunk0 = wave * H::CHW, slot = chunk0 / H::CPS, vec = (chunk0 % H::CPS) * 64;
        int ti = ti0 + slot, tj = tj0 + slot;
        ti = ti < nbM ? ti : nbM - 1;
        tj = tj < nbN ? tj : nbN - 1;
        const int within = (vec / H::RS) * B + vec % H::RS;            // 16-byte vector inside the tile's 4 k-groups
        const unsigned char *rowA = pA + (int64_t)ti * nbK * H::TILE_BYTES + (within + (int)(ui * U) % B) * 16;
        const unsigned char *rowB = pB + (int64_t)tj * nbK * H::TILE_BYTES + (within + (int)(uj * U) % B) * 16;
        const uint32_t ldsA = lds_base + chunk0 * 1024, ldsB = ldsA + H::OP_BYTES;
        const uint32_t needA = (H::ROW_BITS << (slot * TU)) << 16, needB = (H::COL_BITS << slot) << 16;   // entry bits that read this slot
        const uint32_t voff = lane * 16;

        // entry of a stage (stages beyond the last repeat the last entry: loaded, never multiplied)
        auto entry_at = [&](int t) -> uint32_t { return s_list[(t < S ? t : S - 1) / H::NSPE]; };
        auto offset = [&](int t, uint32_t ent) -> uint32_t {           // (a row of tiles is at most SMALL_MAX_NBK tiles: 64 MiB)
            return (ent & 0xffffu) * H::TILE_BYTES + (uint32_t)(((t < S ? t : S - 1) % H::NSPE) * (B * 64));
        };
        // a slot that no tile pair of the entry reads is not fetched: its load goes to one place that is cache resident, so that the
        // number of loads in flight stays fixed
        auto issue_a = [&](const unsigned char *from, uint32_t boff) { dma_chunks<H::CHW>(from, voff, ldsA + boff); };
        auto issue_b = [&](const unsigned char *from, uint32_t boff) { dma_chunks<H::CHW>(from, voff, ldsB + boff); };
        auto sync_next = [&]() {
            __builtin_amdgcn_s_waitcnt(waitcnt_imm(H::LPW * (NBUF - 2), 0));
            __syncthreads();
        };
        auto frag_off = [&](int wsel, int blk) -> int {
            const int s = TU > 1 ? wsel + 2 * (blk * 16 / H::RS) : 0;
            const int ro = TU > 1 ? (blk * 16) % H::RS : wsel * (U / 2) + blk * 16;
            return s * H::RS * 64 + ((lane >> 4) * H::RS + ro + (lane & 15)) * 16;
        };
        struct Frags {
            half8 a[NB], b[NB];
        };
        auto load_frag = [&](Frags &f, uint32_t boff, auto idx) {
            constexpr int i = decltype(idx)::value;
            const unsigned char *bufA = smem + boff;
            if constexpr (i == 0) f.a[0] = *reinterpret_cast<const half8 *>(bufA + frag_off(wr, 0));
            else if constexpr (i <= NB) f.b[i - 1] = *reinterpret_cast<const half8 *>(bufA + H::OP_BYTES + frag_off(wc, i - 1));
            else f.a[i - NB] = *reinterpret_cast<const half8 *>(bufA + frag_off(wr, i - NB));
        };
        // ---- prologue: the first entries by one read (each in turn, their latencies were half of it)
        const uint32_t firsts = entry_at(lane);
#pragma unroll
        for (int t = 0; t < NBUF; t++) {
            const uint32_t e = (uint32_t)__builtin_amdgcn_readlane((int)firsts, t), koff = offset(t, e);
            issue_a((e & needA) ? rowA + koff : pA, t * H::STAGE_BYTES);
            issue_b((e & needB) ? rowB + koff : pB, t * H::STAGE_BYTES);
        }
        // The buffer of stage t -- once that is in registers, of stage t + NBUF -- and the next one's, which is formed before the
        // sync: behind it a wave's first reads of LDS wait for their address.  (By t % NBUF where they are used the compiler
        // put up to 13 scalar instructions there, which depended on the order of the kernel's arguments: 384 x 4736 x 416 at
        // tile 32 33.4 or 34.3 us, 32.75 then; 1056 x 1568 x 1312 17.34 or 17.5, 17.07 then.)
        int t = 0;
        uint32_t buf = 0;
        auto next_buf = [&]() {
            uint32_t next = buf + H::STAGE_BYTES == NBUF * H::STAGE_BYTES ? 0u : buf + H::STAGE_BYTES;
            asm volatile("" : "+s"(next));
            return next;
        };
        uint32_t e_cur = entry_at(0), e_new = entry_at(NBUF);
        __builtin_amdgcn_s_waitcnt(waitcnt_imm(H::LPW * (NBUF - 1), 0));
        __syncthreads();
        Frags f0, f1;
        static_for<2 * NB>([&](auto i) { load_frag(f0, 0, i); });
#define SPAMM_FENCE() __builtin_amdgcn_sched_barrier(0)
        // (every slot of the stages that are fetched here is, whether its entry reads it or not: all but the last few are full ones)
        auto full_stage = [&](const Frags &cur, Frags &nxt) {
            const uint32_t next = next_buf();
            sync_next();
            const uint32_t en = __builtin_amdgcn_readfirstlane(e_new);
            e_new = entry_at(t + 1 + NBUF);
            SPAMM_FENCE();
            uint32_t koff = 0;
            static_for<NB * NB>([&](auto idx) {
                constexpr int i = decltype(idx)::value, r = i / NB, c = i % NB, A_AT = NB == 4 ? 8 : 2, B_AT = NB == 4 ? 12 : 3;
                acc[r][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(cur.a[r], cur.b[c], acc[r][c], 0, 0, 0);
                if constexpr (i < 2 * NB) load_frag(nxt, next, idx);
                if constexpr (i == A_AT - 1) koff = offset(t + NBUF, en);
                if constexpr (i == A_AT) issue_a(rowA + koff, buf);
                if constexpr (i == B_AT) issue_b(rowB + koff, buf);
                SPAMM_FENCE();
            });
            t++;
            buf = next;
        };
        while (__builtin_expect(t + 1 < Sfull, 1)) {
            full_stage(f0, f1);
            full_stage(f1, f0);
        }
        e_cur = entry_at(t);
        auto partial_stage = [&](const Frags &cur, Frags &nxt) {
            const uint32_t next = next_buf();
            sync_next();
            const uint32_t en = t + NBUF < S ? __builtin_amdgcn_readfirstlane(e_new) : (__builtin_amdgcn_readfirstlane(e_new) & 0xffffu);
            const uint32_t ec = t < S ? (__builtin_amdgcn_readfirstlane(e_cur) >> 16) >> (TU > 1 ? wr * TU + wc : 0) : 0u;
            e_cur = entry_at(t + 1);
            e_new = entry_at(t + 1 + NBUF);
            const uint32_t koff = offset(t + NBUF, en);
            SPAMM_FENCE();
            static_for<H::NP * H::NP>([&](auto pair) {
                constexpr int p = decltype(pair)::value, px = p / H::NP, py = p % H::NP, bit = 2 * px * TU + 2 * py;
                if ((ec >> bit) & 1u) {
#pragma unroll
                    for (int r = 0; r < H::RB; r++)
#pragma unroll
                        for (int c = 0; c < H::RB; c++)
                            acc[px * H::RB + r][py * H::RB + c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                                cur.a[px * H::RB + r], cur.b[py * H::RB + c], acc[px * H::RB + r][py * H::RB + c], 0, 0, 0);
                }
                if constexpr (p == 0) {
                    SPAMM_FENCE();
                    static_for<2 * NB>([&](auto i) { load_frag(nxt, next, i); });
                    issue_a((en & needA) ? rowA + koff : pA, buf);
                    issue_b((en & needB) ? rowB + koff : pB, buf);
                    SPAMM_FENCE();
                }
            });
            SPAMM_FENCE();
            t++;
            buf = next;
        };
        while (t < S) {
            partial_stage(f0, f1);
            if (t >= S) break;
            partial_stage(f1, f0);
        }
#undef SPAMM_FENCE
        __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, 0));                 // the ring still holds clamped loads
    }

    // ---- epilogue: as k_gemm's
    if (S > 0) {
        const uint32_t lane_off = (uint32_t)(32 * (lane >> 5)) * (uint32_t)N + 4 * (lane & 31);     // bytes
#pragma unroll
        for (int r = 0; r < NB; r++) {
            const int row0 = urow + (TU > 1 ? (wr + 2 * (r * 16 / B)) * B + (r * 16) % B : wr * (U / 2) + r * 16);
            if (row0 >= M) continue;
#pragma unroll
            for (int c = 0; c < NB; c += 2) {
                const int col0 = ucol + (TU > 1 ? (wc + 2 * (c * 16 / B)) * B + (c * 16) % B : wc * (U / 2) + c * 16);
                if (col0 >= N) continue;
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const float x = acc[r][c][i], y = acc[r][c + 1][i];
                    const auto sw = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(y), false, false);
                    float *out = C + (uint32_t)((row0 + i) * N + col0);
                    asm volatile("global_store_dword %0, %1, %2 nt" :: "v"(lane_off), "v"(sw[0]), "s"(out) : "memory");
                    asm volatile("global_store_dword %0, %1, %2 nt" :: "v"(lane_off), "v"(sw[1]), "s"(out + 4 * N) : "memory");
                }
            }
        }
    }
    store_gate();
}

// The arguments come in the order of their use, and all that are read lie in the first 128 bytes: a line of them that nothing
// has asked for yet is 0.2 to 0.4 us away when it is needed (256^3 10.44 -> 10.27 us, fp16 2048^3 at tile 32, 5 % kept 25.15 ->
// 24.74 against M, N and C in a third line).
template <int B, int U>
__global__ __launch_bounds__(256, 2) void k_small(const unsigned char *pA, const unsigned char *pB, int nbM, int nbK, int nbN, SmallGrid sg,
                                                  float tau, float *C, UnitGate g) {
    small_unit_body<B, U, (U == 128 ? 4 : 6)>(pA, pB, nbM, nbK, nbN, sg, tau, C, g);
}

// Units of 128 by three workgroups per CU (small_three).
template <int B>
__global__ __launch_bounds__(256, 3) void k_small_three(const unsigned char *pA, const unsigned char *pB, int nbM, int nbK, int nbN,
                                                        SmallGrid sg, float tau, float *C, UnitGate g) {
    small_unit_body<B, 128, 3>(pA, pB, nbM, nbK, nbN, sg, tau, C, g);
}

// ---------------------------------------------------------------- one word of k tiles (K / tile <= 64), the usual small problem
// The same unit, with the list in a register.  A wave of such a kernel is alone on its SIMD and issues one instruction in some
// five clocks, so the time to its first stage is a number of instructions: 7900 clocks in the kernel above (fp16 2048^3, 5 % kept: gate 1500
// behind the norms' arrival, list 900, the ring's first loads 1600, which wait for each entry in turn), 4600 here.  Every wave forms the whole
// list for itself -- lane = k, a lane's place by counting bits, one permutation of the lanes -- without LDS, without a sync, and takes a
// stage's entry out of it by v_readlane.  Norms, operands and C are addressed by a buffer's scalar offset, one scalar instruction a load, and
// all arguments are asked for at once.  A slot that no tile pair of an entry reads, and stages beyond the last, are loads from a
// buffer of no bytes: they keep the number of loads in flight fixed and fetch nothing (their offset is one of the operand's all the same).
// Kernels alone, the list in LDS -> this: 256^3 5.35 -> 3.45 us (its gate alone 3.2 -> 1.9), 1056 x 1568 x 1312 9.0 -> 6.4, 1024^3 at tile 64 6.1 ->
// 4.5, fp16 2048^3 at tile 32 5 % kept 11.6 -> 9.4, 75 % 26.5 -> 23, 4096^3 at tile 64 10 % 33.7 -> 31.
// What bounds it now: launch and arguments 700 clocks, norms 1200, gate and list 1000, the ring's first loads at 64 bytes a clock 1100, a stage
// of 128 x 128 x 32 some 600 (of which its loads alone take 440), C at 64 bytes a clock.
typedef int i32x4s __attribute__((ext_vector_type(4)));

// Raw buffer of `bytes` from p on (gfx950: 32-bit data, no swizzle, no stride)
__device__ __forceinline__ i32x4s raw_buffer(const void *p, int bytes) {
    const uint64_t a = (uint64_t)(uintptr_t)p;
    return i32x4s{(int)(uint32_t)a, (int)(uint32_t)(a >> 32), bytes, 0x00020000};
}

// As dma_load, from a buffer: lane l's 16 bytes from soff + voff(l) + IMM land at lds_addr + IMM + 16 * l.
template <int N>
__device__ __forceinline__ void dma_buffer(const i32x4s &rsrc, uint32_t voff, uint32_t soff, uint32_t lds_addr) {
    if constexpr (N == 2)
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds\n\tbuffer_load_dwordx4 %1, %2, %3 offen offset:1024 lds"
                     :
                     : "s"(lds_addr), "v"(voff), "s"(rsrc), "s"(soff)
                     : "memory", "m0");
    else
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                     :
                     : "s"(lds_addr), "v"(voff), "s"(rsrc), "s"(soff)
                     : "memory", "m0");
}

template <int B, int U, int RING>
__device__ __forceinline__ void small_word_body(const unsigned char *pA, const unsigned char *pB, int nbM, int nbK, int nbN, SmallGrid sg,
                                                float tau, float *C, UnitGate g) {
    using H = SmallCfg<B, U, RING>;
    constexpr int NBUF = H::NBUF, MT = H::MT, TU = H::TU, TT = H::TT, NB = H::NB, BLK = MT / TU;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    // all arguments at once: a line of them asked for later is another 0.3 us
    asm volatile("" : "+s"(pA), "+s"(pB), "+s"(nbM), "+s"(nbK), "+s"(nbN), "+s"(tau), "+s"(C), "+s"(g.nA), "+s"(g.nBt), "+s"(g.kept),
                 "+s"(g.counts), "+s"(g.mask));
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wr = wave >> 1, wc = wave & 1, mode = sg.mode;
    const uint32_t unit = (blockIdx.x & ((1u << sg.xcd_shift) - 1u)) * (uint32_t)sg.chunk + (blockIdx.x >> sg.xcd_shift);
    if (unit >= (uint32_t)sg.n_units) return;
    const uint32_t macro = unit / (H::PD * H::PD), part = unit % (H::PD * H::PD), ui = part / H::PD, uj = part % H::PD;
    const int mi = (int)__umulhi(macro + 1u, sg.mac_rec), mj = (int)macro - mi * sg.nMacN;
    const int M = nbM * B, N = nbN * B;
    const int urow = mi * 256 + (int)ui * U, ucol = mj * 256 + (int)uj * U;
    if (urow >= M || ucol >= N) return;
    const int ti0 = urow / B, tj0 = ucol / B;                          // first tile of the unit

    // ---- gate: lane = k, norms of the macro tile's rows and columns, the unit's own first (rows clamped; a lane beyond the last k
    // reads what follows, or nothing behind the map's end)
    const bool multiply = (mode & SMALL_MULTIPLY) != 0;
    const int rows_in = nbM - ti0, cols_in = nbN - tj0;                // of the unit's tile rows and columns, those below exist
    uint32_t a[MT], b[MT];
    {
        const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((void *)g.nA, 0, nbM * nbK * 4, 0x00020000);
        const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc((void *)g.nBt, 0, nbN * nbK * 4, 0x00020000);
        const int stride = nbK * 4;
        auto load = [&](int blk) {
            const int i0 = mi * MT + ((ti0 + blk * TU) & (MT - 1)), j0 = mj * MT + ((tj0 + blk * TU) & (MT - 1));
#pragma unroll
            for (int x = 0; x < TU; x++) {
                const int i = i0 + x < nbM ? i0 + x : nbM - 1, j = j0 + x < nbN ? j0 + x : nbN - 1;
                a[blk * TU + x] = __builtin_amdgcn_raw_buffer_load_b32(ra, lane * 4, i * stride, 0);
                b[blk * TU + x] = __builtin_amdgcn_raw_buffer_load_b32(rb, lane * 4, j * stride, 0);
            }
        };
        load(0);
        if (multiply) {
#pragma unroll
            for (int blk = 1; blk < BLK; blk++) load(blk);
        }
    }
    const int anchor = multiply ? list_anchor(mi, mj, MT, nbM, nbK, nbN) : 0;
    const uint64_t live = nbK >= 64 ? ~0ull : (1ull << nbK) - 1ull;
    const bool mine = (live >> lane) & 1ull;
    float au[TU], bu[TU];
#pragma unroll
    for (int x = 0; x < TU; x++) {                                     // (what does not exist is kept at no threshold: NaN)
        au[x] = mine && x < rows_in ? __uint_as_float(a[x]) : __builtin_nanf("");
        bu[x] = x < cols_in ? __uint_as_float(b[x]) : __builtin_nanf("");
    }
    uint32_t ub = 0;                                                   // the unit's tiles that keep this lane's k
#pragma unroll
    for (int t = TT - 1; t >= 0; t--) ub = ub + ub + (au[t / TU] * bu[t % TU] >= tau ? 1u : 0u);

    // What the gate leaves behind: wave x has row x of the unit's tiles (a tile shared by several units is written by the first)
    auto store_gate = [&]() {
        if (!(mode & SMALL_GATE)) return;
        const int units_n = (N + U - 1) / U;
        if (wave < TU) {
            uint64_t word = 0;
#pragma unroll
            for (int y = 0; y < TU; y++) {
                const uint64_t m = __ballot((ub >> (wave * TU + y)) & 1u);
                word = lane == y ? m : word;
            }
            if ((ui * U) % B == 0 && (uj * U) % B == 0 && lane < TU && wave < rows_in && lane < cols_in) {
                const uint32_t tile = (uint32_t)((ti0 + wave) * nbN + tj0 + lane);
                g.mask[tile] = word;
                g.counts[tile] = __builtin_popcountll(word);
            }
        }
        // the unit's kept products, a word of its own; their total is minus the number of units (see k_small)
        if (wave == 3) {
            int total = 0;
#pragma unroll
            for (int t = 0; t < TT; t++) total += __builtin_popcountll(__ballot((ub >> t) & 1u));
            if (lane == 0) {
                g.kept->units[urow / U * units_n + ucol / U] = (uint32_t)(((ui * U) % B == 0 && (uj * U) % B == 0) ? total : 0);
                if (unit == 0) g.kept->total = -((M + U - 1) / U * units_n);
            }
        }
    };
    if (!multiply) {
        store_gate();
        return;
    }

    // ---- list: kept by every tile of the macro tile (rounding is monotone, so the product of the smallest norms decides, unless one is
    // not finite, or below zero), then the others, each group rotated to the anchor
    uint32_t amin = a[0], bmin = b[0], big = a[0] > b[0] ? a[0] : b[0];
#pragma unroll
    for (int x = 1; x < MT; x++) {
        amin = a[x] < amin ? a[x] : amin;
        bmin = b[x] < bmin ? b[x] : bmin;
        const uint32_t m = a[x] > b[x] ? a[x] : b[x];
        big = m > big ? m : big;
    }
    bool full = __uint_as_float(amin) * __uint_as_float(bmin) >= tau;
    if (__ballot(big >= 0x7f800000u) != 0ull) {
        full = true;
#pragma unroll 1
        for (int x = 0; x < MT; x++) {
#pragma unroll
            for (int y = 0; y < MT; y++) {
                float ax = __uint_as_float(a[0]);
#pragma unroll
                for (int z = 1; z < MT; z++) ax = x == z ? __uint_as_float(a[z]) : ax;
                full = full && ax * __uint_as_float(b[y]) >= tau;
            }
        }
    }
    const bool interior = (mi + 1) * MT <= nbM && (mj + 1) * MT <= nbN;
    const uint64_t F = interior ? __ballot(full) & live : 0ull, P = __ballot(ub != 0u) & ~F;
    const int n_full = __builtin_popcountll(F), n = n_full + __builtin_popcountll(P), S = n * H::NSPE, Sfull = n_full * H::NSPE;
    f32x4 acc[NB][NB];
#pragma unroll
    for (int r = 0; r < NB; r++)
#pragma unroll
        for (int c = 0; c < NB; c++) acc[r][c] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    const __amdgpu_buffer_rsrc_t rc = __builtin_amdgcn_make_buffer_rsrc((void *)C, 0, M * N * 4, 0x00020000);
    constexpr int NT = 2;                                              // cache policy of the stores of C: non-temporal
    if (S == 0) {
        constexpr int LPR = U / 4;                                     // lanes per row
        const i32x4s zero = {0, 0, 0, 0};
        const int c0 = ucol + (lane % LPR) * 4;
        if (c0 < N)
            for (int r = wave * (64 / LPR) + lane / LPR; r < U && urow + r < M; r += 4 * (64 / LPR))
                __builtin_amdgcn_raw_buffer_store_b128(zero, rc, ((urow + r) * N + c0) * 4, 0, NT);
    } else {
        // every lane goes to its place: full entries, partial ones, and what is not kept behind them
        auto below = [](uint64_t m) { return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u)); };
        const uint64_t below_a = (1ull << anchor) - 1ull;
        int pf = below(F) - __builtin_popcountll(F & below_a), pp = below(P) - __builtin_popcountll(P & below_a);
        pf = pf < 0 ? pf + n_full : pf;
        pp = (pp < 0 ? pp + n : pp + n_full);
        int place = n + below(~(F | P));
        place = (F >> lane) & 1ull ? pf : ((P >> lane) & 1ull ? pp : place);
        const uint32_t list = (uint32_t)__builtin_amdgcn_ds_permute(place * 4, (int)(ub | (uint32_t)lane << 16));      // lane i: entry i

        // ---- staging, as k_small's: a wave copies CHW consecutive 1 KiB chunks of the A part and of the B part of a stage
        const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)smem;
        const int chunk0 = wave * H::CHW, slot = chunk0 / H::CPS, vec = (chunk0 % H::CPS) * 64;
        int ti = ti0 + slot, tj = tj0 + slot;
        ti = ti < nbM ? ti : nbM - 1;
        tj = tj < nbN ? tj : nbN - 1;
        const int within = (vec / H::RS) * B + vec % H::RS;            // 16-byte vector inside the tile's 4 k-groups
        const int row_bytes = nbK * H::TILE_BYTES;
        i32x4s rA = raw_buffer(pA + (int64_t)ti * row_bytes, row_bytes), rB = raw_buffer(pB + (int64_t)tj * row_bytes, row_bytes);
        const uint32_t voffA = (uint32_t)(lane + within + (int)(ui * U) % B) * 16, voffB = (uint32_t)(lane + within + (int)(uj * U) % B) * 16;
        const uint32_t ldsA = lds_base + chunk0 * 1024, ldsB = ldsA + H::OP_BYTES;
        const uint32_t needA = H::ROW_BITS << (slot * TU), needB = H::COL_BITS << slot;   // entry bits that read this slot

        // stage t's entry (of the last one's k, and with no tile, beyond it) and what its loads start from
        auto entry_at = [&](int t) -> uint32_t { return (uint32_t)__builtin_amdgcn_readlane((int)list, (t < S ? t : S - 1) / H::NSPE); };
        auto offset = [&](int t, uint32_t ent) -> uint32_t {
            const uint32_t k = (ent >> 16) * H::TILE_BYTES;
            if constexpr (H::NSPE == 1) return k;
            else return k + (uint32_t)(t % H::NSPE) * (B * 64);
        };
        auto issue_a = [&](uint32_t koff, uint32_t boff) { dma_buffer<H::CHW>(rA, voffA, koff, ldsA + boff); };
        auto issue_b = [&](uint32_t koff, uint32_t boff) { dma_buffer<H::CHW>(rB, voffB, koff, ldsB + boff); };
        auto sync_next = [&]() {
            __builtin_amdgcn_s_waitcnt(waitcnt_imm(H::LPW * (NBUF - 2), 0));
            __syncthreads();
        };
        auto frag_off = [&](int wsel, int blk) -> int {
            const int s = TU > 1 ? wsel + 2 * (blk * 16 / H::RS) : 0;
            const int ro = TU > 1 ? (blk * 16) % H::RS : wsel * (U / 2) + blk * 16;
            return s * H::RS * 64 + ((lane >> 4) * H::RS + ro + (lane & 15)) * 16;
        };
        struct Frags {
            half8 a[NB], b[NB];
        };
        auto load_frag = [&](Frags &f, uint32_t boff, auto idx) {
            constexpr int i = decltype(idx)::value;
            const unsigned char *bufA = smem + boff;
            if constexpr (i == 0) f.a[0] = *reinterpret_cast<const half8 *>(bufA + frag_off(wr, 0));
            else if constexpr (i <= NB) f.b[i - 1] = *reinterpret_cast<const half8 *>(bufA + H::OP_BYTES + frag_off(wc, i - 1));
            else f.a[i - NB] = *reinterpret_cast<const half8 *>(bufA + frag_off(wr, i - NB));
        };
        // ---- prologue
        const int all = row_bytes;
#pragma unroll
        for (int t = 0; t < NBUF; t++) {
            const uint32_t e = entry_at(t), koff = offset(t, e), bits = t < S ? e : 0u;
            rA.z = (bits & needA) ? all : 0;
            rB.z = (bits & needB) ? all : 0;
            issue_a(koff, t * H::STAGE_BYTES);
            issue_b(koff, t * H::STAGE_BYTES);
        }
        int t = 0;
        uint32_t buf = 0;
        auto next_buf = [&]() {
            uint32_t next = buf + H::STAGE_BYTES == NBUF * H::STAGE_BYTES ? 0u : buf + H::STAGE_BYTES;
            asm volatile("" : "+s"(next));
            return next;
        };
        __builtin_amdgcn_s_waitcnt(waitcnt_imm(H::LPW * (NBUF - 1), 0));
        __syncthreads();
        Frags f0, f1;
        static_for<2 * NB>([&](auto i) { load_frag(f0, 0, i); });
#define SPAMM_FENCE() __builtin_amdgcn_sched_barrier(0)
        // (every slot of a full stage is fetched, and of the partial ones that follow the last of them what the list's bits ask for or not)
        auto full_stage = [&](const Frags &cur, Frags &nxt) {
            const uint32_t next = next_buf();
            sync_next();
            SPAMM_FENCE();
            uint32_t en = 0, koff = 0;
            static_for<NB * NB>([&](auto idx) {
                constexpr int i = decltype(idx)::value, r = i / NB, c = i % NB, A_AT = NB == 4 ? 8 : 2, B_AT = NB == 4 ? 12 : 3;
                acc[r][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(cur.a[r], cur.b[c], acc[r][c], 0, 0, 0);
                if constexpr (i < 2 * NB) load_frag(nxt, next, idx);
                if constexpr (i == A_AT - 2) {
                    en = entry_at(t + NBUF);
                    rA.z = rB.z = t + NBUF < S ? all : 0;
                }
                if constexpr (i == A_AT - 1) koff = offset(t + NBUF, en);
                if constexpr (i == A_AT) issue_a(koff, buf);
                if constexpr (i == B_AT) issue_b(koff, buf);
                SPAMM_FENCE();
            });
            t++;
            buf = next;
        };
        while (__builtin_expect(t + 1 < Sfull, 1)) {
            full_stage(f0, f1);
            full_stage(f1, f0);
        }
        auto partial_stage = [&](const Frags &cur, Frags &nxt) {
            const uint32_t next = next_buf();
            const uint32_t ec = (entry_at(t) & 0xffffu) >> (TU > 1 ? wr * TU + wc : 0);
            const uint32_t en = entry_at(t + NBUF), koff = offset(t + NBUF, en), bits = t + NBUF < S ? en : 0u;
            rA.z = (bits & needA) ? all : 0;
            rB.z = (bits & needB) ? all : 0;
            sync_next();
            SPAMM_FENCE();
            static_for<H::NP * H::NP>([&](auto pair) {
                constexpr int p = decltype(pair)::value, px = p / H::NP, py = p % H::NP, bit = 2 * px * TU + 2 * py;
                if ((ec >> bit) & 1u) {
#pragma unroll
                    for (int r = 0; r < H::RB; r++)
#pragma unroll
                        for (int c = 0; c < H::RB; c++)
                            acc[px * H::RB + r][py * H::RB + c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                                cur.a[px * H::RB + r], cur.b[py * H::RB + c], acc[px * H::RB + r][py * H::RB + c], 0, 0, 0);
                }
                if constexpr (p == 0) {
                    SPAMM_FENCE();
                    static_for<2 * NB>([&](auto i) { load_frag(nxt, next, i); });
                    issue_a(koff, buf);
                    issue_b(koff, buf);
                    SPAMM_FENCE();
                }
            });
            SPAMM_FENCE();
            t++;
            buf = next;
        };
        while (t < S) {
            partial_stage(f0, f1);
            if (t >= S) break;
            partial_stage(f1, f0);
        }
#undef SPAMM_FENCE
        __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, 0));                 // the ring still holds loads of nothing

        // ---- C, as k_gemm's epilogue: a store is 32 lanes of each of two rows
        const int lane_off = 32 * (lane >> 5) * N + 4 * (lane & 31);     // bytes
        const int col00 = ucol + (TU > 1 ? wc * B : wc * (U / 2));
#pragma unroll
        for (int r = 0; r < NB; r++) {
            const int row0 = urow + (TU > 1 ? (wr + 2 * (r * 16 / B)) * B + (r * 16) % B : wr * (U / 2) + r * 16);
            if (row0 >= M) continue;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int soff = ((row0 + i) * N + col00) * 4;
#pragma unroll
                for (int c = 0; c < NB; c += 2) {
                    constexpr auto delta = [](int c) { return TU > 1 ? 2 * (c * 16 / B) * B + (c * 16) % B : c * 16; };
                    if (col00 + delta(c) >= N) continue;
                    const auto sw = __builtin_amdgcn_permlane16_swap(__float_as_uint(acc[r][c][i]), __float_as_uint(acc[r][c + 1][i]), false, false);
                    __builtin_amdgcn_raw_buffer_store_b32(sw[0], rc, lane_off + delta(c) * 4, soff, NT);
                    __builtin_amdgcn_raw_buffer_store_b32(sw[1], rc, lane_off + delta(c) * 4, soff + 16 * N, NT);
                }
            }
        }
    }
    store_gate();
}

// Stages in the ring.  Units of 64, ring of 4 | 5 | 6: short lists lose by a stage more (256^3 3.40 | 3.44 | 3.52 us, 1056 x 1568 x 1312
// 6.35 | 6.38 | 6.56), long ones by one less (1024 x 8192 x 1024 at tile 128, 30 % kept 15.2 | 13.2 | 13.0, 1024 x 2048 x 1024 dense 11.7 | 10.55 |
// 10.47).  Units of 128: 4, 6 and 8 are even alone, and behind the passes 6 and 8 lose 3 % (fp16 2048^3, 5 %: 18.6 | 19.2 | 19.6).
template <int U>
static constexpr int WORD_RING = U == 128 ? 4 : 5;

// The arguments, in the order of their use; a kernel for each tile size and unit.  They are functions of the names of the other form's templates, so
// that whoever lists a call's kernels sees the one-launch kernel, and three to a CU; B and U tell them apart, by which a list of full names shows
// the form.
template <int B, int U>
struct WordArgs {
    const unsigned char *pA, *pB;
    int nbM, nbK, nbN;
    SmallGrid sg;
    float tau;
    float *C;
    UnitGate g;
};
#define SPAMM_WORD(B, U)                                                                                     \
    __global__ __launch_bounds__(256, 2) void k_small(WordArgs<B, U> a) {                                    \
        small_word_body<B, U, WORD_RING<U>>(a.pA, a.pB, a.nbM, a.nbK, a.nbN, a.sg, a.tau, a.C, a.g);         \
    }
#define SPAMM_WORD_THREE(B)                                                                                  \
    __global__ __launch_bounds__(256, 3) void k_small_three(WordArgs<B, 128> a) {                            \
        small_word_body<B, 128, 3>(a.pA, a.pB, a.nbM, a.nbK, a.nbN, a.sg, a.tau, a.C, a.g);                  \
    }
SPAMM_WORD(32, 64)
SPAMM_WORD(32, 128)
SPAMM_WORD(64, 64)
SPAMM_WORD(64, 128)
SPAMM_WORD(128, 64)
SPAMM_WORD(128, 128)
SPAMM_WORD_THREE(32)
SPAMM_WORD_THREE(64)
SPAMM_WORD_THREE(128)
#undef SPAMM_WORD
#undef SPAMM_WORD_THREE

// Units of 128 in C, as many as 256 CUs would have for the same share of a CU: what the lines below balance is workgroups per
// CU and k_gemm's rounds of a macro tile per CU, so on a partition of fewer CUs they lie at as many units less.
static int64_t per_256_cus(int64_t units, int n_cu) { return (units * 256 + n_cu - 1) / n_cu; }
static int64_t units_of_128(int64_t M, int64_t N, int n_cu) { return per_256_cus(((M + 127) / 128) * ((N + 127) / 128), n_cu); }

// Unit by units of 128 in C: the wide one from half a unit per CU on.  Whole fp16 multiplies of inputs that change, 2 %, 10 %, 30 %
// kept and dense, narrow -> wide.  K = 2048 at tile 32 (K = 4096 at tiles 64 and 128 alike): 100 units 9.7 -> 11.7, 11.6 -> 14.1, 13.7 -> 17.3, 19.5 ->
// 21.6 us; 128 units 10.5 -> 12.6, 12.2 -> 14.9, 14.5 -> 18.5, 20.3 -> 22.0; 144 units 10.5 -> 12.3, 12.5 -> 14.5, 16.4 -> 18.0, 24.9 -> 22.1;
// 196 units 11.7 -> 13.2, 13.5 -> 15.5, 18.2 -> 19.0, 31.4 -> 23.8; 256 units 12.5 -> 13.7, 15.0 -> 16.1, 20.2 -> 20.3, 33.1 -> 26.9.  K = 6144
// at tile 32: 128 units 23.8 -> 26.1, 27.7 -> 31.4, 32.9 -> 35.5, 53.5 -> 55.6; 144 units 24.3 -> 25.6, 29.3 -> 30.3, 36.8 -> 34.5, 69.8 -> 54.9; 256
// units 29.8 -> 29.7, 41.1 -> 35.6, 49.4 -> 43.2, 94.1 -> 69.2.  Beyond 128 units, where four narrow ones a unit no longer run at once, two per CU,
// the line is a choice: a sparse product of few k pays up to 2 us for the 3 to 35 that a dense one, or one of more k, saves.  At 128
// units themselves, where the line was drawn before the list was a register, the narrow one is ahead by 1 to 4 us.
static int small_unit(int64_t units128) { return units128 >= 128 ? 128 : 64; }

// Clearly more than two units of 128 per CU: a ring of three stages leaves room for a third workgroup on the CU, whose loads
// and syncs fill the others' waits.  Ring of four, two workgroups -> this, whole fp16 multiplies of inputs that change, band of 10 % | 1 / (1 + d)^2,
// 40 % | dense.  K = 2048 at tile 32: 522 units 24.0 -> 25.3 | 35.6 -> 36.4 | 56.4 -> 53.5 us; 550 units 25.8 -> 24.7 | 38.5 -> 37.3 |
// 60.5 -> 55.3; 600 units 27.4 -> 26.1 | 43.2 -> 39.6 | 64.2 -> 57.3; 640 units 26.9 -> 27.1 | 47.4 -> 45.0 | 58.6 -> 56.1; 768 units 30.3 -> 29.1 | 50.2 ->
// 47.1 | 63.6 -> 61.7; 1024 units 36.2 -> 36.5 | 57.0 -> 58.2; 1296 units 47.9 -> 47.2 | 77.2 -> 72.6.  K = 4096 at tile 64: 522 units 38.0 -> 36.5 | 62.1 ->
// 64.5 | 111 -> 105; 600 units 37.9 -> 36.5 | 68.6 -> 62.8 | 121 -> 109; 768 units 43.6 -> 41.9 | 76.7 -> 71.4 | 118 -> 115; 1024 units 52.8 -> 51.5 | 89.5 ->
// 95.5.  K = 8192 at tile 128: 576 units 59.2 -> 62.5 | 102 -> 98.8 | 202 -> 195; 640 units 64.8 -> 67.5 | 114 -> 111 | 209 -> 205; 768 units 74.5 -> 70.8 | 126 -> 115 |
// 222 -> 219.  From 513 to some 540 units, where a second turn of two per CU is short, neither is the better one, and bands, whose few
// long lists want the longer ring, lose up to 1.5 us; from 550 on this one is ahead but for bands at tile 128.  The line is at 600 from when the
// list was not in a register and bands lost up to there.  A list too long for three in a CU's LDS keeps the ring of four.
static bool small_three(int64_t units128, int64_t nbK) {
    return units128 > 600 && 3 * (small_lds_bytes_(16384, 3, nbK) + 2048) <= 160 * 1024;
}

// (WORD: one word of k tiles)
template <int B, int U, bool THREE, bool WORD>
static constexpr auto small_kernel() {
    if constexpr (THREE && WORD) return static_cast<void (*)(WordArgs<B, 128>)>(&k_small_three);
    else if constexpr (THREE) return &k_small_three<B>;
    else if constexpr (WORD) return static_cast<void (*)(WordArgs<B, U>)>(&k_small);
    else return &k_small<B, U>;
}

template <int B, int U, bool THREE, bool WORD>
static size_t small_lds(int64_t nbK) {
    using H = SmallCfg<B, U, (THREE ? 3 : (WORD ? WORD_RING<U> : (U == 128 ? 4 : 6)))>;
    return WORD ? (size_t)H::STAGE_BYTES * H::NBUF : small_lds_bytes_(H::STAGE_BYTES, H::NBUF, nbK);
}

template <int B, int U, bool THREE>
static hipError_t launch_small_(const void *pA, const void *pB, const GateBuffers &g, int64_t M, int64_t K, int64_t N,
                                int mode, float tau, float *C, int n_xcd, hipStream_t s) {
    using H = SmallCfg<B, U, 4>;
    const int nbM = (int)(M / B), nbK = (int)(K / B), nbN = (int)(N / B);
    const int nMacM = (nbM + H::MT - 1) / H::MT, nMacN = (nbN + H::MT - 1) / H::MT;
    const int n_units = nMacM * nMacN * H::PD * H::PD;
    const unsigned grid = (unsigned)((n_units + n_xcd - 1) / n_xcd * n_xcd);
    const SmallGrid sg = {nMacN, 0xffffffffu / (uint32_t)nMacN, n_units, (n_units + n_xcd - 1) / n_xcd, __builtin_ctz((unsigned)n_xcd), mode};
    const unsigned char *a = (const unsigned char *)pA, *b = (const unsigned char *)pB;
    const UnitGate w = {g.nA, g.nBt, g.kept, g.counts, g.mask};
    if (nbK <= 64)
        small_kernel<B, U, THREE, true>()<<<grid, 256, small_lds<B, U, THREE, true>(nbK), s>>>(
            WordArgs<B, U>{a, b, nbM, nbK, nbN, sg, tau, C, w});
    else
        small_kernel<B, U, THREE, false>()<<<grid, 256, small_lds<B, U, THREE, false>(nbK), s>>>(a, b, nbM, nbK, nbN, sg, tau, C, w);
    return hipGetLastError();
}

template <int B, int U, bool THREE>
static hipError_t small_attr() {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(small_kernel<B, U, THREE, true>()),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)small_lds<B, U, THREE, true>(64));
    if (e != hipSuccess) return e;
    return hipFuncSetAttribute(reinterpret_cast<const void *>(small_kernel<B, U, THREE, false>()), hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int)small_lds<B, U, THREE, false>(SMALL_MAX_NBK));
}

template <int B>
static hipError_t small_attrs() {
    hipError_t e;
    if ((e = small_attr<B, 128, true>()) != hipSuccess || (e = small_attr<B, 128, false>()) != hipSuccess) return e;
    return small_attr<B, 64, false>();
}

hipError_t small_init() {
    hipError_t e;
    if ((e = small_attrs<32>()) != hipSuccess || (e = small_attrs<64>()) != hipSuccess) return e;
    return small_attrs<128>();
}

// Gate, schedule and GEMM apart -> this kernel, by units of 128 in C; "m" is the number of macro tiles (four units each), of which k_gemm runs
// 256 at a time.  Whole fp16 multiplies, three sets of operands and workspaces in turn on one stream; "from HBM": on operands converted
// before, 768 MiB of other writes since.
//
// tau > 0, at most 6 units per CU; exponential decay, 5 % kept | 1 / (1 + d)^2, 10 % | 25 % | 40 %.  K = 2048 at tile 32: 640 units 40.3 -> 24.4 |
// 43.3 -> 27.4 | 55.4 -> 36.0 | 63.4 -> 45.0 us; 840 units 45.0 -> 28.6 | 48.7 -> 33.7 | 62.5 -> 44.1 | 66.3 -> 50.6; 1024 units 48.0 -> 29.7 | 52.0 ->
// 35.6 | 65.8 -> 48.1 | 66.5 -> 58.5; 1444 units 53.7 -> 43.3 | 58.3 -> 49.6 | 71.0 -> 67.9 | 72.6 -> 78.4.  K = 4096 at tile 64: 840 units 56.6 ->
// 39.3 | 57.1 -> 47.3 | 72.7 -> 65.2 | 83.3 -> 81.2; 1024 units 60.8 -> 43.2 | 60.3 -> 53.1 | 79.4 -> 77.3 | 93.0 -> 95.5; 1296 units 62.2 -> 49.7 |
// 80.3 -> 64.3 | 106 -> 91 | 122 -> 122; 1444 units 66.2 -> 54.9 | 85.4 -> 70.8 | 112 -> 98 | 131 -> 126.  K = 8192 at tile 64: 840 units 80.8 -> 63.6 |
// 88.3 -> 78.9 | 113 -> 112 | 135 -> 136; 1024 units 84.6 -> 71.8 | 94.7 -> 91.4 | 121 -> 126 | 147 -> 153; 1296 units 92.2 -> 85.6 | 124 -> 114 | 173 -> 164 |
// 219 -> 200; 1444 units 97.5 -> 93.4 | 129 -> 123 | 178 -> 172 | 224 -> 222.  From HBM, K = 8192 at tile 64: 1024 units 57 -> 47 | 72 -> 68 | 99 -> 101 | 123 ->
// 138; 1296 units 62 -> 57 | 94 -> 79 | 134 -> 128 | 183 -> 168.
// In the one round that k_gemm fills (833 to 1024 units) K ends at 8192, where a quarter kept is even: beyond, 5 % | 10 % | 40 %: 840 units, K = 12288
// 112 -> 95 | 118 -> 111 | 180 -> 207, K = 16384 138 -> 123 | 146 -> 138 | 233 -> 266; 1024 units, K = 12288 119 -> 107 | 130 -> 129 | 192 -> 217, K = 16384
// 149 -> 136 | 165 -> 164 | 260 -> 297.  Beyond 6 units per CU: 1600 units, K = 3072 60.6 -> 51.6 | 70.3 -> 62.6 | 113 -> 116; 1936 units, K = 5120 86 -> 78 |
// 107 -> 102 | 179 -> 192; 2304 units, K = 5120 94 -> 85 | 127 -> 118 | 200 -> 223, K = 8192 130 -> 130 | 179 -> 178 | 324 -> 331.
//
// tau <= 0, everything is kept and the rounds are known.  Tile 64, K = 1024 | 2048 | 4096 | 8192.  With m = 160 to 192 a round is a third empty: 640
// units 42.2 -> 31.9 | 66.3 -> 55.2 | 116 -> 108 | 210 -> 209; 704 units 43.8 -> 33.3 | 68.3 -> 57.6 | 120 -> 111 | 215 -> 211; 768 units 44.6 -> 35.2 |
// 70.6 -> 60.0 | 123 -> 114 | 220 -> 218; but 600 units 41.0 -> 35.9 | 64.5 -> 62.2 | 112 -> 122 | 206 -> 233; 841 units 48.4 -> 43.2 | 75.4 -> 77.8 | 131 -> 157 |
// 237 -> 298; 1024 units 52.0 -> 44.1 | 82.4 -> 77.2 | 141 -> 147 | 247 -> 281.  With m = 257 to 324 a second round is mostly empty: 1088 units 74.8 -> 49.2 | 121 ->
// 91 | 210 -> 168 | 383 -> 321; 1296 units 77.9 -> 58.5 | 125 -> 108 | 216 -> 200 | 398 -> 394; 1444 units 78.7 -> 60.0 | 127 -> 111 | 223 -> 208 | 407 -> 424.  (The
// lines were drawn by K = 2048 and more, and by the schedule before k_order_few, which took 4 us more of the other side: K = 1024 gains at every
// one of these sizes now, and so do 520 and 576 units: 62.1 -> 54.9 and 62.5 -> 55.3 at K = 2048, even at 8192.)
//
// Gate and multiply called apart (`stages`) form mask and list twice, which costs less than the schedule does (fp32 passes, tau to a fraction, both
// stages, 1 / (1 + d)^2, 10 % | 25 % | 40 % kept): 1120 units, K = 2048 at tile 32 104 -> 83 | 120 -> 94 | 120 -> 103, K = 4096 at tile 64 130 -> 105 | 153 -> 129 |
// 170 -> 149; 1200 units 106 -> 86 | 120 -> 99 | 120 -> 109 and 134 -> 111 | 150 -> 132 | 173 -> 155; 1444 units 110 -> 94 | 122 -> 113 | 125 -> 123 and 141 ->
// 119 | 167 -> 146 | 187 -> 174.  In the round that k_gemm fills: 840 units, K = 2048 at tile 32 99.7 -> 77.4 | 114 -> 88 | 118 -> 95, K = 4128 117 -> 103 | 132 ->
// 119 | 144 -> 138, K = 8192 at tile 64 152 -> 137 | 177 -> 170 | 196 -> 194; 1024 units 103 -> 80 | 119 -> 93 | 118 -> 103, 123 -> 111 | 142 -> 134 | 154 -> 152 and 162 ->
// 152 | 186 -> 183 | 212 -> 213.  (Its lines -- 1200 units, and in that round one word of 64 k and K = 4096 -- are from before the list was a register and
// the gate of few instructions; up to 1536 units and K = 8192 this kernel is ahead, or even, throughout.)
bool small_fits(int64_t M, int64_t K, int64_t N, int tile, float tau, bool stages, int n_cu) {
    const int64_t units128 = units_of_128(M, N, n_cu), m = per_256_cus(((M + 255) / 256) * ((N + 255) / 256), n_cu);
    if (K / tile > SMALL_MAX_NBK || n_cu > 256) return false;
    static_assert(SMALL_MAX_UNITS >= 6 * 256 && SMALL_MAX_UNITS >= 4 * 127, "units of either size");
    if (units128 <= 512) return true;
    if (stages) return tau > 0.0f && units128 <= 1200 && (units128 <= 832 || units128 > 1024 || (K <= 4096 && K / tile <= 64));
    if (tau > 0.0f) return units128 <= SMALL_MAX_UNITS && (units128 <= 832 || units128 > 1024 || K <= 8192);
    return (m >= 160 && m <= 192) || (m >= 257 && m <= 324);
}

template <int B>
static hipError_t launch_small_(const void *pA, const void *pB, const GateBuffers &g, int64_t M, int64_t K, int64_t N,
                                int mode, float tau, float *C, int n_cu, int n_xcd, hipStream_t s) {
    const int64_t units128 = units_of_128(M, N, n_cu);
    if (small_unit(units128) != 128) return launch_small_<B, 64, false>(pA, pB, g, M, K, N, mode, tau, C, n_xcd, s);
    if (small_three(units128, K / B)) return launch_small_<B, 128, true>(pA, pB, g, M, K, N, mode, tau, C, n_xcd, s);
    return launch_small_<B, 128, false>(pA, pB, g, M, K, N, mode, tau, C, n_xcd, s);
}

hipError_t launch_small(const void *packedA, const void *packedB, const GateBuffers &g, int64_t M, int64_t K, int64_t N,
                        int tile, int mode, float tau, float *C, int n_cu, int n_xcd, hipStream_t s) {
    switch (tile) {
        case 32: return launch_small_<32>(packedA, packedB, g, M, K, N, mode, tau, C, n_cu, n_xcd, s);
        case 64: return launch_small_<64>(packedA, packedB, g, M, K, N, mode, tau, C, n_cu, n_xcd, s);
        case 128: return launch_small_<128>(packedA, packedB, g, M, K, N, mode, tau, C, n_cu, n_xcd, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace spamm
