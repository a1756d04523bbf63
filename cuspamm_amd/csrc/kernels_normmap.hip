// Stage 1: fused fp32 -> fp16 conversion + tile Frobenius norm map.
//
// Replaces the reference's norm kernels (cuSpAMM.cu:21-71 fp32, :74-123 fp16)
// and its host-side element-wise __float2half (tool.cu:418,432).  HBM-bound:
// per element 4 bytes read, 2 bytes written.  The fp16 copy is written in the
// packed tile layout described in spamm_internal.h so that the gated GEMM can
// stream MFMA operands without any transposition.
//
// Norm accumulation order (fp32, bit-identical to the host checker):
//   chunk(r,q) = ((((0 + x0^2) + x1^2) + ... ) + x7^2) over 8 consecutive
//   elements along the contraction axis (x = fp16-rounded value; squares are
//   exact in fp32); chunk index c = r*(b/8)+q; lane L = c%64 accumulates
//   chunks c = L, 64+L, 128+L, ... in ascending order; then a 6-step xor
//   butterfly (1,2,4,8,16,32) across the 64 lanes; norm = sqrtf(sum).
#include <type_traits>

#include "spamm_internal.h"

namespace spamm {

typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4n __attribute__((ext_vector_type(4)));
typedef _Float16 half8n __attribute__((ext_vector_type(8)));

// Convert two floats to fp16 (round-to-nearest-even), add their squares to s
// in order (a then b) and return the packed pair.
__device__ __forceinline__ uint32_t cvt_pack2(float a, float b, float &s) {
    _Float16 ha = (_Float16)a;
    _Float16 hb = (_Float16)b;
    float fa = (float)ha;
    float fb = (float)hb;
    s = s + fa * fa;
    s = s + fb * fb;
    half2v v = {ha, hb};
    return __builtin_bit_cast(uint32_t, v);
}

__device__ __forceinline__ float butterfly64(float v) {
#pragma unroll
    for (int s = 1; s < 64; s <<= 1) v = v + __shfl_xor(v, s, 64);
    return v;
}

// One workgroup per strip of B rows x SW columns (SW/B tiles).  A wave-wide load is one strip row of
// 1 KiB (fp32, SW = 256) or a row each of two or four 8-row groups.  The
// tiles of a strip pass through LDS in PH phases of SW/B/PH tiles each, sized so that at most
// ~42 KiB are resident and three workgroups fit a CU; all loads are issued before the first phase.
//   load    a lane takes whole 8-row groups; all loads of a lane
//           are in flight together.
//   convert fp32 input, A role: a lane holds half a chunk (4 of 8 elements along k); the odd lane
//           continues the even lane's running sum (DPP) so that the chunk is summed left to
//           right.  B role: a lane holds 8 rows x 4 columns and transposes in registers into 4
//           k-contiguous vectors.  fp16 input: a lane's 16 bytes are a whole chunk (A role) or,
//           over 8 rows, an 8 x 8 block transposed in registers (B role).
//   stage   fp16 vectors go to LDS in the packed tile layout (k-group segments padded by 16
//           bytes against bank conflicts), chunk sums to LDS at their canonical index.
//   store   after one barrier: the tiles are copied out with contiguous 1 KiB wave stores (a
//           packed tile is one contiguous block in memory), and one wave per tile applies the
//           canonical reduction.
template <int B, int SW, int PH>
struct NormCfg {
    static constexpr int TPP = SW / B / PH;          // tiles resident in LDS together
    static constexpr int QN = B / 8;                 // k-groups per tile
    static constexpr int QS = B * 16 + 16;           // bytes per k-group segment in LDS (padded)
    static constexpr int TS = QN * QS;               // bytes per tile in LDS
    static constexpr int PITCH = QN + 1;             // padded row of the chunk-sum table
    static constexpr int CH = B * PITCH;             // floats per tile in the chunk-sum table
};

// `strip`: which strip of the operand; s_pack / s_chunk / s_skip / s_seen: NormCfg's TPP * TS bytes, TPP * CH floats, TPP and NWV
// ints of LDS
template <int B, int ROLE, int SW, bool IN16, int PH, int NWV>
__device__ __forceinline__ void normmap_strip(const void *__restrict__ Xv, int64_t ld, int64_t cols, int64_t nbr, int64_t nbc,
                                              int64_t nstrip, uint4 *__restrict__ packed, float *__restrict__ nm,
                                              float *__restrict__ nmT, uint4 *__restrict__ packed2, float *__restrict__ nm2,
                                              const float *__restrict__ rowmax, float tau_skip, bool keep_copy, unsigned strip,
                                              unsigned char *s_pack, float *s_chunk, int *s_skip, int *s_seen) {
    using L = NormCfg<B, SW, PH>;
    constexpr int TPS = SW / B;           // tiles per strip
    constexpr int TPP = TPS / PH;         // tiles per phase (resident in LDS together)
    static_assert(TPP * PH == TPS && TPP >= 1, "phases must divide the strip's tiles");
    // Lane -> element mapping: LPR lanes of EPL columns (4 floats or 8 halves, 16 bytes) are a strip row; a
    // wave-wide load is a row of each of GPW 8-row groups.  A lane's columns lie in one tile; with PH > 1 the tiles
    // pass through LDS PH phases one after the other and in phase ph only the lanes of that
    // phase's tiles stage their data.  Tiles of 128 as strips of several in as many phases put up to
    // 128 KiB in registers per workgroup, staged, copied and reduced in turns with little else on the CU
    // to read meanwhile; as single tiles (SW = B: a load is rows of several 8-row groups) a workgroup is
    // what it is at tile 64.  Both passes, phased -> single: fp32 1024^2 18.6 -> 5.6 us, 4096^2 50 -> 36,
    // A = B in one read 8192^2 145 -> 90; fp16 1024^2 13 -> 4.6, 16384^2 tau-aware 302 -> 276.
    constexpr int EPL = IN16 ? 8 : 4;                  // columns per lane
    constexpr int LPR = SW / EPL;                      // lanes per strip row
    constexpr int GPW = 64 / LPR;                      // 8-row groups a wave-wide load touches (a row of each)
    static_assert(LPR * GPW == 64 && (GPW == 1 || PH == 1), "a wave-wide load is whole strip rows");
    constexpr int GSTEP = NWV * GPW;                   // 8-row groups between a lane's groups
    static_assert(B % (8 * GSTEP) == 0, "every wave takes whole 8-row groups");
    static_assert(PH == 1 || PH == 2 || PH == 4, "phases are made of whole waves");
    constexpr int QN = L::QN, QS = L::QS, TS = L::TS, PITCH = L::PITCH, CH = L::CH;
    constexpr int VPT = B * B / 8;        // 16-byte vectors per tile
    constexpr int NGW = B / (8 * GSTEP);  // 8-row groups per lane
    constexpr int STEPS = VPT / 64;
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int64_t I = strip / nstrip;                 // tile row of the strip
    const int64_t sc = strip % nstrip;
    const int64_t col0 = sc * SW;
    const int cl = EPL * (lane % LPR);                // first column of this lane inside the strip
    const int g0 = wave * GPW + lane / LPR;           // first 8-row group of this lane; then every GSTEP-th
    const int t = cl / B, cin = cl % B;               // tile of the strip, column inside the tile
    const bool valid = col0 + cl < cols;
    const int64_t eoff = (I * B) * ld + col0 + cl;

    // fp32 input: v holds the lane's elements; fp16 input (the reference's own input type,
    // para.h:1): h16 holds them as loaded -- the conversion is then the identity and only the
    // packing and the norms remain.
    f32x4 v[IN16 ? 1 : NGW][8];
    u32x4n h16[IN16 ? NGW : 1][8];
    if (IN16) {
        // every lane loads unconditionally (a lane beyond the last column reads the strip's first
        // columns instead and zeroes the values afterwards): with the loads inside a branch the
        // compiler waits for each one before it issues the next
        const _Float16 *src = static_cast<const _Float16 *>(Xv) + (valid ? eoff : (I * B) * ld + col0);
#pragma unroll
        for (int i = 0; i < NGW; i++)
#pragma unroll
            for (int j = 0; j < 8; j++) {
                h16[i][j] = __builtin_nontemporal_load(
                    reinterpret_cast<const u32x4n *>(src + (int64_t)(8 * (g0 + GSTEP * i) + j) * ld));
            }
        if (!valid) {
#pragma unroll
            for (int i = 0; i < NGW; i++)
#pragma unroll
                for (int j = 0; j < 8; j++) h16[i][j] = u32x4n{0u, 0u, 0u, 0u};
        }
    } else {
#pragma unroll
        for (int i = 0; i < NGW; i++)
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const int r = 8 * (g0 + GSTEP * i) + j;
                if (!valid)
                    v[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                else
                    v[i][j] = __builtin_nontemporal_load(
                        reinterpret_cast<const f32x4 *>(static_cast<const float *>(Xv) + eoff + (int64_t)r * ld));
            }
    }
    // LDS position of the 16-byte vector of free index x inside a k-group segment.  The fp16-input
    // B role writes 8 neighbouring x per lane, lanes 128 bytes apart: the low three bits of x are
    // xor-ed with the next three so that the lanes of one store spread over the banks.
    auto vpos = [](int x, bool swz) -> int { return swz ? (x ^ ((x >> 3) & 7)) : x; };

    float seen = 0.0f;                                // sum of the chunk sums that the lane has staged

    // ROLE 2 = the same matrix is both operands (A = B): one read of X, both packed layouts and
    // both norm maps (A role first -> packed/nm, then B role -> packed2/nm2/nmT), LDS reused.
    auto stage_a = [&](int ph) {
        const int q = cin / 8, h = (cin % 8) / 4;
        if (PH > 1 && t / TPP != ph) return;
        const int t = (cl / B) % TPP;      // tile inside the phase
        if constexpr (IN16) {
            // the lane's 16 bytes are one whole chunk (8 consecutive k of row r): already a packed vector
#pragma unroll
            for (int i = 0; i < NGW; i++)
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    const int r = 8 * (g0 + GSTEP * i) + j;
                    const half8n hv = __builtin_bit_cast(half8n, h16[i][j]);
                    float s8 = 0.0f;
#pragma unroll
                    for (int e = 0; e < 8; e++) { const float f = (float)hv[e]; s8 = s8 + f * f; }
                    *reinterpret_cast<u32x4n *>(s_pack + t * TS + q * QS + r * 16) = h16[i][j];
                    s_chunk[t * CH + r * PITCH + q] = s8;
                    seen += s8;
                }
        } else {
#pragma unroll
        for (int i = 0; i < NGW; i++)
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const int r = 8 * (g0 + GSTEP * i) + j;
                const _Float16 h0 = (_Float16)v[i][j].x, h1 = (_Float16)v[i][j].y;
                const _Float16 h2 = (_Float16)v[i][j].z, h3 = (_Float16)v[i][j].w;
                const float f0 = (float)h0, f1 = (float)h1, f2 = (float)h2, f3 = (float)h3;
                float s = 0.0f;
                s = s + f0 * f0; s = s + f1 * f1; s = s + f2 * f2; s = s + f3 * f3;
                // odd lane: continue from the even neighbour's sum (elements 0..3 of the chunk)
                const float nb = __builtin_bit_cast(
                    float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, s), 0xA0, 0xF, 0xF, false));
                float s8 = nb;
                s8 = s8 + f0 * f0; s8 = s8 + f1 * f1; s8 = s8 + f2 * f2; s8 = s8 + f3 * f3;
                const half2v p0 = {h0, h1}, p1 = {h2, h3};
                uint2 o;
                o.x = __builtin_bit_cast(uint32_t, p0);
                o.y = __builtin_bit_cast(uint32_t, p1);
                *reinterpret_cast<uint2 *>(s_pack + t * TS + q * QS + r * 16 + h * 8) = o;
                if (h) s_chunk[t * CH + r * PITCH + q] = s8;
                seen += s8;
            }
        }
    };
    auto stage_b = [&](int ph) {
        if (PH > 1 && t / TPP != ph) return;
        const int t = (cl / B) % TPP;      // tile inside the phase
        if constexpr (IN16) {
            // the lane holds 8 rows (one k-group) x 8 columns: transposed in registers into 8
            // k-contiguous vectors, one per column
#pragma unroll
            for (int i = 0; i < NGW; i++) {
                const int kg = g0 + GSTEP * i;
                half8n rows[8];
#pragma unroll
                for (int j = 0; j < 8; j++) rows[j] = __builtin_bit_cast(half8n, h16[i][j]);
#pragma unroll
                for (int c = 0; c < 8; c++) {
                    half8n o;
                    float sc_ = 0.0f;
#pragma unroll
                    for (int j = 0; j < 8; j++) {
                        o[j] = rows[j][c];
                        const float f = (float)rows[j][c];
                        sc_ = sc_ + f * f;
                    }
                    *reinterpret_cast<u32x4n *>(s_pack + t * TS + kg * QS + vpos(cin + c, true) * 16) =
                        __builtin_bit_cast(u32x4n, o);
                    s_chunk[t * CH + (cin + c) * PITCH + kg] = sc_;
                    seen += sc_;
                }
            }
        } else {
#pragma unroll
        for (int i = 0; i < NGW; i++) {
            const int kg = g0 + GSTEP * i;
            uint4 o[4];
            float s[4] = {0.0f, 0.0f, 0.0f, 0.0f};
            o[0].x = cvt_pack2(v[i][0].x, v[i][1].x, s[0]);
            o[0].y = cvt_pack2(v[i][2].x, v[i][3].x, s[0]);
            o[0].z = cvt_pack2(v[i][4].x, v[i][5].x, s[0]);
            o[0].w = cvt_pack2(v[i][6].x, v[i][7].x, s[0]);
            o[1].x = cvt_pack2(v[i][0].y, v[i][1].y, s[1]);
            o[1].y = cvt_pack2(v[i][2].y, v[i][3].y, s[1]);
            o[1].z = cvt_pack2(v[i][4].y, v[i][5].y, s[1]);
            o[1].w = cvt_pack2(v[i][6].y, v[i][7].y, s[1]);
            o[2].x = cvt_pack2(v[i][0].z, v[i][1].z, s[2]);
            o[2].y = cvt_pack2(v[i][2].z, v[i][3].z, s[2]);
            o[2].z = cvt_pack2(v[i][4].z, v[i][5].z, s[2]);
            o[2].w = cvt_pack2(v[i][6].z, v[i][7].z, s[2]);
            o[3].x = cvt_pack2(v[i][0].w, v[i][1].w, s[3]);
            o[3].y = cvt_pack2(v[i][2].w, v[i][3].w, s[3]);
            o[3].z = cvt_pack2(v[i][4].w, v[i][5].w, s[3]);
            o[3].w = cvt_pack2(v[i][6].w, v[i][7].w, s[3]);
#pragma unroll
            for (int c = 0; c < 4; c++) {
                *reinterpret_cast<uint4 *>(s_pack + t * TS + kg * QS + (cin + c) * 16) = o[c];
                s_chunk[t * CH + (cin + c) * PITCH + kg] = s[c];
                seen += s[c];
            }
        }
        }
    };
    // packed tiles out (256 threads x 16 bytes = 4 KiB per step, contiguous per tile)
    auto copy_out_as = [&](int ph, bool as_b, uint4 *__restrict__ pk, bool prune, auto keep) {
#pragma unroll
        for (int i = 0; i < TPP * VPT / (64 * NWV); i++) {
            const int vi = threadIdx.x + 64 * NWV * i;
            const int tt = vi / VPT, iv = vi % VPT;
            const int64_t Jt = sc * TPS + ph * TPP + tt;
            if (Jt < nbc && !(prune && s_skip[tt])) {
                const uint4 d = *reinterpret_cast<const uint4 *>(s_pack + tt * TS + (iv / B) * QS + vpos(iv % B, IN16 && as_b) * 16);
                const int64_t tile = as_b ? Jt * nbr + I : I * nbc + Jt;
                const u32x4n dv = *reinterpret_cast<const u32x4n *>(&d);
                u32x4n *to = reinterpret_cast<u32x4n *>(pk + tile * VPT + iv);
                if constexpr (decltype(keep)::value) asm volatile("global_store_dwordx4 %0, %1, off sc1\n\ts_nop 1" :: "v"(to), "v"(dv) : "memory");
                else __builtin_nontemporal_store(dv, to);
            }
        }
    };
    // (a strip of nothing but zeros, which no threshold above zero keeps, is not left in the cache)
    auto copy_out = [&](int ph, bool as_b, uint4 *__restrict__ pk, bool prune) {
        int any = 0;
#pragma unroll
        for (int w = 0; w < NWV; w++) any |= s_seen[w];
        if (keep_copy && __builtin_amdgcn_readfirstlane(any)) copy_out_as(ph, as_b, pk, prune, std::true_type{});
        else copy_out_as(ph, as_b, pk, prune, std::false_type{});
    };
    // norms: one wave per tile, canonical order.  With `prune` (tau known and positive) the wave
    // also decides whether any product can keep the tile.  The A pass of its own has the row maxima
    // (B's norm map is complete by then): fl(n * n') <= fl(n * max_j nB[k,j]) for every partner norm
    // n' because rounding is monotone, so a tile whose product with the maximum is below tau is never
    // read by the GEMM and its fp16 copy need not be written.  The other passes know no partner, and
    // their copies serve any tau > 0 afterwards: they leave out tiles of norm zero (0 * n' is 0 or NaN).
    auto norms = [&](int ph, bool as_b, float *__restrict__ nmo, float *__restrict__ nmTo, bool prune) {
        for (int tt = wave; tt < TPP; tt += NWV) {
            const int64_t Jt = sc * TPS + ph * TPP + tt;
            if (Jt >= nbc) break;
            const bool bounded = prune && rowmax != nullptr;
            const float rmax = bounded ? rowmax[Jt] : 0.0f;
            float partial = 0.0f;
#pragma unroll
            for (int it = 0; it < STEPS; it++) {
                const int c = it * 64 + lane;
                partial = partial + s_chunk[tt * CH + (c / QN) * PITCH + (c % QN)];
            }
            partial = butterfly64(partial);
            if (lane == 0) {
                const float nv = sqrtf(partial);
                nmo[I * nbc + Jt] = nv;
                if (as_b) nmTo[Jt * nbr + I] = nv;
                if (prune) s_skip[tt] = bounded ? nv * rmax < tau_skip : nv == 0.0f;
            }
        }
    };
    // one operand role: the strip's tiles go through LDS phase by phase
    auto emit_role = [&](bool as_b, uint4 *__restrict__ pk, float *__restrict__ nmo, float *__restrict__ nmTo,
                         bool prune) {
#pragma unroll
        for (int ph = 0; ph < PH; ph++) {
            if (ph) __syncthreads();           // the previous phase's tiles have been copied out
            seen = 0.0f;
            if (as_b) stage_b(ph); else stage_a(ph);
            const bool used = __ballot(seen != 0.0f) != 0ull;
            if (lane == 0) s_seen[wave] = used;
            __syncthreads();
            if (prune) {
                norms(ph, as_b, nmo, nmTo, true);
                __syncthreads();
                copy_out(ph, as_b, pk, true);
            } else {
                copy_out(ph, as_b, pk, false);
                norms(ph, as_b, nmo, nmTo, false);
            }
        }
    };
    const bool prune = tau_skip > 0.0f;
    if (ROLE == 0) {
        emit_role(false, packed, nm, nullptr, prune);
    } else if (ROLE == 1) {
        emit_role(true, packed, nm, nmT, prune);
    } else {
        // one pass for both roles: no row maxima yet, so only tiles of norm zero are left out
        emit_role(false, packed, nm, nullptr, prune);
        // (With two groups per lane the second role converts again: kept from the first, values and squares were 174 registers a
        // lane, of which 168 leave room for the third workgroup that a CU's LDS holds.  Tau-aware squares of 16384: 472 -> 417 us for 0.07 %
        // of a narrow band, 1188 -> 1133 for 10 % of a wide one.)
        if constexpr (!IN16 && NGW > 1) {
#pragma unroll
            for (int i = 0; i < NGW; i++)
#pragma unroll
                for (int j = 0; j < 8; j++) asm volatile("" : "+v"(v[i][j]));
        }
        __syncthreads();
        emit_role(true, packed2, nm2, nmT, prune);
    }
}

template <int B, int ROLE, int SW, bool IN16, int PH = 1, int NWV = 4>
__global__ __launch_bounds__(64 * NWV, 1) void k_normmap(
    const void *__restrict__ Xv, int64_t ld, int64_t cols, int64_t nbr, int64_t nbc, int64_t nstrip, uint4 *__restrict__ packed,
    float *__restrict__ nm, float *__restrict__ nmT, uint4 *__restrict__ packed2, float *__restrict__ nm2,
    const float *__restrict__ rowmax, float tau_skip, bool keep_copy) {
    using L = NormCfg<B, SW, PH>;
    __shared__ __attribute__((aligned(16))) unsigned char s_pack[L::TPP * L::TS];
    __shared__ float s_chunk[L::TPP * L::CH];
    __shared__ int s_skip[L::TPP], s_seen[NWV];
    normmap_strip<B, ROLE, SW, IN16, PH, NWV>(Xv, ld, cols, nbr, nbc, nstrip, packed, nm, nmT, packed2, nm2, rowmax, tau_skip,
                                              keep_copy, blockIdx.x, s_pack, s_chunk, s_skip, s_seen);
}

// Both operands in one launch: the first n_b workgroups are B's strips, the others A's.  One after the other,
// small passes are a few microseconds of memory latency each; together they share it (and neither sees the
// other's norms: a tau-aware call then leaves out tiles of norm zero only, in both copies).
template <int B, int SW, bool IN16, int PH, int NWV>
__global__ __launch_bounds__(64 * NWV) void k_normmap_pair(const void *__restrict__ A, const void *__restrict__ Bm, int64_t nbM,
                                                           int64_t nbK, int64_t nbN, unsigned n_b, int64_t strips_a, int64_t strips_b,
                                                           uint4 *__restrict__ packedA, uint4 *__restrict__ packedB,
                                                           float *__restrict__ nmA, float *__restrict__ nmB,
                                                           float *__restrict__ nmBt, float tau_skip, bool keep_copy) {
    using L = NormCfg<B, SW, PH>;
    __shared__ __attribute__((aligned(16))) unsigned char s_pack[L::TPP * L::TS];
    __shared__ float s_chunk[L::TPP * L::CH];
    __shared__ int s_skip[L::TPP], s_seen[NWV];
    if (blockIdx.x < n_b)
        normmap_strip<B, 1, SW, IN16, PH, NWV>(Bm, nbN * B, nbN * B, nbK, nbN, strips_b, packedB, nmB, nmBt, nullptr, nullptr,
                                               nullptr, tau_skip, keep_copy, blockIdx.x, s_pack, s_chunk, s_skip, s_seen);
    else
        normmap_strip<B, 0, SW, IN16, PH, NWV>(A, nbK * B, nbK * B, nbM, nbK, strips_a, packedA, nmA, nullptr, nullptr, nullptr,
                                               nullptr, tau_skip, keep_copy, blockIdx.x - n_b, s_pack, s_chunk, s_skip, s_seen);
}

// ---- the same strip in fewer instructions, with one 8-row group per lane and one phase.  In a small launch (at most KEEP_INPUT_MAX bytes
// of input) there is little to stream: a workgroup's waves are almost alone on their SIMDs, issue an instruction in some five clocks, and the pass takes as long as its chain of instructions.  So everything is
// addressed by 32-bit offsets into buffers that begin at the strip -- rows by the scalar offset, a lane beyond the last column or a tile
// beyond the last one by an offset that the buffer does not hold, without a branch --, the strip's place comes from a reciprocal
// instead of a 64-bit division, and a wave reduces all its tiles' norms together, by lane exchanges that are not LDS operations.
// Both operands in one launch, alone, inputs from HBM, the streaming kernel -> this: 256^3 3.83 -> 3.01 us (of which 1.55 are an empty
// launch), 1024^3 at tile 64 4.48 -> 4.14, 1056 x 1568 x 1312 8.2 -> 7.4, fp16 1024 x 2048 x 1024 5.93 -> 4.82, 2048^3 at tile 32 10.3 -> 8.1,
// 512^3 at tile 128 3.50 -> 3.39 (one wave adds a lane's 32 chunks in their order).
// Large inputs are bound by the HBM, and take it where it is not slower (launch_normmap); passes alone: tile 32 5024 x 4128 fp32 22.2 -> 21.0 us,
// tau-aware 23.0 -> 20.6, fp16 5024^2 20.5 -> 19.3, tau-aware 17.8 -> 16.2, 12032^2 155 -> 153.5; fp32 tile 64 4096^2 A = B 25.9 -> 24.2, both operands in
// one launch 33.6 -> 32.4, 8192^2 61.7 -> 61.0.  Reads alone reach 6.8 to 7.2 TB/s there; as soon as one workgroup in sixteen writes its
// tile the whole comes to 5.5 to 5.8, in whatever order or policy (4 GiB read, 1/16, 3/16, all of the copies written: 624 -> 770, 870, 1090 us).
// Buffer loads are of whole 32-bit words (an address's lowest two bits need not count): a matrix of halves that begins between two
// of them (whole_words) stays with the streaming kernel, whose loads are global ones and take any address.
//
// Sum over the 64 lanes, in every lane: the same additions as butterfly64.  (Behind the steps of 1 and 2 all lanes of a quad hold one sum, so
// that a mirrored quad is the neighbour; likewise for 8.)
__device__ __forceinline__ float butterfly64_dpp(float v) {
    auto dpp = [](float x, auto ctrl) {
        const int i = __builtin_bit_cast(int, x);
        return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(i, i, decltype(ctrl)::value, 0xF, 0xF, false));
    };
    v = v + dpp(v, std::integral_constant<int, 0xB1>{});       // lanes 1, 0, 3, 2 of a quad
    v = v + dpp(v, std::integral_constant<int, 0x4E>{});       // lanes 2, 3, 0, 1
    v = v + dpp(v, std::integral_constant<int, 0x141>{});      // half a row mirrored: the other quad
    v = v + dpp(v, std::integral_constant<int, 0x140>{});      // a row mirrored: the other half
    const auto r16 = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, v), __builtin_bit_cast(uint32_t, v), false, false);
    v = __builtin_bit_cast(float, (uint32_t)r16[0]) + __builtin_bit_cast(float, (uint32_t)r16[1]);
    const auto r32 = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, v), __builtin_bit_cast(uint32_t, v), false, false);
    return __builtin_bit_cast(float, (uint32_t)r32[0]) + __builtin_bit_cast(float, (uint32_t)r32[1]);
}

// A strip's place: row and column of strips by a reciprocal, exact while strips * nstrip <= 2^32; else (0) by a division.
inline uint32_t strip_reciprocal(uint32_t strips, uint32_t nstrip) { return (uint64_t)strips * nstrip < 0xffffffffull ? 0xffffffffu / nstrip : 0u; }

// KEEP: the input's lines stay in the caches (keep_input).
template <int B, int ROLE, int SW, bool IN16, int NWV, bool KEEP>
__device__ __forceinline__ void normmap_strip_lean(const void *X, uint32_t cols, uint32_t nbr, uint32_t nbc, uint32_t nstrip, uint32_t rec,
                                                    void *packed, float *nm, float *nmT, void *packed2, float *nm2, const float *rowmax,
                                                    float tau_skip, bool keep_copy, uint32_t strip, unsigned char *s_pack, float *s_chunk,
                                                    int *s_skip, int *s_seen) {
    using L = NormCfg<B, SW, 1>;
    constexpr int TPP = L::TPP, QN = L::QN, QS = L::QS, TS = L::TS, PITCH = L::PITCH, CH = L::CH;
    constexpr int E = IN16 ? 2 : 4, EPL = 16 / E;      // bytes per element, elements per lane
    constexpr int LPR = SW / EPL, GPW = 64 / LPR;      // lanes per strip row, 8-row groups of a wave
    static_assert(B == 8 * NWV * GPW, "a lane has one 8-row group");
    constexpr int VPT = B * B / 8, STEPS = VPT / 64;   // 16-byte vectors per tile; chunks per lane of its norm
    constexpr int NT = TPP > NWV ? TPP / NWV : 1;      // tiles per wave of the norms
    constexpr uint32_t NOWHERE = 0x80000000u, TB = B * B * 2;          // an offset no output buffer here holds; bytes of a tile
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t I = rec ? __umulhi(strip + 1u, rec) : strip / nstrip, sc = strip - I * nstrip, col0 = sc * SW, J0 = sc * TPP;
    const uint32_t ld = cols * E;                      // bytes per row (of which B are less than 4 GiB)
    const int cl = EPL * (lane % LPR);                 // first column of this lane inside the strip
    const int t = cl / B, cin = cl % B;                // tile of the strip, column inside the tile
    const int g = wave * GPW + lane / LPR;             // 8-row group of this lane
    const __amdgpu_buffer_rsrc_t in = __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned char *>(static_cast<const unsigned char *>(X)) + (uint64_t)I * B * ld + (uint64_t)col0 * E, 0,
                                                                        (int)((B - 1) * ld + (cols - col0) * E), 0x00020000);
    u32x4n x[8];
    {
        const uint32_t voff = col0 + cl < cols ? (uint32_t)(lane / LPR) * 8u * ld + (uint32_t)cl * E : 0xffffff00u;
        uint32_t soff = (uint32_t)(wave * GPW * 8) * ld;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            x[j] = __builtin_bit_cast(u32x4n, __builtin_amdgcn_raw_buffer_load_b128(in, (int)voff, (int)soff, KEEP ? 0 : 2));
            soff += ld;
        }
    }
    auto vpos = [](int f, bool swz) -> int { return swz ? (f ^ ((f >> 3) & 7)) : f; };     // (as in normmap_strip)
    float seen = 0.0f;
    auto stage_a = [&]() {
        const int q = cin / 8, h = (cin % 8) / 4;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const int r = 8 * g + j;
            if constexpr (IN16) {
                const half8n hv = __builtin_bit_cast(half8n, x[j]);
                float s8 = 0.0f;
#pragma unroll
                for (int e = 0; e < 8; e++) { const float f = (float)hv[e]; s8 = s8 + f * f; }
                *reinterpret_cast<u32x4n *>(s_pack + t * TS + q * QS + r * 16) = x[j];
                s_chunk[t * CH + r * PITCH + q] = s8;
                seen += s8;
            } else {
                const f32x4 v = __builtin_bit_cast(f32x4, x[j]);
                const _Float16 h0 = (_Float16)v.x, h1 = (_Float16)v.y, h2 = (_Float16)v.z, h3 = (_Float16)v.w;
                const float f0 = (float)h0, f1 = (float)h1, f2 = (float)h2, f3 = (float)h3;
                float s = 0.0f;
                s = s + f0 * f0; s = s + f1 * f1; s = s + f2 * f2; s = s + f3 * f3;
                float s8 = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, s), 0xA0, 0xF, 0xF, false));
                s8 = s8 + f0 * f0; s8 = s8 + f1 * f1; s8 = s8 + f2 * f2; s8 = s8 + f3 * f3;
                const half2v p0 = {h0, h1}, p1 = {h2, h3};
                uint2 o;
                o.x = __builtin_bit_cast(uint32_t, p0);
                o.y = __builtin_bit_cast(uint32_t, p1);
                *reinterpret_cast<uint2 *>(s_pack + t * TS + q * QS + r * 16 + h * 8) = o;
                if (h) s_chunk[t * CH + r * PITCH + q] = s8;
                seen += s8;
            }
        }
    };
    auto stage_b = [&]() {
#pragma unroll
        for (int c = 0; c < EPL; c++) {
            u32x4n o;
            float s = 0.0f;
#pragma unroll
            for (int j = 0; j < 8; j += 2) {
                if constexpr (IN16) {
                    const _Float16 h0 = __builtin_bit_cast(half8n, x[j])[c], h1 = __builtin_bit_cast(half8n, x[j + 1])[c];
                    const float f0 = (float)h0, f1 = (float)h1;
                    s = s + f0 * f0;
                    s = s + f1 * f1;
                    const half2v p = {h0, h1};
                    o[j / 2] = __builtin_bit_cast(uint32_t, p);
                } else {
                    o[j / 2] = cvt_pack2(__builtin_bit_cast(f32x4, x[j])[c], __builtin_bit_cast(f32x4, x[j + 1])[c], s);
                }
            }
            *reinterpret_cast<u32x4n *>(s_pack + t * TS + g * QS + vpos(cin + c, IN16) * 16) = o;
            s_chunk[t * CH + (cin + c) * PITCH + g] = s;
            seen += s;
        }
    };
    // one operand role
    auto emit = [&](bool as_b, void *pk, float *nmo, float *nmTo) {
        const bool prune = tau_skip > 0.0f;
        seen = 0.0f;
        if (as_b) stage_b(); else stage_a();
        const bool used = __ballot(seen != 0.0f) != 0ull;
        if (lane == 0) s_seen[wave] = used;
        __syncthreads();
        // norms in the canonical order: lane n of a wave ends up with its n-th tile's
        const int t0 = wave * NT;
        auto norms = [&]() {
            if (t0 >= TPP) return;
            float nv = 0.0f;
#pragma unroll
            for (int n = 0; n < NT; n++) {
                float partial = 0.0f;
#pragma unroll
                for (int it = 0; it < STEPS; it++) {
                    const int c = it * 64 + lane;
                    partial = partial + s_chunk[(t0 + n) * CH + (c / QN) * PITCH + (c % QN)];
                }
                partial = butterfly64_dpp(partial);
                nv = lane == n ? partial : nv;
            }
            nv = sqrtf(nv);
            const uint32_t Jt = J0 + t0 + lane;
            if (lane < NT && Jt < nbc) {
                nmo[(uint64_t)I * nbc + Jt] = nv;
                if (as_b) nmTo[(uint64_t)Jt * nbr + I] = nv;
                if (prune) s_skip[t0 + lane] = rowmax != nullptr ? nv * rowmax[Jt] < tau_skip : nv == 0.0f;
            }
        };
        // (what is stored where, and for a tau-aware pass what is left out: as in normmap_strip)
        if (prune) {
            norms();
            __syncthreads();
        }
        int any = 0;
#pragma unroll
        for (int w = 0; w < NWV; w++) any |= s_seen[w];
        const uint32_t step = as_b ? nbr * TB : TB;    // bytes from a tile to the next of the strip (all of them: less than 2 GiB)
        const uint64_t first = as_b ? (uint64_t)J0 * nbr + I : (uint64_t)I * nbc + J0;
        const __amdgpu_buffer_rsrc_t out = __builtin_amdgcn_make_buffer_rsrc(static_cast<unsigned char *>(pk) + first * TB, 0, 0x7fffffff, 0x00020000);
        auto copy = [&](auto cached) {
#pragma unroll
            for (int i = 0; i < TPP * VPT / (64 * NWV); i++) {
                const int vi = threadIdx.x + 64 * NWV * i, tt = vi / VPT, iv = vi % VPT;
                const u32x4n d = *reinterpret_cast<const u32x4n *>(s_pack + tt * TS + (iv / B) * QS + vpos(iv % B, IN16 && as_b) * 16);
                uint32_t at = (uint32_t)tt * step + (uint32_t)iv * 16u;
                at = J0 + tt < nbc && !(prune && s_skip[tt]) ? at : NOWHERE;
                __builtin_amdgcn_raw_buffer_store_b128(d, out, (int)at, 0, decltype(cached)::value ? 16 : 2);      // sc1, or non-temporal
            }
        };
        if (keep_copy && __builtin_amdgcn_readfirstlane(any)) copy(std::true_type{});
        else copy(std::false_type{});
        if (!prune) norms();
    };
    if constexpr (ROLE != 1) emit(false, packed, nm, nullptr);
    if constexpr (ROLE == 1) emit(true, packed, nm, nmT);
    if constexpr (ROLE == 2) {
        __syncthreads();
        emit(true, packed2, nm2, nmT);
    }
}

template <int B, int ROLE, int SW, bool IN16, int NWV, bool KEEP>
__global__ __launch_bounds__(64 * NWV) void k_normmap_lean(const void *X, uint32_t cols, uint32_t nbr, uint32_t nbc, uint32_t nstrip,
                                                            uint32_t rec, void *packed, float *nm, float *nmT, void *packed2, float *nm2,
                                                            const float *rowmax, float tau_skip, bool keep_copy) {
    using L = NormCfg<B, SW, 1>;
    __shared__ __attribute__((aligned(16))) unsigned char s_pack[L::TPP * L::TS];
    __shared__ float s_chunk[L::TPP * L::CH];
    __shared__ int s_skip[L::TPP], s_seen[NWV];
    asm volatile("" : "+s"(X), "+s"(packed), "+s"(nm), "+s"(nmT), "+s"(tau_skip));        // (all arguments at once)
    normmap_strip_lean<B, ROLE, SW, IN16, NWV, KEEP>(X, cols, nbr, nbc, nstrip, rec, packed, nm, nmT, packed2, nm2, rowmax, tau_skip, keep_copy,
                                                blockIdx.x, s_pack, s_chunk, s_skip, s_seen);
}

template <int B, int SW, bool IN16, int NWV, bool KEEP>
__global__ __launch_bounds__(64 * NWV) void k_normmap_pair_lean(const void *A, const void *Bm, uint32_t nbM, uint32_t nbK, uint32_t nbN,
                                                                 uint32_t n_b, uint32_t strips_a, uint32_t rec_a, uint32_t strips_b,
                                                                 uint32_t rec_b, void *packedA, void *packedB, float *nmA, float *nmB,
                                                                 float *nmBt, float tau_skip, bool keep_copy) {
    using L = NormCfg<B, SW, 1>;
    __shared__ __attribute__((aligned(16))) unsigned char s_pack[L::TPP * L::TS];
    __shared__ float s_chunk[L::TPP * L::CH];
    __shared__ int s_skip[L::TPP], s_seen[NWV];
    asm volatile("" : "+s"(A), "+s"(Bm), "+s"(packedA), "+s"(packedB), "+s"(nmA), "+s"(nmB), "+s"(nmBt), "+s"(tau_skip));
    if (blockIdx.x < n_b)
        normmap_strip_lean<B, 1, SW, IN16, NWV, KEEP>(Bm, nbN * B, nbK, nbN, strips_b, rec_b, packedB, nmB, nmBt, nullptr, nullptr, nullptr, tau_skip,
                                                 keep_copy, blockIdx.x, s_pack, s_chunk, s_skip, s_seen);
    else
        normmap_strip_lean<B, 0, SW, IN16, NWV, KEEP>(A, nbK * B, nbM, nbK, strips_a, rec_a, packedA, nmA, nullptr, nullptr, nullptr, nullptr, tau_skip,
                                                 keep_copy, blockIdx.x - n_b, s_pack, s_chunk, s_skip, s_seen);
}

// rowmax[k] = max_j nB[k, j] (nB row-major [nbK x nbN]); one wave per row.  NaNs are ignored:
// a NaN product is never kept.
__global__ __launch_bounds__(256) void k_rowmax(const float *__restrict__ nB, int64_t nbK, int64_t nbN,
                                                float *__restrict__ rowmax) {
    const int lane = threadIdx.x & 63;
    const int64_t k = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (k >= nbK) return;
    float m = 0.0f;
    for (int64_t j = lane; j < nbN; j += 64) m = fmaxf(m, nB[k * nbN + j]);
#pragma unroll
    for (int s = 1; s < 64; s <<= 1) m = fmaxf(m, __shfl_xor(m, s, 64));
    if (lane == 0) rowmax[k] = m;
}

// ------------------------------------------------------------- utilities
// Packed fp16 -> row-major fp16 bit patterns (read-back helper, not on the
// hot path).  One thread per 16-byte vector.
__global__ void k_unpack(const uint4 *__restrict__ packed, int64_t rows, int64_t cols, int B,
                         int role, uint16_t *__restrict__ out) {
    const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t nvec = rows * cols / 8;
    if (v >= nvec) return;
    const int64_t vpt = (int64_t)B * B / 8;
    const int64_t tile = v / vpt;
    const int iv = (int)(v % vpt);
    const int kg = iv / B, r = iv % B;
    const uint4 d = packed[v];
    const uint32_t wds[4] = {d.x, d.y, d.z, d.w};
    if (role == 0) {
        const int64_t nbK = cols / B;
        const int64_t I = tile / nbK, Kt = tile % nbK;
        uint16_t *o = out + (I * B + r) * cols + Kt * B + kg * 8;
        for (int e = 0; e < 8; e++) o[e] = (uint16_t)(wds[e >> 1] >> ((e & 1) * 16));
    } else {
        const int64_t nbK = rows / B;
        const int64_t J = tile / nbK, Kt = tile % nbK;
        for (int e = 0; e < 8; e++)
            out[(Kt * B + kg * 8 + e) * cols + J * B + r] =
                (uint16_t)(wds[e >> 1] >> ((e & 1) * 16));
    }
}

__global__ void k_transpose_nm(const float *__restrict__ nB, int64_t nbK, int64_t nbN,
                               float *__restrict__ nBt) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nbK * nbN) return;
    const int64_t k = i / nbN, j = i % nbN;
    nBt[j * nbK + k] = nB[i];
}

// Synthetic inputs (tool.cu:370-436 plus a seeded uniform factor): the hash
// and the single fp32 multiply are the same integer / IEEE operations as in
// the host checker, so device and host inputs are bit-identical.
__device__ __forceinline__ float hash_uniform(uint64_t seed, uint64_t idx) {
    uint64_t z = idx + seed * 0x9E3779B97F4A7C15ull + 0x632BE59BD9B4E019ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z ^= z >> 31;
    const uint32_t k = (uint32_t)(z >> 40);
    return (float)k * 1.1920928955078125e-07f - 1.0f;
}

__global__ __launch_bounds__(256) void k_fill_decay(float *__restrict__ X, int64_t rows,
                                                    int64_t cols, const float *__restrict__ table,
                                                    uint64_t seed, int random) {
    const int64_t n4 = rows * cols / 4;
    for (int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v < n4;
         v += (int64_t)gridDim.x * blockDim.x) {
        const int64_t e0 = v * 4;
        const int64_t i = e0 / cols, j0 = e0 % cols;
        float o[4];
#pragma unroll
        for (int c = 0; c < 4; c++) {
            const int64_t j = j0 + c;
            const int64_t d = i > j ? i - j : j - i;
            const float u = random ? hash_uniform(seed, (uint64_t)(e0 + c)) : 1.0f;
            o[c] = u * table[d];
        }
        reinterpret_cast<float4 *>(X)[v] = make_float4(o[0], o[1], o[2], o[3]);
    }
}

// ---------------------------------------------------------------- launchers
constexpr unsigned NARROW_STRIPS = 512;     // of 256 columns, in a launch: two per CU

// Which of a pass's accesses leave their lines in the 256 MB memory-side cache.  Whole calls on three sets of operands and
// workspaces in turn, on one stream, so that nothing of a call is there when the set comes round again; bands, 10 % kept.
// Copies, written through (sc1) instead of non-temporally up to 448 MiB an operand: the multiply reads them, or what of them
// still lies there, from that cache.  1056 x 1568 x 1312 13.2 -> 12.3 us, 2048^3 19.4 -> 18.2, 3072^3 43.6 -> 37.6, 4096^3 71 -> 59,
// 6144^3 168 -> 157, 7168^3 225 -> 202, dense 8192^3 884 -> 865, 10240^3 492 -> 459, 12288^3 703 -> 673; fp16 4096^3 61 -> 50,
// 8192^3 224 -> 209, 10048^3 402 -> 371, 14336^3 876 -> 844; A = B 4096^2 63 -> 51, 7168^2 192 -> 171, 9216^2 320 -> 297.  Beyond, the
// copies drive each other out: 16384^3 1309 -> 1297, tau-aware 1206 -> 1213; 20032^3 2195 -> 2210, tau-aware 2013 -> 2012.
// Strips of nothing but zeros, most of a narrow band's operands, are written past it all the same: left out of that rule, and
// then with it, by the strips before the lean ones, 8192^3 of a band 278 -> 276 -> 261, A = B 235 -> 237 to 246 -> 224, 9216^2 332 -> 317 -> 309.
// Input, by ordinary loads up to 32 MiB a launch: a producer's output of that size may be there.  2048^3 19.4 -> 18.2, fp16
// 16.8 -> 15.4, 1056 x 1568 x 1312 13.1 -> 12.2; beyond it takes the copies' place (4096^3 58.8 -> 61.3, 6144^3 157 -> 163, 7168^3 203 ->
// 226, 8192^3 248 -> 267; fp16 4096^3 49.4 -> 48.6, 8192^3 208 -> 217).
constexpr int64_t KEEP_INPUT_MAX = 32ll << 20, KEEP_COPY_MAX = 448ll << 20;
static bool keep_input(int64_t bytes) { return bytes <= KEEP_INPUT_MAX; }
static bool keep_copy(int64_t bytes) { return bytes <= KEEP_COPY_MAX; }

// The lean strips' buffer loads are of whole 32-bit words.  (Rows are multiples of 64 bytes: where the first begins decides.  Floats always do.)
static bool whole_words(const void *X) { return ((uintptr_t)X & 3u) == 0; }

template <int ROLE, bool IN16>
static hipError_t launch_normmap(const void *X, int64_t rows, int64_t cols, int tile, void *packed, float *nm,
                                 float *nmT, hipStream_t s, void *packed2 = nullptr, float *nm2 = nullptr,
                                 const float *rowmax = nullptr, float tau_skip = 0.0f) {
    const int64_t nbr = rows / tile, nbc = cols / tile;
    const bool keep = keep_input(rows * cols * (IN16 ? 2 : 4)), words = !IN16 || whole_words(X);
    const auto strips = [&](int64_t sw) { return (unsigned)(nbr * ((cols + sw - 1) / sw)); };
#define SPAMM_NORMMAP(T, SW, PH, NWV)                                                                                              \
    k_normmap<T, ROLE, SW, IN16, PH, NWV><<<strips(SW), 64 * NWV, 0, s>>>(X, cols, cols, nbr, nbc, (cols + SW - 1) / SW, (uint4 *)packed, \
                                                                          nm, nmT, (uint4 *)packed2, nm2, rowmax, tau_skip,        \
                                                                          keep_copy(rows * cols * 2))
#define SPAMM_LEAN_(T, SW, NWV, KEEP)                                                                                                     \
    do {                                                                                                                                  \
        const uint32_t ns = (uint32_t)((cols + SW - 1) / SW);                                                                             \
        k_normmap_lean<T, ROLE, SW, IN16, NWV, KEEP><<<strips(SW), 64 * NWV, 0, s>>>(                                                     \
            X, (uint32_t)cols, (uint32_t)nbr, (uint32_t)nbc, ns, strip_reciprocal(strips(SW), ns), packed, nm, nmT, packed2, nm2, rowmax, \
            tau_skip, keep_copy(rows * cols * 2));                                                                                        \
    } while (0)
#define SPAMM_LEAN(T, SW, NWV)                            \
    do {                                                  \
        if (keep && words) SPAMM_LEAN_(T, SW, NWV, true); \
        else if (words) SPAMM_LEAN_(T, SW, NWV, false);   \
        else if constexpr (IN16) SPAMM_NORMMAP(T, SW, 1, NWV); \
    } while (0)
#define SPAMM_LEAN_IF_KEPT(T, SW, NWV)                    \
    do {                                                  \
        if (keep && words) SPAMM_LEAN_(T, SW, NWV, true); \
        else SPAMM_NORMMAP(T, SW, 1, NWV);                \
    } while (0)
    // strip widths and waves: one 8-row group per lane, at most ~42 KiB of LDS and so three workgroups or more per CU.
    // fp16 input: 256 columns, two rows per load (512 in phases before: tile 64 1024^2, both passes, 6.2 -> 4.1 us, 4096^2
    // 28.4 -> 26.3, 16384^2 A = B 303 -> 291; tile 32 2048^2 8.0 -> 7.3, 8192^2 tau-aware 93 -> 87).
    switch (tile) {
        case 32:
            if constexpr (IN16) SPAMM_LEAN(32, 256, 2);
            else SPAMM_LEAN(32, 256, 4);
            break;
        case 64:
            // fp32 input: strips of 128 columns where there are few (1024^2, both passes: 5.4 -> 4.4 us; 4096^2 36.1 ->
            // 36.7), of 256 by eight waves on middling grids (N = 8192: 0.066 / 0.058 -> 0.063 / 0.056 ms), by four waves,
            // two groups per lane, on large ones (N = 16384: as fast or 1 % faster; against the lean strip by eight waves both 2 to 4 % slower
            // in plain passes of 16384^2, even at 12032^2, 2 % faster at 20032^2 and 5 % in tau-aware squares of a narrow band)
            // fp16 input, 3 to 4 strips of 256 columns per CU (of a whole chip), of which three run at once: strips of 512 in
            // two phases by eight waves are one turn instead of two.  256 -> 512, A and B pass alone, A = B with the fill of C
            // behind it: 4096^2 12.5 -> 11.1 us, 12.8 -> 11.6, 42.1 -> 39.1; 3840^2 11.2 -> 10.5, 11.1 -> 10.9, 39.7 -> 37.5;
            // 3648^2 10.5 -> 10.1, 10.3 -> 10.5, 38.4 -> 36.4; 3584^2 8.9 -> 9.1, 9.5 -> 9.9, 37.0 -> 35.8
            if constexpr (IN16) {
                if (strips(256) > 768u && strips(256) <= 1024u) SPAMM_NORMMAP(64, 512, 2, 8);
                else SPAMM_LEAN_IF_KEPT(64, 256, 4);
            } else if (strips(256) <= NARROW_STRIPS) SPAMM_LEAN(64, 128, 4);
            else if (strips(256) <= 8192u) SPAMM_LEAN(64, 256, 8);
            else SPAMM_NORMMAP(64, 256, 1, 4);
            break;
        // tile 128: strips of one tile.  Only the fp32 B role of a large matrix keeps strips of two tiles in two phases by
        // four waves: N = 32768 830 against 867 us, 16384 225 / 231, 12800 159 / 158, 8192 72 / 67.
        case 128:
            if constexpr (IN16) {
                if constexpr (ROLE == 2) return hipErrorInvalidValue;      // (two passes, or the pair, are faster)
                else SPAMM_LEAN_IF_KEPT(128, 128, 4);
            } else {
                if constexpr (ROLE == 1)
                    if (strips(256) > 6000u) {
                        SPAMM_NORMMAP(128, 256, 2, 4);
                        break;
                    }
                SPAMM_LEAN_IF_KEPT(128, 128, 8);
            }
            break;
        default: return hipErrorInvalidValue;
    }
#undef SPAMM_LEAN_IF_KEPT
#undef SPAMM_LEAN
#undef SPAMM_LEAN_
#undef SPAMM_NORMMAP
    return hipGetLastError();
}

hipError_t launch_normmap_a(const void *X, bool in16, int64_t rows, int64_t cols, int tile, void *packed,
                            float *nm, const float *rowmax, float tau_skip, hipStream_t s) {
    return in16 ? launch_normmap<0, true>(X, rows, cols, tile, packed, nm, nullptr, s, nullptr, nullptr, rowmax, tau_skip)
                : launch_normmap<0, false>(X, rows, cols, tile, packed, nm, nullptr, s, nullptr, nullptr, rowmax, tau_skip);
}

template <int B, int SW, int PH, int NWV, bool IN16>
static void launch_pair(const void *A, const void *Bm, int64_t nbM, int64_t nbK, int64_t nbN, void *packedA, void *packedB,
                        float *nmA, float *nmB, float *nmBt, float tau_skip, hipStream_t s) {
    const int64_t strips_a = (nbK * B + SW - 1) / SW, strips_b = (nbN * B + SW - 1) / SW;
    const unsigned n_b = (unsigned)(nbK * strips_b), n_a = (unsigned)(nbM * strips_a);
    const int64_t a = nbM * nbK * B * B, b = nbK * nbN * B * B;
    const bool keep = keep_input((a + b) * (IN16 ? 2 : 4)), words = !IN16 || (whole_words(A) && whole_words(Bm));
    const bool cached = keep_copy(2 * (a > b ? a : b));
    auto lean = [&](auto kept) {
        k_normmap_pair_lean<B, SW, IN16, NWV, decltype(kept)::value><<<n_a + n_b, 64 * NWV, 0, s>>>(
            A, Bm, (uint32_t)nbM, (uint32_t)nbK, (uint32_t)nbN, n_b, (uint32_t)strips_a, strip_reciprocal(n_a, (uint32_t)strips_a),
            (uint32_t)strips_b, strip_reciprocal(n_b, (uint32_t)strips_b), packedA, packedB, nmA, nmB, nmBt, tau_skip, cached);
    };
    auto streaming = [&](auto) {                                   // (a kernel only where it is called)
        k_normmap_pair<B, SW, IN16, PH, NWV><<<n_a + n_b, 64 * NWV, 0, s>>>(A, Bm, nbM, nbK, nbN, n_b, strips_a, strips_b, (uint4 *)packedA,
                                                                            (uint4 *)packedB, nmA, nmB, nmBt, tau_skip, cached);
    };
    if (keep && words) lean(std::true_type{});
    else if constexpr (B == 32 || (B == 64 && !IN16)) {            // (as launch_normmap)
        if (words) lean(std::false_type{});
        else if constexpr (IN16) streaming(0);
    } else streaming(0);
}

// Where the two passes are worth running as one, by the strips of both operands, counted as tile rows of 1 KiB (256
// columns of floats, 512 of halves, whatever width the passes take).  Whole multiplies, two passes -> one:
// 256^3 14.6 -> 10.7 us, 2048^3 28.3 -> 23.9, 4096^3 87.2 -> 83.9, 6144^3 184 -> 182, 8192^3 912.5 -> 909.5; tile 64
// beyond that runs four waves per workgroup in passes of their own.  A tau-aware A pass of its own (behind k_rowmax)
// writes less: 3 us less at 4096^3, where the second launch and k_rowmax cost 8, and 13 us less at 8192^3.
bool normmap_pair_fits(bool in16, bool tau_aware, int64_t M, int64_t K, int64_t N, int tile) {
    const int64_t sw = in16 ? 512 : 256;
    const int64_t strips = (M / tile) * ((K + sw - 1) / sw) + (K / tile) * ((N + sw - 1) / sw);
    return strips <= (tau_aware ? 4096 : 16384);
}

hipError_t launch_normmap_pair(const void *A, const void *Bm, bool in16, int64_t M, int64_t K, int64_t N, int tile, void *packedA,
                               float *nmA, void *packedB, float *nmB, float *nmBt, float tau_skip, hipStream_t s) {
    const int64_t nbM = M / tile, nbK = K / tile, nbN = N / tile;
#define SPAMM_PAIR(T, SW, NWV, IN16) \
    launch_pair<T, SW, 1, NWV, IN16>(A, Bm, nbM, nbK, nbN, packedA, packedB, nmA, nmB, nmBt, tau_skip, s)
    // (strips as the passes of their own have them)
    switch (tile) {
        case 32:
            if (in16) SPAMM_PAIR(32, 256, 2, true);
            else SPAMM_PAIR(32, 256, 4, false);
            break;
        case 64:
            if (in16) SPAMM_PAIR(64, 256, 4, true);
            else if (nbM * ((K + 255) / 256) + nbK * ((N + 255) / 256) <= NARROW_STRIPS) SPAMM_PAIR(64, 128, 4, false);
            else SPAMM_PAIR(64, 256, 8, false);
            break;
        case 128:
            if (in16) SPAMM_PAIR(128, 128, 4, true);
            else SPAMM_PAIR(128, 128, 8, false);
            break;
        default: return hipErrorInvalidValue;
    }
#undef SPAMM_PAIR
    return hipGetLastError();
}

hipError_t launch_rowmax(const float *nB, int64_t nbK, int64_t nbN, float *rowmax, hipStream_t s) {
    k_rowmax<<<(unsigned)((nbK + 3) / 4), 256, 0, s>>>(nB, nbK, nbN, rowmax);
    return hipGetLastError();
}

hipError_t launch_normmap_ab(const void *X, bool in16, int64_t n, int tile, void *packedA, float *nmA,
                             void *packedB, float *nmB, float *nmBt, float tau_skip, hipStream_t s) {
    return in16 ? launch_normmap<2, true>(X, n, n, tile, packedA, nmA, nmBt, s, packedB, nmB, nullptr, tau_skip)
                : launch_normmap<2, false>(X, n, n, tile, packedA, nmA, nmBt, s, packedB, nmB, nullptr, tau_skip);
}

hipError_t launch_normmap_b(const void *X, bool in16, int64_t rows, int64_t cols, int tile, void *packed,
                            float *nm, float *nmT, float tau_skip, hipStream_t s) {
    return in16 ? launch_normmap<1, true>(X, rows, cols, tile, packed, nm, nmT, s, nullptr, nullptr, nullptr, tau_skip)
                : launch_normmap<1, false>(X, rows, cols, tile, packed, nm, nmT, s, nullptr, nullptr, nullptr, tau_skip);
}

hipError_t launch_unpack(const void *packed, int64_t rows, int64_t cols, int tile, int role,
                         uint16_t *out, hipStream_t s) {
    const int64_t nvec = rows * cols / 8;
    k_unpack<<<(unsigned)((nvec + 255) / 256), 256, 0, s>>>((const uint4 *)packed, rows, cols, tile,
                                                            role, out);
    return hipGetLastError();
}

hipError_t launch_transpose_normmap(const float *nB, int64_t nbK, int64_t nbN, float *nBt,
                                    hipStream_t s) {
    const int64_t n = nbK * nbN;
    k_transpose_nm<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(nB, nbK, nbN, nBt);
    return hipGetLastError();
}

hipError_t launch_fill_decay(float *X, int64_t rows, int64_t cols, const float *table,
                             uint64_t seed, int random, hipStream_t s) {
    const int64_t n4 = rows * cols / 4;
    int64_t blocks = (n4 + 255) / 256;
    if (blocks > 65536) blocks = 65536;
    k_fill_decay<<<(unsigned)blocks, 256, 0, s>>>(X, rows, cols, table, seed, random);
    return hipGetLastError();
}

}  // namespace spamm
