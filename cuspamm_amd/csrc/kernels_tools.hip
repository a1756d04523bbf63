// Error-report tooling around the multiply (not on the hot path).
//
// The reference compares SpAMM against a dense cuBLAS product and prints
// ||C_dense - C_spamm||_F, ||C_dense||_F, ||C_spamm||_F (check_simple_gpu,
// tool.cu:227-280; COUNTERRTRANS, tool.cu:6-24).  Here the dense product is
// the product of the same fp16 operands, formed block by block and reduced on the
// fly (it is never stored): exactly, in whole numbers on the 8-bit integer matrix
// pipeline (k_limbs, k_error_limbs), or on the fp64 one (k_error_dense,
// v_mfma_f64_16x16x4_f64) where values are too large for that, K is too long, the
// planes too big or the product too small.  Next to it the tau-derived bound
// sqrt(sum_ij (sum_{k dropped} nA[i,k]*nB[k,j])^2).
//
// What bounds k_error_dense: the fp64 matrix pipeline (128 operations per clock and CU) and the VALU's
// conversions beside it -- fp16 to fp64 is two instructions per value, one of them at a
// quarter of the rate, and they take the place of MFMAs.  So a wave's block of C is as large as
// the number of blocks allows: each converted value serves NBR or NBC MFMAs.  4096^3:
// 2229 us with 32 x 32 per wave and 4-byte loads, 2109 now (65 TFLOP/s; the pipeline's 128 operations at the clock
// that the chip holds under them, about 2 GHz); 1984 x 2176 x 768: 196 -> 158.  In whole numbers instead (one call, its
// host wait included): 4096^3 2046 -> 661 us on uniform values in [-1, 1) (4 bytes each, 16 products, 3.3 Pop/s),
// 444 where 3 bytes do, 203 on exp(-d / 100); 1984 x 768 x 2176 151 -> 72, 60, 54; 64 rows of 4096^3 186 -> 86, 68, 45.
// An operand with a value of 127 or more has been read by k_limbs for nothing, which writes no planes then, and blocks of 64 x 64
// of C are formed in fp64 by k_error_limbs itself, two workgroups per CU where k_error_dense has three, so its loads go out
// three steps ahead instead of one (1088^3 107 -> 98 us, 1536 x 1024 x 1024 107 -> 97, 1280^3 123 -> 117 to 122).  Against a report that
// is never split: 1024^3 55 -> 58, 1280^3 102 -> 117 to 122, 4096^3, by k_error_dense behind it, 2046 -> 2092.
// The scalar bound of 64 x 64 x 64 tiles 52 -> 7 us, the per-tile one 51 -> 4; results go straight to host memory (a
// clearing launch before and a copy after each were 25 us a call).
#include "gemm_device.h"
#include "reduce_device.h"

namespace spamm {

typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef _Float16 half8t __attribute__((ext_vector_type(8)));

// Stores to one address queue (32768 waves that all found such values took 0.6 ms): a workgroup sets one of 16 flags, unless
// it finds it set, and who set that first the one that is read.
constexpr int RANGE_FLAGS = 16;
struct alignas(128) RangeFlag {
    unsigned long long call;
};

struct ReportWorkspace {
    Tickets tickets;                    // workgroups of the running launch that have finished; zero between launches
    RangeFlag range[1 + RANGE_FLAGS];   // k_limbs: the last call of which an operand held values without limbs
    double part[1];                     // per workgroup: its sums (report_workspace_bytes says how many)
};

// Whether an operand of this call held values that k_limbs has no limbs for.  (By the call's number: the flags need not be
// put back.)
__device__ __forceinline__ bool out_of_range(const ReportWorkspace *ws, unsigned long long call) {
    return ws->range[0].call == call;
}

// Sums of all workgroups' N values, by the workgroup that finishes last, to host_out (pinned host memory): in a
// fixed order, so that a repeated call gives the same number.  `own`: the workgroup's values, in thread i the i-th.
template <int N>
__device__ __forceinline__ void finish_sums(ReportWorkspace *ws, double own, ReportSums *host_out, unsigned long long *host_seq,
                                            unsigned long long seq) {
    __shared__ double s_fin[4][N];
    if (threadIdx.x < N)
        agent_store(reinterpret_cast<unsigned long long *>(&ws->part[(size_t)blockIdx.x * N + threadIdx.x]), __builtin_bit_cast(unsigned long long, own));
    if (!last_workgroup(&ws->tickets)) return;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    double v[N];
#pragma unroll
    for (int i = 0; i < N; i++) v[i] = 0.0;
#pragma unroll 4
    for (unsigned b = threadIdx.x; b < gridDim.x; b += 256)
#pragma unroll
        for (int i = 0; i < N; i++)
            v[i] += __builtin_bit_cast(double, agent_load(reinterpret_cast<unsigned long long *>(&ws->part[(size_t)b * N + i])));
#pragma unroll
    for (int i = 0; i < N; i++) {
        for (int off = 32; off > 0; off >>= 1) v[i] += __shfl_down(v[i], off, 64);
        if (lane == 0) s_fin[wave][i] = v[i];
    }
    __syncthreads();
    if (threadIdx.x != 0) return;
    ReportSums out = {};
#pragma unroll
    for (int i = 0; i < N; i++) out.v[i] = s_fin[0][i] + s_fin[1][i] + s_fin[2][i] + s_fin[3][i];
    publish_result(host_out, out, host_seq, seq);
}

// A wave owns NBR x NBC blocks of v_mfma_f64_16x16x4_f64 (4 accumulator doubles per lane each), four waves (2 x 2) a
// workgroup.  Operands come straight from the packed fp16 copies: a packed 16-byte vector holds 8 consecutive k of one
// row (A) / column (B); of every four k-groups lane group q = lane / 16 takes the q-th, one 16-byte load per lane and
// operand block for 32 k, and element e of the vectors makes MFMA step e.  Which k goes to which step is the same for A
// and B, and the sum over k does not care.  fp16 -> fp64 is exact.
template <int NBR, int NBC, int DEPTH = 2>
__device__ __forceinline__ void dense_block(const _Float16 *__restrict__ pA, const _Float16 *__restrict__ pB, int64_t K, int64_t N, int tile,
                                            const float *__restrict__ C, int64_t br, int64_t bc, double &e2, double &d2, double &c2) {
    const int lane = threadIdx.x & 63, l16 = lane & 15, q = lane >> 4;
    const int64_t nbK = K / tile, tile_halves = (int64_t)tile * tile;
    const _Float16 *srcA[NBR], *srcB[NBC];
#pragma unroll
    for (int t = 0; t < NBR; t++) {
        const int64_t r = br + t * 16 + l16;
        srcA[t] = pA + (r / tile) * nbK * tile_halves + (r % tile) * 8 + (int64_t)q * tile * 8;
    }
#pragma unroll
    for (int t = 0; t < NBC; t++) {
        const int64_t c = bc + t * 16 + l16;
        srcB[t] = pB + (c / tile) * nbK * tile_halves + (c % tile) * 8 + (int64_t)q * tile * 8;
    }
    f64x4 acc[NBR][NBC];
#pragma unroll
    for (int a = 0; a < NBR; a++)
#pragma unroll
        for (int b = 0; b < NBC; b++) acc[a][b] = f64x4{0.0, 0.0, 0.0, 0.0};
    struct Vecs {
        half8t a[NBR], b[NBC];
    };
    // four k-groups are 32 * tile halves, and a tile's are followed by the next k tile's
    const int64_t steps = K / 32, stride = (int64_t)32 * tile;
    auto load = [&](Vecs &v, int64_t s) {
        const int64_t off = (s < steps ? s : steps - 1) * stride;
#pragma unroll
        for (int t = 0; t < NBR; t++) v.a[t] = *reinterpret_cast<const half8t *>(srcA[t] + off);
#pragma unroll
        for (int t = 0; t < NBC; t++) v.b[t] = *reinterpret_cast<const half8t *>(srcB[t] + off);
    };
    auto multiply = [&](const Vecs &v) {
#pragma unroll
        for (int e = 0; e < 8; e++) {
            double a[NBR], b[NBC];
#pragma unroll
            for (int t = 0; t < NBR; t++) a[t] = (double)(float)v.a[t][e];
#pragma unroll
            for (int t = 0; t < NBC; t++) b[t] = (double)(float)v.b[t][e];
#pragma unroll
            for (int ta = 0; ta < NBR; ta++)
#pragma unroll
                for (int tb = 0; tb < NBC; tb++)
                    acc[ta][tb] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[ta], b[tb], acc[ta][tb], 0, 0, 0);
        }
    };
    Vecs v[DEPTH];                          // steps whose loads are under way or done
#pragma unroll
    for (int i = 0; i < DEPTH - 1; i++) load(v[i], i);
    int64_t s = 0;
    for (; s + DEPTH <= steps; s += DEPTH)
#pragma unroll
        for (int i = 0; i < DEPTH; i++) {
            load(v[(i + DEPTH - 1) % DEPTH], s + i + DEPTH - 1);
            multiply(v[i]);
        }
#pragma unroll
    for (int i = 0; i < DEPTH - 1; i++)
        if (s + i < steps) multiply(v[i]);
    // accumulator i of lane l in block (ta, tb): row 4 i + l / 16, column l % 16
#pragma unroll
    for (int ta = 0; ta < NBR; ta++)
#pragma unroll
        for (int tb = 0; tb < NBC; tb++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const double c = (double)C[(br + ta * 16 + 4 * i + q) * N + bc + tb * 16 + l16];
                const double d = acc[ta][tb][i];
                e2 += (c - d) * (c - d);
                d2 += d * d;
                c2 += c * c;
            }
}

template <int NBR, int NBC>
__global__ __launch_bounds__(256, NBR * NBC > 8 ? 2 : 3) void k_error_dense(const _Float16 *__restrict__ pA, const _Float16 *__restrict__ pB,
                                                                        int64_t K, int64_t N, int tile, const float *__restrict__ C,
                                                                        int64_t row0, int64_t row1, int nwg_n,
                                                                        ReportWorkspace *__restrict__ ws, ReportSums *__restrict__ host_out,
                                                                        unsigned long long *__restrict__ host_seq, unsigned long long seq) {
    __shared__ double red[4][3];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wr = wave >> 1, wc = wave & 1;
    const int64_t br = row0 + (int64_t)(blockIdx.x / nwg_n) * (NBR * 32) + wr * (NBR * 16);
    const int64_t bc = (int64_t)(blockIdx.x % nwg_n) * (NBC * 32) + wc * (NBC * 16);
    double e2 = 0, d2 = 0, c2 = 0;
    if (br < row1 && bc < N) {              // (whole blocks: rows and columns come in multiples of 64)
        dense_block<NBR, NBC>(pA, pB, K, N, tile, C, br, bc, e2, d2, c2);
        for (int off = 32; off > 0; off >>= 1) {
            e2 += __shfl_down(e2, off, 64);
            d2 += __shfl_down(d2, off, 64);
            c2 += __shfl_down(c2, off, 64);
        }
    }
    if (lane == 0) {
        red[wave][0] = e2;
        red[wave][1] = d2;
        red[wave][2] = c2;
    }
    __syncthreads();
    double own = 0.0;
    if (threadIdx.x < 3) own = red[0][threadIdx.x] + red[1][threadIdx.x] + red[2][threadIdx.x] + red[3][threadIdx.x];
    finish_sums<3>(ws, own, host_out, host_seq, seq);
}

// ---- the dense product in whole numbers ----
//
// Every finite fp16 value is a whole number of 2^-24, so values below 127 in magnitude are four signed bytes
// ("limbs", balanced digits to the base 256) and a product of fp16 matrices is a sum of 8-bit integer products, at
// some thirty times the fp64 pipeline's rate each and exact in 32-bit accumulators: limb i of A times limb j of B
// adds to order i + j.  A block needs only the limbs its largest value reaches (the values of a matrix that decays
// need fewer with every factor of 256, and a block of zeros none), so 0 to 16 products take the place of one.  What the
// fp64 pipeline rounds at every step is exact here up to the last addition.
//
// k_limbs splits the packed copies: per block of 64 rows (columns of B) x 64 k the number of limbs it needs, and that
// many planes of 4 KiB: [limb][16 rows][lane][16 bytes], a lane's 16 bytes an operand of v_mfma_i32_16x16x64_i8
// (lane l: row l % 16, 16 k from l / 16; which k goes where is the same for A and B).
typedef int i32x4 __attribute__((ext_vector_type(4)));
constexpr int LIMB_BLOCK = 64, LIMB_PLANE = LIMB_BLOCK * LIMB_BLOCK, LIMBS = 4;
constexpr float LIMB_MAX = 127.0f;

struct LimbOperand {
    const _Float16 *packed;     // the whole operand's packed copy
    int8_t *planes;             // [block rows][nkb][LIMBS][LIMB_PLANE]
    uint8_t *cls;               // [block rows][nkb]: limbs of the block
    int64_t row0;               // first row (column of B) to be split, a multiple of 64
    int64_t n_blocks;           // blocks of 64 rows, times nkb
};

__global__ __launch_bounds__(256) void k_limbs(LimbOperand a, LimbOperand b, int64_t K, int tile, int nkb, unsigned long long call,
                                               ReportWorkspace *__restrict__ ws) {
    __shared__ unsigned int s_used[4];
    __shared__ bool s_fits[4];
    const bool is_a = (int64_t)blockIdx.x < a.n_blocks;
    const LimbOperand op = is_a ? a : b;
    const int64_t blk = is_a ? blockIdx.x : blockIdx.x - a.n_blocks;
    const int kb = (int)(blk % nkb);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t r = op.row0 + (blk / nkb) * LIMB_BLOCK + wave * 16 + (lane & 15);
    const int64_t k = (int64_t)kb * LIMB_BLOCK + (lane >> 4) * 16;
    half8t h0 = {}, h1 = {};
    if (k < K) {                // (K is a multiple of 32: the last block may end halfway)
        const _Float16 *src = op.packed + ((r / tile) * (K / tile) + k / tile) * ((int64_t)tile * tile) + (k % tile) * tile + (r % tile) * 8;
        h0 = *reinterpret_cast<const half8t *>(src);
        h1 = *reinterpret_cast<const half8t *>(src + (int64_t)tile * 8);
    }
    unsigned int w[16], used = 0;
    bool fits = true;
#pragma unroll
    for (int e = 0; e < 16; e++) {
        const float x = (float)(e < 8 ? h0[e & 7] : h1[e & 7]);
        fits = fits && __builtin_fabsf(x) < LIMB_MAX;                   // (false for a NaN)
        const int v = (int)((__builtin_fabsf(x) < LIMB_MAX ? x : 0.0f) * 16777216.0f);       // exact
        w[e] = ((unsigned int)v + 0x00808080u) ^ 0x00808080u;           // byte i is digit i
        used |= w[e];
    }
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) used |= __shfl_xor(used, off, 64);
    fits = __ballot(!fits) == 0ull;
    if (lane == 0) {
        s_used[wave] = used;
        s_fits[wave] = fits;
    }
    __syncthreads();
    if (!(s_fits[0] && s_fits[1] && s_fits[2] && s_fits[3])) {          // nothing will read the planes
        unsigned long long *flag = &ws->range[1 + blockIdx.x % RANGE_FLAGS].call;
        if (threadIdx.x == 0 && agent_load(flag) != call &&
            __hip_atomic_exchange(flag, call, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != call)
            agent_store(&ws->range[0].call, call);
        return;
    }
    used = s_used[0] | s_used[1] | s_used[2] | s_used[3];
    const int limbs = used == 0 ? 0 : (31 - __builtin_clz(used)) / 8 + 1;
    if (threadIdx.x == 0) op.cls[blk] = (uint8_t)limbs;
    int8_t *out = op.planes + blk * (LIMBS * LIMB_PLANE) + threadIdx.x * 16;
#pragma unroll
    for (int l = 0; l < LIMBS; l++) {
        if (l >= limbs) break;
        i32x4 v;
#pragma unroll
        for (int g = 0; g < 4; g++) {
            // bytes l of four words
            const unsigned int lo = __builtin_amdgcn_perm(w[4 * g + 1], w[4 * g], 0x0c0c0400u + 0x0101u * l);
            const unsigned int hi = __builtin_amdgcn_perm(w[4 * g + 3], w[4 * g + 2], 0x0c0c0400u + 0x0101u * l);
            v[g] = (int)(lo | hi << 16);
        }
        // (written through: the planes are read by every XCD; 1984 x 768 x 2176 46.3 -> 44.9 us, 4096^3 algebraic 219 -> 214)
        asm volatile("global_store_dwordx4 %0, %1, off sc1\n\ts_nop 1" :: "v"(out + l * LIMB_PLANE), "v"(v) : "memory");
    }
}

// One workgroup owns 64 x 64 of C, a wave 32 x 32 of it: 4 accumulator registers x 4 MFMA blocks x 7 orders, so that two
// waves share a SIMD.  The k blocks are sorted by the limbs they need on both sides (whole numbers: the sum does not
// care) and taken in steps of as many blocks of a kind as have LIMB_STEP planes or fewer; each kind has a loop of its own.  A
// step's planes are multiplied from LDS, which two waves share each, while direct global->LDS loads bring the next step's, whatever
// its kind.  (Where a wave loaded its operands to registers, kind by kind, every plane passed the L1 twice and
// a kind, of two or three blocks on the average, began with a wait: kernel alone, 4096^3 exp(-d / 100) 241 -> 201 us, uniform 780 ->
// 670, 4096^3 algebraic 252 -> 187.)  What bounds it, per step of the two
// workgroups of a CU, 4096^3: 0.99 us on exp(-d / 100) (24 steps a workgroup, its fixed costs included), where their MFMAs take 0.4
// and LDS 0.5 (4 KiB written and 8 read per plane), 1.3 us on uniform values (64 steps), where they take 0.9 and 0.7; without the
// reads the calls were 10 % shorter, without the loads 12 %.  Planes in a ring of 16 with loads up to two steps ahead: 6 % longer (addresses); steps of 6 planes by three
// workgroups per CU: decaying values 5 to 10 % shorter, uniform ones 50 % longer (4 + 4 limbs take two steps, and
// 168 registers are too few).
// Groups of GB x GB workgroups that share operands in an L2 run on one XCD; the groups, row by row, go round
// the XCDs, each row turned by two against the one above, so that those of a diagonal, which have much the same work, are
// spread over them.
constexpr int ORDERS = 2 * LIMBS - 1;
constexpr int64_t LIMB_MAX_K = 32768 - 64;      // an order adds up to 4 products of at most 2^14 per k in 31 bits
constexpr int LIMB_MAX_KB = 32768 / LIMB_BLOCK;
constexpr int LIMB_STEP = 2 * LIMBS;            // planes
constexpr int LIMB_MAX_STEPS = LIMB_MAX_KB + LIMBS * LIMBS;

// log2 of the blocks of a kind, (limbs of A - 1) * LIMBS + limbs of B - 1, that a step takes
__host__ __device__ constexpr int limb_per_step(int kind) {
    const int planes = kind / LIMBS + kind % LIMBS + 2;
    return planes == 2 ? 2 : (planes <= 4 ? 1 : 0);
}

// Sum over the wave, in lane 63.
template <int CTRL, int ROWS>
__device__ __forceinline__ double add_dpp(double v) {
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)u, CTRL, ROWS, 0xf, false);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(u >> 32), CTRL, ROWS, 0xf, false);
    return v + __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
}
__device__ __forceinline__ double wave_sum(double v) {
    v = add_dpp<0xB1, 0xf>(v);          // lane ^ 1, lane ^ 2, the other half and the other quarter of 16 lanes
    v = add_dpp<0x4E, 0xf>(v);
    v = add_dpp<0x141, 0xf>(v);
    v = add_dpp<0x140, 0xf>(v);
    v = add_dpp<0x142, 0xa>(v);         // the last lane of 16 to the next 16, of 32 to the next 32
    return add_dpp<0x143, 0xc>(v);
}

__global__ __launch_bounds__(256, 2) void k_error_limbs(const int8_t *__restrict__ plA, const uint8_t *__restrict__ clsA,
                                                        const int8_t *__restrict__ plB, const uint8_t *__restrict__ clsB, int nkb,
                                                        int nbi, int nbj, int gb, int ngj, int n_xcd, const _Float16 *__restrict__ pA,
                                                        const _Float16 *__restrict__ pB, int64_t K, int64_t N, int tile,
                                                        const float *__restrict__ C, int64_t row0, ReportWorkspace *__restrict__ ws,
                                                        ReportSums *__restrict__ host_out, unsigned long long *__restrict__ host_seq,
                                                        unsigned long long seq, bool dense_here) {
    __shared__ __attribute__((aligned(16))) unsigned char s_planes[2][LIMB_STEP][LIMB_PLANE];     // of this step and the next
    __shared__ __attribute__((aligned(16))) uint16_t s_desc[LIMB_MAX_STEPS][LIMB_STEP];           // plane of A or (bit 15) of B, or none
    __shared__ double red[4][3];
    __shared__ int s_count[LIMBS * LIMBS];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wr = wave >> 1, wc = wave & 1;
    const int l16 = lane & 15, q = lane >> 4;
    const int x = (int)blockIdx.x % n_xcd, at = (int)blockIdx.x / n_xcd, in_group = at % (gb * gb), group = at / (gb * gb);
    const int gi = (group * n_xcd + x) / ngj, gj = ((group * n_xcd + x) % ngj + 2 * (ngj - gi % ngj)) % ngj;
    const int bi = gi * gb + in_group / gb, bj = gj * gb + in_group % gb;
    const bool inside = bi < nbi && bj < nbj;
    // (asked for before anything is waited for: the blocks' limbs, which mean nothing in fp64)
    int la[2], lb[2];
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const int kb = h * 256 + (int)threadIdx.x, at = kb < nkb ? kb : 0;
        la[h] = clsA[inside ? (int64_t)bi * nkb + at : 0];
        lb[h] = clsB[inside ? (int64_t)bj * nkb + at : 0];
        if (kb >= nkb) la[h] = 0;
    }
    const bool fp64 = out_of_range(ws, seq);
    if (fp64 && !dense_here) {
        if (blockIdx.x == 0 && threadIdx.x == 0) publish_result(host_out, ReportSums{{-1.0, 0.0, 0.0}}, host_seq, seq);
        return;
    }
    double e2 = 0, d2 = 0, c2 = 0;
    if (inside && fp64) {
        dense_block<2, 2, 4>(pA, pB, K, N, tile, C, row0 + (int64_t)bi * LIMB_BLOCK + wr * 32, (int64_t)bj * LIMB_BLOCK + wc * 32, e2, d2, c2);
    } else if (inside) {
        // ---- k blocks by kind
        constexpr int KINDS = LIMBS * LIMBS;
        constexpr uint32_t NO_PLANE = 0xffffu;
        if (threadIdx.x < KINDS) s_count[threadIdx.x] = 0;
        for (int i = threadIdx.x; i < nkb + KINDS; i += 256) reinterpret_cast<u32x4 *>(s_desc)[i] = u32x4{~0u, ~0u, ~0u, ~0u};
        __syncthreads();
        int kind[2], nth[2];
#pragma unroll
        for (int h = 0; h < 2; h++) {
            kind[h] = la[h] && lb[h] ? (la[h] - 1) * LIMBS + lb[h] - 1 : -1;
            nth[h] = kind[h] >= 0 ? atomicAdd(&s_count[kind[h]], 1) : 0;
        }
        __syncthreads();
        // lane i of every wave: blocks of kind i, and the first step of the kind behind it
        const int blocks = lane < KINDS ? s_count[lane] : 0, per = limb_per_step(lane % KINDS);
        int behind = (blocks + (1 << per) - 1) >> per;
        const int own_steps = behind;
#pragma unroll
        for (int off = 1; off < KINDS; off <<= 1) {
            const int o = __shfl_up(behind, off, 64);
            if (lane >= off) behind += o;
        }
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int at = kind[h] < 0 ? 0 : kind[h], each = limb_per_step(at);
            const int first = __shfl(behind - own_steps, at, 64);
            if (kind[h] < 0) continue;
            uint16_t *d = &s_desc[first + (nth[h] >> each)][(nth[h] & ((1 << each) - 1)) * (la[h] + lb[h])];
            const int plane = (h * 256 + (int)threadIdx.x) * LIMBS;
#pragma unroll
            for (int l = 0; l < LIMBS; l++) {
                if (l < la[h]) d[l] = (uint16_t)(plane + l);
                if (l < lb[h]) d[la[h] + l] = (uint16_t)(0x8000 + plane + l);
            }
        }
        __syncthreads();

        // ---- loads: wave w brings planes w and w + 4 of a step; lane i holds what they are in step 64 n + i
        const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)&s_planes[0][0][0] + wave * LIMB_PLANE;
        const unsigned char *baseA = reinterpret_cast<const unsigned char *>(plA) + (int64_t)bi * nkb * (LIMBS * LIMB_PLANE);
        const unsigned char *baseB = reinterpret_cast<const unsigned char *>(plB) + (int64_t)bj * nkb * (LIMBS * LIMB_PLANE);
        const uint32_t voff = lane * 16;
        uint32_t desc[2] = {NO_PLANE, NO_PLANE};
        int step = 0;                                           // the one whose loads are issued next
        auto issue = [&]() {
            if ((step & 63) == 0) {
                const int s = step + lane;
#pragma unroll
                for (int h = 0; h < 2; h++) desc[h] = s < nkb + KINDS ? s_desc[s][wave + 4 * h] : NO_PLANE;
            }
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const uint32_t d = __builtin_amdgcn_readlane(desc[h], step & 63);
                if (d != NO_PLANE) {
                    const unsigned char *from = (d & 0x8000u ? baseB : baseA) + (int64_t)(d & 0x7fffu) * LIMB_PLANE;
                    const uint32_t to = lds_base + ((step & 1) * LIMB_STEP + 4 * h) * LIMB_PLANE;
                    dma_load<0>(from, voff, to);
                    dma_load<1024>(from, voff, to);
                    dma_load<2048>(from, voff, to);
                    dma_load<3072>(from, voff, to);
                }
            }
            step++;
        };
        issue();
        i32x4 acc[ORDERS][2][2];
#pragma unroll
        for (int o = 0; o < ORDERS; o++)
#pragma unroll
            for (int t = 0; t < 4; t++) acc[o][t >> 1][t & 1] = i32x4{0, 0, 0, 0};
        const unsigned char *vecs = &s_planes[0][0][0] + lane * 16;
        static_for<KINDS>([&](auto kind_) {
            constexpr int LA = decltype(kind_)::value / LIMBS + 1, LB = decltype(kind_)::value % LIMBS + 1;
            constexpr int PER = 1 << limb_per_step(decltype(kind_)::value);
            for (int left = __builtin_amdgcn_readlane(blocks, decltype(kind_)::value); left > 0; left -= PER) {
                __builtin_amdgcn_s_setprio(0);
                __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, 0));
                __syncthreads();       // the step's planes are there for all waves, and all have read the step before
                const unsigned char *half = vecs + (step - 1 & 1) * (LIMB_STEP * LIMB_PLANE);
                issue();
                i32x4 a[PER][LA][2], b[PER][LB][2];
#pragma unroll
                for (int e = 0; e < PER; e++) {
#pragma unroll
                    for (int l = 0; l < LA; l++)
#pragma unroll
                        for (int t = 0; t < 2; t++)
                            a[e][l][t] = *reinterpret_cast<const i32x4 *>(half + (e * (LA + LB) + l) * LIMB_PLANE + (2 * wr + t) * 1024);
#pragma unroll
                    for (int l = 0; l < LB; l++)
#pragma unroll
                        for (int t = 0; t < 2; t++)
                            b[e][l][t] = *reinterpret_cast<const i32x4 *>(half + (e * (LA + LB) + LA + l) * LIMB_PLANE + (2 * wc + t) * 1024);
                }
                __builtin_amdgcn_s_setprio(1);         // (the SIMD's other wave is another workgroup's: 1 %)
#pragma unroll
                for (int e = 0; e < PER; e++) {
                    if (e && left <= e) break;
#pragma unroll
                    for (int i = 0; i < LA; i++)
#pragma unroll
                        for (int j = 0; j < LB; j++)
#pragma unroll
                            for (int t = 0; t < 4; t++)
                                acc[i + j][t >> 1][t & 1] =
                                    __builtin_amdgcn_mfma_i32_16x16x64_i8(a[e][i][t >> 1], b[e][j][t & 1], acc[i + j][t >> 1][t & 1], 0, 0, 0);
                }
            }
        });
        // accumulator i of lane l in block t: row 4 (l / 16) + i, column l % 16; orders 0 to 3 and 4 to 6 are added in
        // 64-bit integers, of which the upper one takes the carry and stays below 2^53: the one rounding is the last
        const float *src = C + (row0 + (int64_t)bi * LIMB_BLOCK + wr * 32 + 4 * q) * N + (int64_t)bj * LIMB_BLOCK + wc * 32 + l16;
#pragma unroll
        for (int t = 0; t < 4; t++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const double cd = (double)src[((t >> 1) * 16 + i) * N + (t & 1) * 16];
                const long long lo = (long long)acc[0][t >> 1][t & 1][i] + ((long long)acc[1][t >> 1][t & 1][i] << 8) +
                                     ((long long)acc[2][t >> 1][t & 1][i] << 16) + ((long long)acc[3][t >> 1][t & 1][i] << 24);
                const long long hi = (long long)acc[4][t >> 1][t & 1][i] + ((long long)acc[5][t >> 1][t & 1][i] << 8) +
                                     ((long long)acc[6][t >> 1][t & 1][i] << 16);
                const double d = fma((double)(hi + (lo >> 32)), 4294967296.0, (double)(unsigned int)lo) * (1.0 / 281474976710656.0);
                e2 += (cd - d) * (cd - d);
                d2 += d * d;
                c2 += cd * cd;
            }
    }
    e2 = wave_sum(e2);
    d2 = wave_sum(d2);
    c2 = wave_sum(c2);
    if (lane == 63) {
        red[wave][0] = e2;
        red[wave][1] = d2;
        red[wave][2] = c2;
    }
    __syncthreads();
    double own = 0.0;
    if (threadIdx.x < 3) own = red[0][threadIdx.x] + red[1][threadIdx.x] + red[2][threadIdx.x] + red[3][threadIdx.x];
    finish_sums<3>(ws, own, host_out, host_seq, seq);
}

// Dropped norm products of every output tile: a wave takes one tile row and BOUND_JB tile columns, lane = k, so that a
// step's loads go out together.  `per_tile` gets the tiles' sums, host_out (unless null) the sum of their squares, each
// workgroup's share of it through the workspace: a 64-bit float add on one address by every wave was 50 us of the
// 52 us that 64 x 64 tiles took.
constexpr int BOUND_JB = 4;
constexpr unsigned BOUND_MAX_WG = 2048;

__global__ __launch_bounds__(256) void k_dropped_bound(const float *__restrict__ nA, const float *__restrict__ nBt,
                                                       int nbM, int nbK, int nbN, float tau, ReportWorkspace *__restrict__ ws,
                                                       ReportSums *__restrict__ host_out, unsigned long long *__restrict__ host_seq,
                                                       unsigned long long seq, double *__restrict__ per_tile) {
    __shared__ double red[4];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int jb = (nbN + BOUND_JB - 1) / BOUND_JB;
    const int64_t units = (int64_t)nbM * jb;
    double sum = 0.0;
    for (int64_t u = (int64_t)blockIdx.x * 4 + wave; u < units; u += (int64_t)gridDim.x * 4) {
        const int i = (int)(u / jb), j0 = (int)(u % jb) * BOUND_JB;
        double s[BOUND_JB];
#pragma unroll
        for (int jj = 0; jj < BOUND_JB; jj++) s[jj] = 0.0;
        for (int k = lane; k < nbK; k += 64) {
            const float a = nA[(int64_t)i * nbK + k];
            float b[BOUND_JB];
#pragma unroll
            for (int jj = 0; jj < BOUND_JB; jj++) b[jj] = nBt[(int64_t)(j0 + jj < nbN ? j0 + jj : nbN - 1) * nbK + k];
#pragma unroll
            for (int jj = 0; jj < BOUND_JB; jj++) {
                const float p = a * b[jj];
                if (!(p >= tau)) s[jj] += (double)a * (double)b[jj];
            }
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1)
#pragma unroll
            for (int jj = 0; jj < BOUND_JB; jj++) s[jj] += __shfl_down(s[jj], off, 64);
        if (lane == 0)
#pragma unroll
            for (int jj = 0; jj < BOUND_JB; jj++)
                if (j0 + jj < nbN) {
                    sum += s[jj] * s[jj];
                    if (per_tile) per_tile[(int64_t)i * nbN + j0 + jj] = s[jj];
                }
    }
    if (!host_out) return;
    if (lane == 0) red[wave] = sum;
    __syncthreads();
    finish_sums<1>(ws, threadIdx.x == 0 ? red[0] + red[1] + red[2] + red[3] : 0.0, host_out, host_seq, seq);
}

__global__ void k_clear_report(ReportWorkspace *ws) {
    if (threadIdx.x <= TICKET_GROUPS) ws->tickets.t[threadIdx.x].n = 0;
    if (threadIdx.x <= RANGE_FLAGS) ws->range[threadIdx.x].call = 0;
}

hipError_t launch_clear_report(void *workspace, hipStream_t s) {
    k_clear_report<<<1, 64, 0, s>>>((ReportWorkspace *)workspace);
    return hipGetLastError();
}

// Blocks per wave of the dense product: 16-wide blocks, rows x columns.  Every SIMD works through the same number of
// waves, so a wave's time (in MFMAs a step, and the share that the conversions add) times the fullest SIMD's number of waves decides.
struct ErrorShape {
    int nbr, nbc;
    double cost;        // per MFMA, relative
};
static const ErrorShape ERROR_SHAPES[3] = {{4, 4, 1.00}, {4, 2, 1.06}, {2, 2, 1.12}};

static int error_shape(int64_t rows, int64_t N, int n_cu, int64_t *n_wg, double *mfmas = nullptr) {
    int best = 0;
    double best_time = 0.0;
    for (int i = 0; i < 3; i++) {
        const ErrorShape &e = ERROR_SHAPES[i];
        const int64_t wg = ((rows + 32 * e.nbr - 1) / (32 * e.nbr)) * ((N + 32 * e.nbc - 1) / (32 * e.nbc));
        const double time = (double)((wg + n_cu - 1) / n_cu) * e.nbr * e.nbc * e.cost;      // (one wave of a workgroup per SIMD)
        if (i == 0 || time < best_time) {
            best = i;
            best_time = time;
            *n_wg = wg;
        }
    }
    if (mfmas) *mfmas = best_time;
    return best;
}

// Workgroups of k_error_limbs: groups of gb x gb, ngj of them side by side.  A group is no wider than C in either direction
// and there is one for every gb x gb blocks that C has, but for what rounds up to whole groups and XCDs: workgroups
// without a block are launched, waited for and added up all the same (1048576 x 64 with 64 of them to a block 6050 us).
struct LimbGrid {
    int nbi, nbj, gb, ngj;
    int64_t n_wg;
};
static LimbGrid limb_grid(int64_t rows, int64_t N, int n_xcd) {
    LimbGrid g;
    g.nbi = (int)(rows / LIMB_BLOCK);
    g.nbj = (int)(N / LIMB_BLOCK);
    const int64_t blocks = (int64_t)g.nbi * g.nbj;
    g.gb = blocks >= 2048 ? 8 : blocks >= 512 ? 4 : 1;
    while (g.gb > g.nbi || g.gb > g.nbj) g.gb /= 2;
    g.ngj = (g.nbj + g.gb - 1) / g.gb;
    const int64_t groups = (int64_t)((g.nbi + g.gb - 1) / g.gb) * g.ngj;
    g.n_wg = (groups + n_xcd - 1) / n_xcd * n_xcd * g.gb * g.gb;
    return g;
}

static int64_t limb_kb(int64_t K) { return (K + LIMB_BLOCK - 1) / LIMB_BLOCK; }

// Bytes of the planes and the blocks' numbers of limbs of both operands; 0: the fp64 pipeline is to be used -- beyond
// what 32 bits add up, beyond 4 GiB of planes, and where the split of the operands, which no block of C shares, takes more than
// 1 / 2.4 of the fp64 product's time.  Both are estimated, in us: of the product 0.033 per MFMA of its fullest SIMD (4096^3 2112,
// 1280^3 94, 64 rows of 4096^2 151), of the split 6 for its launches, two passes over 2 bytes a value at 3 TB/s, and the
// scratch's allocation where the context does not keep it.  fp64 -> whole numbers, whole calls, on uniform values | exp(-d / 100) |
// values too large for limbs, by the estimates' ratio: 1.5, 512 x 256 x 512 27.4 -> 27.1 | 26.4 | 31.0 and 65536 x 1024 x 64 151 ->
// 147 | 61 | 226; 2.2, 512 x 384 x 512 32.2 -> 29.4 | 28.1 | 35.7; 2.4, 4096 x 256 x 512 35.6 -> 31.7 | 27.8 | 46.9 and 32768 x 512 x 128
// 88 -> 62 | 41 | 118; 2.6, 1024 x 512 x 1024 37.1 -> 34.0 | 32.1 | 40.1; 2.7, 65536 x 512 x 128 150 -> 102 | 58 | 193; 2.8, 512^3 36.9 ->
// 31.4 | 30.1 | 40.1; 4.3, 1024^3 55.2 -> 41.4 | 38.5 | 58.4; 5.3, 65536 x 512 x 256 281 -> 157 | 80 | 326; 8.6, 1280^3 102 -> 54 | 45 |
// 122.  What the line weighs is the tenth to half that large values lose against what the others gain, 5 to 20 % just below it.  With
// K below 256 a block's fixed costs outweigh its few products: 4096 x 64 x 4096 59 -> 75 | 66 | 70, K = 128 92 -> 83 | 67 | 103, K = 192 122 ->
// 92 | 68 | 134.  (Both lines were drawn when the product loaded its operands to registers and took longer.)
size_t limb_bytes(int64_t rows, int64_t K, int64_t N, int n_cu) {
    if (K > LIMB_MAX_K || K < 256) return 0;
    const size_t blocks = (size_t)(rows / LIMB_BLOCK + N / LIMB_BLOCK) * (size_t)limb_kb(K);
    if (blocks >= (1u << 31) / (LIMBS * LIMB_PLANE / 2)) return 0;       // 4 GiB
    const size_t bytes = blocks * (LIMBS * LIMB_PLANE) + blocks;
    int64_t n_wg = 0;
    double mfmas = 0.0;
    (void)error_shape(rows, N, n_cu, &n_wg, &mfmas);
    const double dense = 0.033 * mfmas * (double)(K / 4);
    const double split = 6.0 + (double)(rows + N) * (double)K * 4.0 / 3.0e6 + (bytes > LIMBS_KEPT ? 500.0 : 0.0);
    return dense < 2.4 * split ? 0 : bytes;
}

size_t report_workspace_bytes(int64_t rows, int64_t N, int n_cu, int n_xcd) {
    int64_t n_wg = 0;
    if (rows > 0) {
        (void)error_shape(rows, N, n_cu, &n_wg);
        const int64_t n_limb = limb_grid(rows, N, n_xcd).n_wg;
        if (n_limb > n_wg) n_wg = n_limb;
    }
    const size_t doubles = 3 * (size_t)n_wg > BOUND_MAX_WG ? 3 * (size_t)n_wg : BOUND_MAX_WG;
    return sizeof(ReportWorkspace) + doubles * sizeof(double);
}

hipError_t launch_error_vs_dense(const void *packedA, const void *packedB, int64_t K, int64_t N, int tile, const float *C,
                                 int64_t row0, int64_t row1, int n_cu, void *workspace, ReportSums *host_out,
                                 unsigned long long *host_seq, unsigned long long seq, hipStream_t s) {
    int64_t n_wg = 0;
    const int shape = error_shape(row1 - row0, N, n_cu, &n_wg);
    const _Float16 *pA = (const _Float16 *)packedA, *pB = (const _Float16 *)packedB;
    ReportWorkspace *ws = (ReportWorkspace *)workspace;
    const int nwg_n = (int)((N + 32 * ERROR_SHAPES[shape].nbc - 1) / (32 * ERROR_SHAPES[shape].nbc));
#define SPAMM_DENSE(NBR, NBC) \
    k_error_dense<NBR, NBC><<<(unsigned)n_wg, 256, 0, s>>>(pA, pB, K, N, tile, C, row0, row1, nwg_n, ws, host_out, host_seq, seq)
    if (shape == 0) SPAMM_DENSE(4, 4);
    else if (shape == 1) SPAMM_DENSE(4, 2);
    else SPAMM_DENSE(2, 2);
#undef SPAMM_DENSE
    return hipGetLastError();
}

hipError_t launch_error_limbs(const void *packedA, const void *packedB, int64_t K, int64_t N, int tile, const float *C,
                              int64_t row0, int64_t row1, int n_cu, int n_xcd, void *limbs, void *workspace, ReportSums *host_out,
                              unsigned long long *host_seq, unsigned long long seq, hipStream_t s) {
    const LimbGrid g = limb_grid(row1 - row0, N, n_xcd);
    const int nkb = (int)limb_kb(K);
    const int64_t blocksA = (int64_t)g.nbi * nkb, blocksB = (int64_t)g.nbj * nkb;
    const _Float16 *pA = (const _Float16 *)packedA, *pB = (const _Float16 *)packedB;
    ReportWorkspace *ws = (ReportWorkspace *)workspace;
    int8_t *planes = (int8_t *)limbs;
    uint8_t *cls = (uint8_t *)limbs + (blocksA + blocksB) * (LIMBS * LIMB_PLANE);
    const LimbOperand a = {pA, planes, cls, row0, blocksA};
    const LimbOperand b = {pB, planes + blocksA * (LIMBS * LIMB_PLANE), cls + blocksA, 0, blocksB};
    k_limbs<<<(unsigned)(blocksA + blocksB), 256, 0, s>>>(a, b, K, tile, nkb, seq, ws);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    // Where fp64 takes larger blocks of C than 64 x 64 the host launches it when it is told to: some 10 us beside the 300
    // and more of such a product.  (Launched behind every call of these sizes it was 4 us on the next one.)
    int64_t n_wg = 0;
    const bool dense_here = error_shape(row1 - row0, N, n_cu, &n_wg) == 2;
    k_error_limbs<<<(unsigned)g.n_wg, 256, 0, s>>>(a.planes, a.cls, b.planes, b.cls, nkb, g.nbi, g.nbj, g.gb, g.ngj, n_xcd, pA, pB, K, N,
                                                   tile, C, row0, ws, host_out, host_seq, seq, dense_here);
    return hipGetLastError();
}

hipError_t launch_dropped_bound(const float *nA, const float *nBt, int64_t nbM, int64_t nbK, int64_t nbN, float tau,
                                void *workspace, ReportSums *host_out, unsigned long long *host_seq, unsigned long long seq,
                                double *per_tile, hipStream_t s) {
    const int64_t wg = (nbM * ((nbN + BOUND_JB - 1) / BOUND_JB) + 3) / 4;
    k_dropped_bound<<<wg < (int64_t)BOUND_MAX_WG ? (unsigned)wg : BOUND_MAX_WG, 256, 0, s>>>(nA, nBt, (int)nbM, (int)nbK, (int)nbN, tau,
                                                                                (ReportWorkspace *)workspace, host_out, host_seq, seq, per_tile);
    return hipGetLastError();
}

}  // namespace spamm
