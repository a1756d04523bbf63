// Internal declarations shared by the translation units of libspamm_gfx950.so.
// Host-side launchers only; kernels live in the .hip files.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace spamm {

// ---------------------------------------------------------------------------
// Packed fp16 operand layout (private to the library).
//
// An operand is cut into b x b tiles; every tile is one contiguous block of
// b*b halves.  Inside a tile the element with free index r (row of A / column
// of B) and contraction index k (column of A / row of B) sits at
//     ((k / 8) * b + r) * 8 + (k % 8)          [units: halves]
// i.e. [k-group][r][8]: a 16-byte vector holds 8 consecutive k of one r, which
// is exactly one lane's share of an MFMA 16x16x32 (or 32x32x16) operand, and 32 consecutive
// r are 512 contiguous bytes.  Tile order: A tile (I,Kt) at I*nbK + Kt,
// B tile (Kt,J) at J*nbK + Kt, so that the k tiles of one output tile are
// consecutive in memory for both operands.
// ---------------------------------------------------------------------------

// Output tiles are grouped into macro tiles of (256/b) x (256/b) tiles
// (256 x 256 elements); one workgroup of the gated GEMM owns one macro tile.
inline int macro_dim(int tile) { return 256 / tile; }

// Macro tiles are scheduled in super tiles of SUPER_M x SUPER_N macro tiles:
// 32 workgroups, one per CU of an XCD, that share operand panels in that
// XCD's L2.
constexpr int SUPER_M = 4;
constexpr int SUPER_N = 8;
constexpr int MAX_XCD = 8;      // an unpartitioned MI355X: 8 XCDs of 32 CUs

// Number of XCDs the schedule is built for: workgroup b of a grid runs on XCD b % n.  Derived
// from the CU count of the device (or partition): 32 CUs per XCD; anything that is not 1, 2, 4 or
// 8 whole XCDs gets one flat sequence (n = 1), which is correct on any device and only gives up
// the sharing of operand panels in an XCD's L2.
inline int xcds_for_cu_count(int cus) {
    for (int n = MAX_XCD; n >= 1; n >>= 1)
        if (cus == n * SUPER_M * SUPER_N) return n;
    return 1;
}

// Workgroups per XCD in the GEMM grid: whole super tiles, dealt round-robin over n_xcd XCDs.
// (Buffers are sized for n_xcd = MAX_XCD, which is an upper bound for every smaller power of two.)
inline int sched_rounds(int tile, int64_t nbM, int64_t nbN, int n_xcd = MAX_XCD) {
    const int MT = 256 / tile;
    const int nMacM = (int)((nbM + MT - 1) / MT), nMacN = (int)((nbN + MT - 1) / MT);
    const int n_super = ((nMacM + SUPER_M - 1) / SUPER_M) * ((nMacN + SUPER_N - 1) / SUPER_N);
    return (n_super + n_xcd - 1) / n_xcd;
}

// One entry of a macro tile's union k list: tile column/row k of the
// operands plus the set of output tiles (bit a*MT+b = tile row a, column b of
// the macro tile) that keep the product with this k.  16 bytes so that the
// GEMM fetches an entry with one scalar load.
struct __attribute__((aligned(16))) MacroEntry {
    uint32_t k;
    uint32_t need;      // bits 0..7: tile rows with any kept product, bits 8..15: tile columns
    uint32_t mask_lo;
    uint32_t mask_hi;
};

// Kept products of a gate: their total (k_gate, k_order), or below zero minus the number of units that C has, and each
// unit's (k_small, row by row).
constexpr int64_t SMALL_MAX_UNITS = 1536;
struct KeptProducts {
    int64_t total;
    uint32_t units[SMALL_MAX_UNITS];
};

struct GateBuffers {
    const float *nA;        // [nbM x nbK]
    const float *nBt;       // [nbN x nbK]  (transposed B norm map)
    KeptProducts *kept;
    int32_t *counts;        // [nbM*nbN]
    uint64_t *mask;         // [nbM*nbN*words]
    MacroEntry *macro_list; // [n_macro*nbK]   union list of k per macro tile
    int32_t *macro_count;   // [n_macro][2]    entries in the union list, of which full (listed first)
    int32_t *macro_work;    // [n_macro]       kept products in the macro tile
    int32_t *order;         // [n_xcd * P]     macro tile of XCD x's q-th workgroup (P = rounds * 32), valid for q < sched[8 + x]
    int32_t *sched;         // [24]            per XCD x: [x] computing items, [8 + x] all items, [16 + x] ticket
                            //                 counter of the persistent GEMM (zero between launches)
};

// tau_skip > 0: tau-aware pass, the fp16 copy of tile (i, k) is written only if
// fl(nA[i,k] * rowmax[k]) >= tau_skip (rowmax[k] = max_j nB[k,j], launch_rowmax)
hipError_t launch_normmap_a(const void *X, bool in16, int64_t rows, int64_t cols, int tile, void *packed,
                            float *nm, const float *rowmax, float tau_skip, hipStream_t s);
hipError_t launch_rowmax(const float *nB, int64_t nbK, int64_t nbN, float *rowmax, hipStream_t s);
// tau_skip > 0: the fp16 copy of tiles of norm zero is not written (no product with them reaches tau)
hipError_t launch_normmap_b(const void *X, bool in16, int64_t rows, int64_t cols, int tile, void *packed,
                            float *nm, float *nmT, float tau_skip, hipStream_t s);
// A = B (square): one pass over X for both operand roles
hipError_t launch_normmap_ab(const void *X, bool in16, int64_t n, int tile, void *packedA, float *nmA,
                             void *packedB, float *nmB, float *nmBt, float tau_skip, hipStream_t s);
// both operands in one launch, for small ones (normmap_pair_fits); tau_skip > 0: tiles of norm zero are not written
bool normmap_pair_fits(bool in16, bool tau_aware, int64_t M, int64_t K, int64_t N, int tile);
hipError_t launch_normmap_pair(const void *A, const void *Bm, bool in16, int64_t M, int64_t K, int64_t N, int tile, void *packedA,
                               float *nmA, void *packedB, float *nmB, float *nmBt, float tau_skip, hipStream_t s);
// error report tooling (kernels_tools.hip).  Results go to host_out, pinned host memory: valid once *host_seq == seq
// (per_tile: once the stream has been waited for).  The workspace's tickets are zero between launches (launch_clear_report once after allocation).
struct ReportSums {
    double v[3];
};
size_t report_workspace_bytes(int64_t rows, int64_t N, int n_cu, int n_xcd);      // rows = 0: the bound only
hipError_t launch_clear_report(void *workspace, hipStream_t s);
hipError_t launch_error_vs_dense(const void *packedA, const void *packedB, int64_t K, int64_t N, int tile, const float *C,
                                 int64_t row0, int64_t row1, int n_cu, void *workspace, ReportSums *host_out,
                                 unsigned long long *host_seq, unsigned long long seq, hipStream_t s);
// the same on the integer matrix pipeline; limbs: limb_bytes() of scratch (0: not for this shape).  Where an operand holds
// values that it cannot take (beyond +-127, inf, NaN) it forms small blocks of C in fp64 itself; a first sum below zero asks
// for launch_error_vs_dense, whose blocks are larger
size_t limb_bytes(int64_t rows, int64_t K, int64_t N, int n_cu);
// Scratch of a report that a context keeps for the next one: that of 8192^3.  A larger one is given back -- to allocate and
// free it takes 0.3 to 0.7 ms, beside 1.3 to 67 ms of reports of 12288^3 and 16384^3 -- and what is kept goes when another
// buffer of the context finds no memory.
constexpr size_t LIMBS_KEPT = ((size_t)512 << 20) + ((size_t)512 << 10);
hipError_t launch_error_limbs(const void *packedA, const void *packedB, int64_t K, int64_t N, int tile, const float *C,
                              int64_t row0, int64_t row1, int n_cu, int n_xcd, void *limbs, void *workspace, ReportSums *host_out,
                              unsigned long long *host_seq, unsigned long long seq, hipStream_t s);
// host_out->v[0] (optional) = sum over tiles of s_ij^2, s_ij = sum_{k dropped} nA[i,k]*nB[k,j]; per_tile (optional): s_ij
hipError_t launch_dropped_bound(const float *nA, const float *nBt, int64_t nbM, int64_t nbK, int64_t nbN, float tau,
                                void *workspace, ReportSums *host_out, unsigned long long *host_seq, unsigned long long seq,
                                double *per_tile, hipStream_t s);
hipError_t launch_unpack(const void *packed, int64_t rows, int64_t cols, int tile, int role,
                         uint16_t *out, hipStream_t s);
hipError_t launch_transpose_normmap(const float *nB, int64_t nbK, int64_t nbN, float *nBt,
                                    hipStream_t s);
hipError_t launch_fill_decay(float *X, int64_t rows, int64_t cols, const float *table,
                             uint64_t seed, int random, hipStream_t s);

size_t gate_lds_bytes(int tile, int64_t nbK, int chunk_cap = 0);   // chunk_cap > 0: at most that many 64-k words of bitmaps in LDS at a time
inline size_t gate_lds_limit() { return 160 * 1024 - 1088; }   // dynamic LDS of k_gate (beside 1 KiB of counts)
// k_order ranks the super tiles of C (4 x 8 macro tiles of 256 x 256) in one workgroup's LDS
constexpr int LPT_MAX_SUPER = 2048;     // the greedy deal's table is laid out for at most this many super tiles,
constexpr int LPT_GREEDY_MAX = 64;      // and it runs while at most this many of them hold any work
constexpr int BAND_DEAL_MAX = 256;      // the grouped row-major deal runs up to this many super tiles with work
inline size_t order_lds_bytes(int tile, int64_t nbM, int64_t nbN) {
    const int MT = 256 / tile;
    const int64_t nMacM = (nbM + MT - 1) / MT, nMacN = (nbN + MT - 1) / MT;
    const size_t n_super = (size_t)(((nMacM + SUPER_M - 1) / SUPER_M) * ((nMacN + SUPER_N - 1) / SUPER_N));
    // two positions (first: the length) and the set of computing macro tiles by super tile, origin by rank, for the
    // table deals 16-bit entries; beyond 512 super tiles the ranking may sort indices padded to a power of
    // two in the place of the last two
    size_t np2 = 1024;
    while (np2 < n_super) np2 *= 2;
    const size_t fixed = (3 * n_super + 2 * MAX_XCD) * sizeof(int);
    const size_t tables = n_super * sizeof(int) + (n_super <= (size_t)LPT_MAX_SUPER ? (n_super + 2 * MAX_XCD) * sizeof(uint16_t) : 0);
    const size_t sorting = n_super > 512 ? np2 * sizeof(int) : 0;
    return fixed + (tables > sorting ? tables : sorting);
}
constexpr int ORDER_MAX_SUPER = 8192;
inline size_t order_lds_limit() { return (size_t)(4 * ORDER_MAX_SUPER + 2 * MAX_XCD) * sizeof(int); }
hipError_t gate_init();   // one-time kernel attribute set-up
hipError_t launch_gate(const GateBuffers &g, int64_t nbM, int64_t nbK, int64_t nbN, int tile,
                       float tau, int n_xcd, int chunk_cap, hipStream_t s);
// per-tile ascending k lists [n_tiles x nbK] from the gate's bitmaps (read-back only)
hipError_t launch_klist(const uint64_t *mask, uint16_t *klist, int64_t n_tiles, int64_t nbK, hipStream_t s);

// tau selection (kernels_tau.hip)
struct TauState {
    unsigned long long want;      // rank (1-based, from the top) still to find inside the prefix
    unsigned long long greater;   // products strictly above the current prefix range
    unsigned long long kept;      // products >= tau (valid after the last pass)
    uint32_t prefix;              // decided high bits, right-aligned
    uint32_t tau_bits;
};
struct TauCounts {
    unsigned long long count;     // products with (double)p >= threshold
    double sum;                   // sum of all products
};
struct TauResult {                // of the bisection so far
    double norm, rate;
    int64_t done;
};
size_t tau_workspace_bytes();
// Results go to *host_out, pinned host memory: valid once *host_seq == seq (the kernel that writes it is the
// last of the call that does anything).
hipError_t launch_tau_clear(void *workspace, hipStream_t s);          // once after allocation, and after a failed call
hipError_t launch_tau_select(const float *nA, const float *nBt, int64_t nbM, int64_t nbK, int64_t nbN,
                             unsigned long long want, void *workspace, TauState *host_out, unsigned long long *host_seq,
                             unsigned long long seq, hipStream_t s);
hipError_t launch_tau_count(const float *nA, const float *nBt, int64_t nbM, int64_t nbK, int64_t nbN, double thr,
                            void *workspace, TauCounts *host_out, unsigned long long *host_seq, unsigned long long seq, hipStream_t s);
// the whole bisection in one launch, for few products
bool tau_tune_small(int64_t nbM, int64_t nbK, int64_t nbN);
hipError_t launch_tau_tune_small(const float *nA, const float *nBt, int64_t nbM, int64_t nbK, int64_t nbN, double expected, double tol,
                                 int max_rounds, TauResult *host_out, unsigned long long *host_seq, unsigned long long seq, hipStream_t s);
// the bisection: `first` starts it (its round 0), then TREE_ROUNDS rounds per pass until done.  *host_seq == seq: it is done
// or the passes are; `call` tells the bisection's launches from those of a later one
constexpr int TREE_ROUNDS = 10;
hipError_t launch_tau_tune(const float *nA, const float *nBt, int64_t nbM, int64_t nbK, int64_t nbN, double expected, double tol,
                           int max_rounds, bool first, int passes, unsigned int call, void *workspace, TauResult *host_out,
                           unsigned long long *host_seq, unsigned long long seq, hipStream_t s);

hipError_t gemm_init();   // one-time kernel attribute set-up
hipError_t launch_gemm(const void *packedA, const void *packedB, const GateBuffers &g, int64_t M,
                       int64_t K, int64_t N, int tile, float *C, int n_xcd, int n_cu, int ring, int shape, hipStream_t s);
// work unit of the gated GEMM: a whole macro tile (256 x 256 of C, one workgroup per CU), half of
// one (128 x 256, two workgroups per CU), a whole one by eight waves, or whole ones by workgroups
// that stay on their CU and draw items from a ticket counter per XCD
// gate and multiply in one launch (kernels_small.hip)
constexpr int64_t SMALL_MAX_NBK = 2048;      // its k list lives in LDS
hipError_t small_init();
bool small_fits(int64_t M, int64_t K, int64_t N, int tile, float tau, bool stages, int n_cu);
constexpr int SMALL_GATE = 1, SMALL_MULTIPLY = 2;    // what launch_small does: either or both
hipError_t launch_small(const void *packedA, const void *packedB, const GateBuffers &g, int64_t M, int64_t K, int64_t N,
                        int tile, int mode, float tau, float *C, int n_cu, int n_xcd, hipStream_t s);
constexpr int GEMM_SHAPE_FULL = 1, GEMM_SHAPE_HALF = 2, GEMM_SHAPE_W8 = 3, GEMM_SHAPE_PERSIST = 4;
constexpr int SCHED_WORDS = 3 * MAX_XCD;     // GateBuffers::sched

}  // namespace spamm
