// Error-report tooling around the multiply (not on the hot path).
//
// The reference compares SpAMM against a dense cuBLAS product and prints
// ||C_dense - C_spamm||_F, ||C_dense||_F, ||C_spamm||_F (check_simple_gpu,
// tool.cu:227-280; COUNTERRTRANS, tool.cu:6-24).  Here the dense product is
// an exact fp64 product of the same fp16 operands, formed on the fp64 matrix
// pipeline (v_mfma_f64_16x16x4_f64) block by block and reduced on the fly (it is
// never stored), next to the tau-derived bound
// sqrt(sum_ij (sum_{k dropped} nA[i,k]*nB[k,j])^2).
//
// What bounds it: the fp64 matrix pipeline (128 operations per clock and CU) and the VALU's
// conversions beside it -- fp16 to fp64 is two instructions per value, one of them at a
// quarter of the rate, and they take the place of MFMAs.  So a wave's block of C is as large as
// the number of blocks allows: each converted value serves NBR or NBC MFMAs.  4096^3:
// 2229 us with 32 x 32 per wave and 4-byte loads, 2109 now (65 TFLOP/s; the pipeline's 128 operations at the clock
// that the chip holds under them, about 2 GHz); 1984 x 2176 x 768: 196 -> 158.  The scalar bound of 64 x 64 x 64
// tiles 52 -> 7 us, the per-tile one 51 -> 4; results go straight to host memory (a clearing launch before and a copy
// after each were 25 us a call): the whole report 2429 -> 2174 us at 4096^3, 380 -> 244 at 1984 x 2176 x 768.
#include "reduce_device.h"

namespace spamm {

typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef _Float16 half8t __attribute__((ext_vector_type(8)));

struct ReportWorkspace {
    unsigned int ticket;                // workgroups of the running launch that have finished; zero between launches
    unsigned int pad_;
    double part[1];                     // per workgroup: its sums (report_workspace_bytes says how many)
};

// Sums of all workgroups' N values, by the workgroup that finishes last, to host_out (pinned host memory): in a
// fixed order, so that a repeated call gives the same number.  `own`: the workgroup's values, in thread i the i-th.
template <int N>
__device__ __forceinline__ void finish_sums(ReportWorkspace *ws, double own, ReportSums *host_out, unsigned long long *host_seq,
                                            unsigned long long seq) {
    __shared__ double s_fin[4][N];
    if (threadIdx.x < N)
        agent_store(reinterpret_cast<unsigned long long *>(&ws->part[(size_t)blockIdx.x * N + threadIdx.x]), __builtin_bit_cast(unsigned long long, own));
    if (!last_workgroup(&ws->ticket)) return;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    double v[N];
#pragma unroll
    for (int i = 0; i < N; i++) v[i] = 0.0;
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
    const int l16 = lane & 15, q = lane >> 4;
    double e2 = 0, d2 = 0, c2 = 0;
    if (br < row1 && bc < N) {              // (whole blocks: rows and columns come in multiples of 64)
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
        Vecs v0, v1;
        load(v0, 0);
        int64_t s = 0;
        for (; s + 1 < steps; s += 2) {
            load(v1, s + 1);
            multiply(v0);
            load(v0, s + 2);
            multiply(v1);
        }
        if (s < steps) multiply(v0);
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

__global__ void k_clear_report(ReportWorkspace *ws) { ws->ticket = 0; }

hipError_t launch_clear_report(void *workspace, hipStream_t s) {
    k_clear_report<<<1, 1, 0, s>>>((ReportWorkspace *)workspace);
    return hipGetLastError();
}

// Blocks per wave of the dense product: 16-wide blocks, rows x columns.  Every SIMD works through the same number of
// waves, so a wave's time (in MFMAs, and the share that the conversions add) times the fullest SIMD's number of waves decides.
struct ErrorShape {
    int nbr, nbc;
    double cost;        // per MFMA, relative
};
static const ErrorShape ERROR_SHAPES[3] = {{4, 4, 1.00}, {4, 2, 1.06}, {2, 2, 1.12}};

static int error_shape(int64_t rows, int64_t N, int n_cu, int64_t *n_wg) {
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
    return best;
}

size_t report_workspace_bytes(int64_t rows, int64_t N, int n_cu) {
    int64_t n_wg = 0;
    if (rows > 0) (void)error_shape(rows, N, n_cu, &n_wg);
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
    if (shape == 0) k_error_dense<4, 4><<<(unsigned)n_wg, 256, 0, s>>>(pA, pB, K, N, tile, C, row0, row1, nwg_n, ws, host_out, host_seq, seq);
    else if (shape == 1) k_error_dense<4, 2><<<(unsigned)n_wg, 256, 0, s>>>(pA, pB, K, N, tile, C, row0, row1, nwg_n, ws, host_out, host_seq, seq);
    else k_error_dense<2, 2><<<(unsigned)n_wg, 256, 0, s>>>(pA, pB, K, N, tile, C, row0, row1, nwg_n, ws, host_out, host_seq, seq);
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
