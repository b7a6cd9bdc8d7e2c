// RandomLayer + Probabilistic nodes on gfx950.
//   y[b,n,d] = sum_a sigmoid(w[n,a,d]/T) * prod_j (x_j a_j + (1-x_j)(1-a_j)),  x_j = x[b, idx[n,j]]
// i.e. the multilinear interpolation of the node's sigmoid table at the point x.
//
// k <= 6: tiled kernels with lanes = batch rows (see below); k > 6: one-thread-per-element kernels
// with atomics.
#include "dl_common.h"

__device__ __forceinline__ float dl_sigmoid(float v) { return 1.0f / (1.0f + expf(-v)); }

typedef float prob_f4 __attribute__((ext_vector_type(4)));
#define PROB_RSRC 0x00020000
#define PROB_HYBRID_EPS 1e-8f

// ---------------------------------------------------------------------------------
// k <= 6 path.  As for the DWN nodes, a wavefront's 64 lanes are 64 batch rows and everything
// that belongs to a node is wave-uniform: its input indices are scalar byte offsets, its sigmoid
// table is read through scalar loads.  Tensors that cross the [batch, feature] boundary are
// re-tiled once: xT [B/64][I][64], gmT [B/64][N*O*k][64], so the row of an
// input (or a column's gradient) for a batch tile is 256 contiguous bytes, whatever the mapping.
//   to_tiles    : [B][C] -> [B/64][C][64], rows past B are zero; carries the tables (tiny): sig[c][a] =
//                 sigmoid(raw[n,a,d] / T), c = n*O + d, and cen, the same less a value of the column's own
//   fwd_t       : per (column, batch tile): fold the table along x_0, x_1, ... ; y leaves through
//                 an LDS transpose as whole rows
//   bwd_t       : one wavefront per column over a chunk of batch tiles.  The product weights factor into those of
//                 the lower and of the upper inputs; that gives dy/dx_j for all j and the table gradient in about
//                 3 * 2^k operations.  Table-gradient partials stay in registers over the chunk,
//                 are summed across lanes once and written per chunk; gm_j goes to gmT.
//   reduce      : fixed-order sum of the chunk partials, times sigmoid'(w/T)/T
//   gather_t    : gx[b,i] = sum over the CSR entries (n,j) of input i (and d) of gmT: a wavefront
//                 owns 16 inputs, sums each in CSR order in a register, rows leave through LDS.
// The temperature of the layer: one value (inv = 1 / max(T, 1e-6)) or every node's own (t_n, a device array [N],
// probabilistic_node.py:277-282 reads each node's buffer).
struct ProbTemp {
    float inv;
    const float *t_n;
};
__device__ __forceinline__ float prob_inv_t_of(const ProbTemp &T, int n) {
    if (!T.t_n) return T.inv;
    const float t = T.t_n[n];
    return 1.0f / (t > 1e-6f ? t : 1e-6f);
}
__global__ __launch_bounds__(256) void prob_sig_table(const float *__restrict__ raw, ProbTemp T, float *__restrict__ sig,
                                                       int N, int L, int O) {
    const long long e = (long long)blockIdx.x * 256 + threadIdx.x;
    if (e >= (long long)N * L * O) return;
    const int a = (int)(e % L);
    const long long c = e / L;
    const int n = (int)(c / O), d = (int)(c % O);
    sig[e] = dl_sigmoid(raw[((size_t)n * L + a) * O + d] * prob_inv_t_of(T, n));
}

// Tables for the backward, element e of [column][2^k]: sig (nullable) the sigmoid table, cen the same less a value of the
// column's own, which no gradient of the inputs depends on: sums of it round by what the table varies, not by what it is.
struct ProbTables {
    const float *raw, *luts;  // probabilistic: weights [N][L][O], hybrid: the table as given, [N O][L]
    ProbTemp T;
    float *sig, *cen;
    int N, L, O;
    bool flat = false;        // hybrid: raw in the table's own layout
};
__device__ __forceinline__ void prob_table_element(const ProbTables &q, long long e) {
    if (e >= (long long)q.N * q.L * q.O) return;
    const int a = (int)(e % q.L);
    const long long c = e / q.L;
    const int n = (int)(c / q.O), d = (int)(c % q.O);
    const float inv = q.luts ? 1.0f : prob_inv_t_of(q.T, n);
    auto value = [&](int at) -> float {
        return q.luts ? q.luts[c * q.L + at] : dl_sigmoid(q.raw[q.flat ? (size_t)c * q.L + at : ((size_t)n * q.L + at) * q.O + d] * inv);
    };
    const float v = value(a);
    if (q.sig) q.sig[e] = v;
    q.cen[e] = v - (q.L > 2 ? 0.5f * value(0) + 0.5f * value(q.L - 1) : value(0));  // (k = 1: the one difference itself)
}

// ceil(C / 64) * tiles blocks of 256 threads, and behind them those that build the tables of `q` (prob_table_blocks): the
// two jobs are independent and each is too short to fill the machine on its own.
// PLANES (the hybrid node's forward): the bit-planes a DWN lookup reads leave in the same pass, one ballot per column of the
// tile in the LDS (word (t, c), bit r = src[64 t + r][c] >= 0.5, 0 past the batch).  HBM bound; x used to be read once by the
// lookup's own packing pass and again by the backward's re-tiling.  Hybrid layer 4096 x 16384 -> 8192 nodes of six inputs,
// forward + backward: 718 -> 683 us.
template <bool PLANES = false>
__global__ __launch_bounds__(256) void prob_to_tiles(const float *__restrict__ src, float *__restrict__ dst, int B, int C,
                                                      int tiles, ProbTables q, unsigned long long *__restrict__ planes = nullptr) {
    __shared__ float tile[64][65];  // [column][row]
    const int cols = (C + 63) / 64, t = blockIdx.x / cols, c0 = (int)(blockIdx.x % cols) * 64;
    if (t >= tiles) {
        prob_table_element(q, ((long long)blockIdx.x - (long long)cols * tiles) * 256 + threadIdx.x);
        return;
    }
    if ((C & 3) == 0 && c0 + 64 <= C && (((uintptr_t)src) & 15) == 0) {
#pragma unroll
        for (int pass = 0; pass < 4; ++pass) {
            const int e = pass * 256 + threadIdx.x;
            const int r = e >> 4, c = (e & 15) * 4;
            const int b = t * 64 + r;
            prob_f4 v = {0.0f, 0.0f, 0.0f, 0.0f};
            if (b < B) v = *reinterpret_cast<const prob_f4 *>(src + (size_t)b * C + c0 + c);
            tile[c][r] = v.x; tile[c + 1][r] = v.y; tile[c + 2][r] = v.z; tile[c + 3][r] = v.w;
        }
    } else {
        for (int e = threadIdx.x; e < 4096; e += 256) {
            const int r = e >> 6, c = e & 63;
            const int b = t * 64 + r;
            tile[c][r] = (b < B && c0 + c < C) ? src[(size_t)b * C + c0 + c] : 0.0f;
        }
    }
    __syncthreads();
    if (PLANES) {
        const int lane = threadIdx.x & 63, cw = (threadIdx.x >> 6) * 16;
        unsigned long long mine = 0;
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            const unsigned long long mask = __ballot(tile[cw + q][lane] >= 0.5f);
            mine = lane == q ? mask : mine;
        }
        if (lane < 16 && c0 + cw + lane < C) planes[(size_t)t * C + c0 + cw + lane] = mine;
    }
#pragma unroll
    for (int pass = 0; pass < 4; ++pass) {
        const int e = pass * 256 + threadIdx.x;
        const int c = e >> 4, r = (e & 15) * 4;
        const prob_f4 v = {tile[c][r], tile[c][r + 1], tile[c][r + 2], tile[c][r + 3]};
        if (c0 + c < C) *reinterpret_cast<prob_f4 *>(dst + ((size_t)t * C + c0 + c) * 64 + r) = v;
    }
}

static inline int prob_table_blocks(const ProbTables &q) { return dl_ceil_div((long long)q.N * q.L * q.O, 256); }
template <bool PLANES = false>
static void prob_launch_to_tiles(const char *name, const float *x, float *xT, int B, int I, const ProbTables &q, hipStream_t s,
                                 unsigned long long *planes = nullptr) {
    const int BT = (B + 63) / 64, grid = dl_ceil_div(I, 64) * BT + prob_table_blocks(q);
    DL_TIMED(name, s, (prob_to_tiles<PLANES><<<grid, 256, 0, s>>>(x, xT, B, I, BT, q, planes)));
}

// table of one column as wave-uniform values
template <int K>
__device__ __forceinline__ void prob_load_table(const float *__restrict__ sig, int c, float (&tab)[1 << K]) {
    const float *row = sig + (size_t)c * (1 << K);
#pragma unroll
    for (int a = 0; a < (1 << K); ++a) tab[a] = row[a];
}

#define PROB_TC 128                    // columns per block
#define PROB_FW 8                      // wavefronts per block
#define PROB_WC (PROB_TC / PROB_FW)    // columns per wavefront
template <int K>
__global__ __launch_bounds__(64 * PROB_FW) void prob_fwd_t(const float *__restrict__ xT, const int *__restrict__ idx32,
                                                            const float *__restrict__ sig, float *__restrict__ y,
                                                            int B, int I, int N, int O, int BT) {
    __shared__ float tile[PROB_TC][65];  // [column][row]
    constexpr int L = 1 << K;
    const int NO = N * O;
    int ctile, t;
    if (!dl_xcd_map((NO + PROB_TC - 1) / PROB_TC, BT, ctile, t)) return;
    const int c0 = ctile * PROB_TC;
    const int lane = threadIdx.x & 63;
    const int wave = dl_uniform(threadIdx.x >> 6);
    const int cend = min(PROB_TC, NO - c0);
    const int wbeg = wave * PROB_WC;
    const __amdgpu_buffer_rsrc_t rs_x = __builtin_amdgcn_make_buffer_rsrc((void *)(xT + (size_t)t * I * 64), 0, I * 256, PROB_RSRC);
    const int lane4 = lane * 4;
    // slot s = (column within my 16) * K + j  ->  lane s % 64 of register s / 64: byte offset of the input's row
    constexpr int NIDX = (PROB_WC * K + 63) / 64;
    int myoff[NIDX];
#pragma unroll
    for (int v = 0; v < NIDX; ++v) {
        const int s = v * 64 + lane;
        const int c = min(c0 + wbeg + min(s / K, PROB_WC - 1), NO - 1);
        myoff[v] = idx32[(size_t)(c / O) * K + s % K] * 256;
    }
    constexpr int CG = 4;  // columns whose input rows are requested together
#pragma unroll
    for (int g = 0; g < PROB_WC; g += CG) {
        if (wbeg + g >= cend) break;  // wave-uniform
        float xs[CG][K];
#pragma unroll
        for (int q = 0; q < CG; ++q)
#pragma unroll
            for (int j = 0; j < K; ++j) {
                const int s = (g + q) * K + j;  // compile-time after unrolling
                const int off = __builtin_amdgcn_readlane(myoff[s / 64], s % 64);
                xs[q][j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs_x, lane4, off, 0));
            }
#pragma unroll
        for (int q = 0; q < CG; ++q) {
            const int cc = wbeg + g + q;
            if (cc >= cend) break;  // wave-uniform
            float tab[L];
            prob_load_table<K>(sig, c0 + cc, tab);
            float v[L / 2 > 0 ? L / 2 : 1];
            {
                const float om = 1.0f - xs[q][0];
#pragma unroll
                for (int a = 0; a < L / 2; ++a) v[a] = fmaf(tab[2 * a + 1], xs[q][0], tab[2 * a] * om);
            }
#pragma unroll
            for (int j = 1; j < K; ++j) {
#pragma unroll
                for (int a = 0; a < (L >> (j + 1)); ++a) v[a] = v[2 * a] + xs[q][j] * (v[2 * a + 1] - v[2 * a]);
            }
            tile[cc][lane] = v[0];
        }
    }
    __syncthreads();
    if (cend == PROB_TC && t * 64 + 64 <= B && (NO & 3) == 0 && (((uintptr_t)y) & 15) == 0) {  // whole tile: 16-byte stores
#pragma unroll
        for (int pass = 0; pass < 64 * PROB_TC / 4 / (64 * PROB_FW); ++pass) {
            const int e = pass * 64 * PROB_FW + threadIdx.x;
            const int r = e / (PROB_TC / 4), c4 = (e % (PROB_TC / 4)) * 4;
            const prob_f4 v = {tile[c4][r], tile[c4 + 1][r], tile[c4 + 2][r], tile[c4 + 3][r]};
            __builtin_nontemporal_store(v, reinterpret_cast<prob_f4 *>(&y[(size_t)(t * 64 + r) * NO + c0 + c4]));
        }
        return;
    }
    for (int e = threadIdx.x; e < 64 * PROB_TC; e += 64 * PROB_FW) {
        const int r = e / PROB_TC, cc = e % PROB_TC;
        const int b = t * 64 + r;
        if (b < B && cc < cend) __builtin_nontemporal_store(tile[cc][r], &y[(size_t)b * NO + c0 + cc]);
    }
}

// v q / (q + 1e-8).  The quotient is rounded as a division is: reciprocal, one Newton step, one correction of the quotient by its
// remainder (Markstein); v_div_fixup for a denominator of 0, infinities and NaN.  Beyond 2^100, where the reciprocal is not in
// fp32's normal range, q + 1e-8 is q.  Forward and backward of 4096 x 16384 -> 8192 hybrid nodes of six inputs: 680 us, 688 with the
// division itself, the same bits.
__device__ __forceinline__ float prob_hybrid_scale(float v, float q) {
    const float n = v * q, d = q + PROB_HYBRID_EPS;
    float r = __builtin_amdgcn_rcpf(d);
    r = fmaf(fmaf(-d, r, 1.0f), r, r);
    float t = n * r;
    t = fmaf(fmaf(-d, t, n), r, t);
    t = __builtin_amdgcn_div_fixupf(t, d, n);
    return fabsf(q) > 0x1p100f && fabsf(q) < INFINITY ? v : t;
}
// u[a] = product over the inputs j of (x_j if bit j of a is set, else 1 - x_j)
template <int KH>
__device__ __forceinline__ void prob_products(const float *x, const float *om, float (&u)[1 << KH]) {
    u[0] = 1.0f;
#pragma unroll
    for (int j = 0; j < KH; ++j)
#pragma unroll
        for (int a = (1 << j) - 1; a >= 0; --a) {
            u[a | (1 << j)] = u[a] * x[j];
            u[a] = u[a] * om[j];
        }
}
// dx[j] = d/dx_j of the multilinear interpolation of v at x
template <int KH>
__device__ __forceinline__ void prob_fold_gradient(const float (&v0)[1 << KH], const float *x, const float *om, float *dx) {
    constexpr int L = 1 << KH;
    float diff[L - 1];  // level j occupies [L - (L >> j), L - (L >> (j + 1)))
    float v[L];
#pragma unroll
    for (int a = 0; a < L; ++a) v[a] = v0[a];
    int base = 0;
#pragma unroll
    for (int j = 0; j < KH; ++j) {
#pragma unroll
        for (int a = 0; a < (L >> (j + 1)); ++a) {
            diff[base + a] = v[2 * a + 1] - v[2 * a];
            v[a] = fmaf(x[j], diff[base + a], v[2 * a]);
        }
        base += L >> (j + 1);
    }
    // bar_KH[0] = 1; dx_j = sum_a bar_{j+1}[a] d_j[a]; bar_j[2a] = bar_{j+1}[a] (1 - x_j), bar_j[2a+1] = bar_{j+1}[a] x_j
    float bar[L];
    bar[0] = 1.0f;
#pragma unroll
    for (int j = KH - 1; j >= 0; --j) {
        const int cnt = L >> (j + 1);
        base -= cnt;
        float sum = 0.0f;
#pragma unroll
        for (int a = 0; a < cnt; ++a) sum = fmaf(bar[a], diff[base + a], sum);
        dx[j] = sum;
        if (j > 0) {
#pragma unroll
            for (int a = cnt - 1; a >= 0; --a) {
                const float w = bar[a];
                bar[2 * a + 1] = w * x[j];
                bar[2 * a] = w * om[j];
            }
        }
    }
}

// Sum the 64 per-row partials of every table entry with L - 1 + (6 - K) exchanges instead of 6 L:
// round r pairs the entries (2i, 2i+1); the half of the wavefront with lane bit (5 - r) set keeps
// the odd one and hands over the even one, so after K rounds a lane holds one entry,
// a = sum_r ((lane >> (5 - r)) & 1) << r, summed over the lanes that differ in the top K bits.
template <int K>
__device__ __forceinline__ float prob_sum_lanes(float (&acc)[1 << K], int lane) {
#pragma unroll
    for (int r = 0; r < K; ++r) {
        const int width = 32 >> r;
        const bool upper = (lane & width) != 0;
#pragma unroll
        for (int i = 0; i < ((1 << K) >> (r + 1)); ++i) {
            const float keep = upper ? acc[2 * i + 1] : acc[2 * i];
            const float send = upper ? acc[2 * i] : acc[2 * i + 1];
            acc[i] = keep + __shfl_xor(send, width);
        }
    }
    float mine = acc[0];
#pragma unroll
    for (int width = 32 >> K; width > 0; width >>= 1) mine += __shfl_xor(mine, width);
    return mine;
}
template <int K>
__device__ __forceinline__ int prob_sum_entry(int lane) {
    int a = 0;
#pragma unroll
    for (int r = 0; r < K; ++r) a |= ((lane >> (5 - r)) & 1) << r;
    return a;
}

// The gradient of the mapped inputs is written once and read once.  Where it is too large for the 256 MB behind the L2s to hold it
// beside x and gx, it is written and read, and gx written, past that cache's keeping (STREAM), which leaves it to what is read
// again.  Forward and backward, us, as ordinary accesses / so: hybrid 1024 x 8192 -> 6000 (147 MB) 136 / 133, 2048 x 8192 -> 4096 (201 MB)
// 196 / 176, 2048 x 8192 -> 8192 (403 MB) 335 / 310, 4096 x 16384 -> 8192 (805 MB) 686 / 659; probabilistic 4096 x 16384 -> 8192, k = 4
// (537 MB) 567 / 534.  Smaller ones lose what the gather would have found there: 512 x 6000 -> 8000 (98 MB) 94 / 96.  (A compile-time
// choice: the two stores of a branch become one without the hint.)
static inline bool prob_gm_stream(int B, int N, int k, int O) { return (double)B * N * O * k * sizeof(float) >= 128e6; }
#define PROB_NT 2  // cache policy of a buffer load: read once

// one wavefront per (column, chunk of batch tiles); W wavefronts, i.e. sixteen columns (or four), per block.
// HYB (hybrid node): the table is used as given and the input gradient carries the factor
// q / (q + 1e-8), q = x_j (1 - x_j), of that node's backward.
// The weight of table entry a is a product over the inputs, so it factors into one over the lower KL and one over the upper
// KU inputs, p[lo, hi] = u[lo] w[hi]: with V[lo] = sum_hi T[lo, hi] w[hi] and Z[hi] = sum_lo T[lo, hi] u[lo] the gradients
// of the lower inputs are those of the interpolation of the 2^KL values V, of the upper ones those of Z, and the table
// gradient is g u[lo] w[hi].  Three times 2^k multiply-adds and little else (k = 6: about 280 instructions per column
// and 64 rows where the fold of the whole table and its reverse took 440), and of arrays of 2^k only the table gradient
// stays in registers: sixteen wavefronts of it fit a CU at every k, where the fold left room for eight at k = 6.
// The sums V and Z are of the table less a value of the column's own (cen): they are taken differences of, and with the
// table itself, whose values are about 0.5, gx stood 3.0e-7 from float64 (2-norm; uniform x, k = 6; hybrid 2.2e-7) where the fold
// gave 2.3e-7 (1.7e-7); with cen 1.6e-7 (1.4e-7).
// gy is the row-major gradient itself: the block's 16 columns are 64 contiguous bytes of a row, the 64 x 16 piece of a
// batch tile is fetched one value per thread a tile ahead and turned through the LDS (two buffers, one barrier per tile).
// W = 4 (at most 12 columns): blocks of four columns, so that at most three wavefronts of a block have none, and four
// blocks on a CU.  65536 rows x 8 columns, k = 6: 84 us in blocks of sixteen and at most 16 chunks, 14.5 in blocks of four.
template <int K, bool HYB, int W, bool STREAM>
__global__ __launch_bounds__(64 * W) void prob_bwd_t(const float *__restrict__ xT, const float *__restrict__ gy,
                                                   const int *__restrict__ idx32, const float *__restrict__ cen,
                                                   float *__restrict__ gmT, float *__restrict__ gpart, int I, int N,
                                                   int O, int BT, int tiles_per_chunk, int want_gm, int B) {
    constexpr int L = 1 << K;
    constexpr int KL = K / 2, KU = K - KL, LL = 1 << KL, LU = 1 << KU;
    __shared__ float gturn[2][W][65];  // [buffer][column][row]
    const int NO = N * O;
    const int lane = threadIdx.x & 63;
    const int c_raw = blockIdx.x * W + dl_uniform(threadIdx.x >> 6);
    const bool live = c_raw < NO;        // wavefronts past the last column still serve the barriers
    const int c = live ? c_raw : NO - 1;
    const int chunk = blockIdx.y;
    const int n = c / O;
    const int lane4 = lane * 4;
    int off[K];
#pragma unroll
    for (int j = 0; j < K; ++j) off[j] = idx32[(size_t)n * K + j] * 256;
    float tab[L];
    prob_load_table<K>(cen, c, tab);
    float acc[L];
#pragma unroll
    for (int a = 0; a < L; ++a) acc[a] = 0.0f;
    const int t0 = chunk * tiles_per_chunk, t1 = min(BT, t0 + tiles_per_chunk);
    float nxs[K], ng = 0.0f;  // operands of the next batch tile, requested one tile ahead
    const int trow = threadIdx.x / W, tcol = threadIdx.x % W;  // my value of the 64 x W piece
    auto request = [&](int t) {
        const __amdgpu_buffer_rsrc_t rs_x = __builtin_amdgcn_make_buffer_rsrc((void *)(xT + (size_t)t * I * 64), 0, I * 256, PROB_RSRC);
#pragma unroll
        for (int j = 0; j < K; ++j) nxs[j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs_x, lane4, off[j], 0));
        const int b = t * 64 + trow, cc = blockIdx.x * W + tcol;
        ng = (b < B && cc < NO) ? gy[(size_t)b * NO + cc] : 0.0f;
    };
    if (t0 < t1) request(t0);
    for (int t = t0; t < t1; ++t) {
        float xs[K], om[K];
#pragma unroll
        for (int j = 0; j < K; ++j) { xs[j] = nxs[j]; om[j] = 1.0f - nxs[j]; }
        const int buf = (t - t0) & 1;
        gturn[buf][tcol][trow] = ng;
        __syncthreads();  // the other buffer is rewritten only after the next barrier: its readers are done by then
        const float g = gturn[buf][threadIdx.x >> 6][lane];
        if (t + 1 < t1) request(t + 1);
        float u[LL], w[LU], dx[K];
        prob_products<KL>(xs, om, u);
        prob_products<KU>(xs + KL, om + KL, w);
        if (want_gm) {
            if constexpr (KL > 0) {
                float V[LL];
#pragma unroll
                for (int lo = 0; lo < LL; ++lo) {
                    V[lo] = tab[lo] * w[0];
#pragma unroll
                    for (int hi = 1; hi < LU; ++hi) V[lo] = fmaf(tab[lo | (hi << KL)], w[hi], V[lo]);
                }
                prob_fold_gradient<KL>(V, xs, om, dx);
            }
            float Z[LU];
#pragma unroll
            for (int hi = 0; hi < LU; ++hi) {
                Z[hi] = tab[hi << KL] * u[0];
#pragma unroll
                for (int lo = 1; lo < LL; ++lo) Z[hi] = fmaf(tab[lo | (hi << KL)], u[lo], Z[hi]);
            }
            prob_fold_gradient<KU>(Z, xs + KL, om + KL, dx + KL);
            if (HYB) {
#pragma unroll
                for (int j = 0; j < K; ++j) {
                    const float q = xs[j] * om[j];
                    dx[j] = prob_hybrid_scale(dx[j], q);
                }
            }
            if (live) {
#pragma unroll
                for (int j = 0; j < K; ++j) {
                    float *at = &gmT[(((size_t)t * NO + c) * K + j) * 64 + lane];
                    if constexpr (STREAM) __builtin_nontemporal_store(g * dx[j], at);
                    else *at = g * dx[j];
                }
            }
        }
#pragma unroll
        for (int lo = 0; lo < LL; ++lo) {
            const float gu = g * u[lo];
#pragma unroll
            for (int hi = 0; hi < LU; ++hi) acc[lo | (hi << KL)] = fmaf(gu, w[hi], acc[lo | (hi << KL)]);
        }
    }
    const float mine = prob_sum_lanes<K>(acc, lane);
    if (live && (lane & ((64 >> K) - 1)) == 0) gpart[((size_t)chunk * NO + c) * L + prob_sum_entry<K>(lane)] = mine;
}

// ---------------------------------------------------------------------------------
// Nodes that read their inputs in order: node n has columns n K .. n K + K - 1 of x [B][N K], one output (what a learned mapping
// hands its nodes).  Sixteen nodes are then 16 K consecutive values of a row, so x and the gradient of x are read and written
// as they lie: no re-tiling of x, no tiled gradient, no gather.  A block is sixteen wavefronts, one per node, and walks the
// batch tiles of a chunk: the 64 x 16 K piece of a tile comes a tile ahead through registers into the LDS (odd stride: a lane's row
// lies on a bank of its own), a wavefront has its K columns and its table in registers, results leave through the LDS, one barrier
// per tile.  The backward writes the gradient over the inputs that it has read, so three pieces take turns: one being
// filled, one in use, one being stored.  Arithmetic and its order are those of prob_fwd_t and prob_bwd_t.
// Bound by HBM forward (x and y once), by vector arithmetic backward.
// 512 x 48000 -> 8000 nodes of six inputs: forward 30 us, backward 62, 3.8 and 3.4 TB/s; re-tiled, two and two launches, 63 and 93.
// The learnable layer's step 1022 -> 951 us with bf16 operands, 2027 -> 1957 with fp32.
#define PROB_ON 16  // nodes per block
// W: values per access, as many as the width of x and the alignment allow.  Accesses go through a buffer descriptor of the
// tile's rows that the batch has (rows past it lie past its end: zeros, nothing stored), with one byte offset per access for all
// tiles, of x and of its gradient.
template <int W>
struct ProbWide;
template <>
struct ProbWide<4> { typedef unsigned type __attribute__((ext_vector_type(4))); };
template <>
struct ProbWide<2> { typedef unsigned type __attribute__((ext_vector_type(2))); };
template <int K, int W>
struct ProbPiece {  // my share of the 64 x 16 K piece of a batch tile
    static constexpr int S = PROB_ON * K + 1, PER_ROW = PROB_ON * K / W, COUNT = 64 * PER_ROW;
    static constexpr int PASSES = (COUNT + 64 * PROB_ON - 1) / (64 * PROB_ON);
    static constexpr unsigned NOWHERE = 0x80000000u;  // past the end of every descriptor: 64 rows of less than 2^23 values
    unsigned off[PASSES];
    float v[PASSES][W];
    static __device__ __forceinline__ int element(int p) { return p * 64 * PROB_ON + (int)threadIdx.x; }
    __device__ __forceinline__ void place(int M, int cols) {
#pragma unroll
        for (int p = 0; p < PASSES; ++p) {
            const int row = element(p) / PER_ROW, col = element(p) % PER_ROW * W;
            off[p] = element(p) < COUNT && col < cols ? (unsigned)(row * M + col) * 4u : NOWHERE;
        }
    }
    // at: column c0 of the tile's first row
    static __device__ __forceinline__ __amdgpu_buffer_rsrc_t tile(const float *at, int M, int c0, int rows) {
        return __builtin_amdgcn_make_buffer_rsrc((void *)at, 0, (unsigned)(min(rows, 64) * M - c0) * 4u, PROB_RSRC);
    }
    __device__ __forceinline__ void request(__amdgpu_buffer_rsrc_t r) {
#pragma unroll
        for (int p = 0; p < PASSES; ++p) {
            if constexpr (W == 4) {
                const typename ProbWide<4>::type q = __builtin_amdgcn_raw_buffer_load_b128(r, off[p], 0, 0);
#pragma unroll
                for (int w = 0; w < 4; ++w) v[p][w] = __uint_as_float(q[w]);
            } else if constexpr (W == 2) {
                const typename ProbWide<2>::type q = __builtin_amdgcn_raw_buffer_load_b64(r, off[p], 0, 0);
                v[p][0] = __uint_as_float(q[0]); v[p][1] = __uint_as_float(q[1]);
            } else {
                v[p][0] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off[p], 0, 0));
            }
        }
    }
    __device__ __forceinline__ void put(float (*piece)[S]) const {
#pragma unroll
        for (int p = 0; p < PASSES; ++p)
            if (COUNT % (64 * PROB_ON) == 0 || element(p) < COUNT) {
#pragma unroll
                for (int w = 0; w < W; ++w) piece[element(p) / PER_ROW][element(p) % PER_ROW * W + w] = v[p][w];
            }
    }
    __device__ __forceinline__ void store(float (*piece)[S], __amdgpu_buffer_rsrc_t r) const {
#pragma unroll
        for (int p = 0; p < PASSES; ++p) {
            if (COUNT % (64 * PROB_ON) != 0 && element(p) >= COUNT) continue;
            const float *from = &piece[element(p) / PER_ROW][element(p) % PER_ROW * W];
            if constexpr (W == 4) {
                const typename ProbWide<4>::type q = {__float_as_uint(from[0]), __float_as_uint(from[1]), __float_as_uint(from[2]), __float_as_uint(from[3])};
                __builtin_amdgcn_raw_buffer_store_b128(q, r, off[p], 0, 0);
            } else if constexpr (W == 2) {
                const typename ProbWide<2>::type q = {__float_as_uint(from[0]), __float_as_uint(from[1])};
                __builtin_amdgcn_raw_buffer_store_b64(q, r, off[p], 0, 0);
            } else {
                __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(*from), r, off[p], 0, 0);
            }
        }
    }
};
// a value of every lane below L as wave-uniform ones
template <int L>
__device__ __forceinline__ void prob_spread(float mine, float (&all)[L]) {
#pragma unroll
    for (int a = 0; a < L; ++a) all[a] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(mine), a));
}

template <int K, int W>
__global__ __launch_bounds__(64 * PROB_ON, 8) void prob_ordered_fwd(const float *__restrict__ x, const float *__restrict__ raw,
                                                                  ProbTemp T, float *__restrict__ sig, float *__restrict__ y, int B,
                                                                  int N, int BT, int tiles_per_chunk) {
    constexpr int L = 1 << K;
    typedef ProbPiece<K, W> Piece;
    __shared__ float xt[2][64][Piece::S], yt[2][64][PROB_ON + 1];
    const int lane = threadIdx.x & 63, wave = dl_uniform(threadIdx.x >> 6);
    const int n0 = blockIdx.x * PROB_ON, n = n0 + wave, M = N * K, cols = min(PROB_ON * K, M - n0 * K);
    const bool live = n < N;
    float tab[L];
    {
        float s = 0.0f;
        if (live && lane < L) {
            s = dl_sigmoid(raw[(size_t)n * L + lane] * prob_inv_t_of(T, n));
            if (blockIdx.y == 0) sig[(size_t)n * L + lane] = s;
        }
        prob_spread<L>(s, tab);
    }
    const int t0 = blockIdx.y * tiles_per_chunk, t1 = min(BT, t0 + tiles_per_chunk);
    Piece next;
    next.place(M, cols);
    auto request = [&](int t) { next.request(Piece::tile(x + (size_t)t * 64 * M + n0 * K, M, n0 * K, B - t * 64)); };
    const int yr = threadIdx.x / PROB_ON, yc = threadIdx.x % PROB_ON;
    auto store = [&](int t, int buf) {
        if (t * 64 + yr < B && n0 + yc < N) y[(size_t)(t * 64 + yr) * N + n0 + yc] = yt[buf][yr][yc];
    };
    request(t0);
    int buf = 0;
    for (int t = t0; t < t1; ++t, buf ^= 1) {
        next.put(xt[buf]);
        __syncthreads();  // (the other piece and the other yt are written again only after the next one)
        if (t + 1 < t1) request(t + 1);
        if (t > t0) store(t - 1, buf ^ 1);
        float xs[K];
#pragma unroll
        for (int j = 0; j < K; ++j) xs[j] = xt[buf][lane][wave * K + j];
        float v[L / 2 > 0 ? L / 2 : 1];
        {
            const float om = 1.0f - xs[0];
#pragma unroll
            for (int a = 0; a < L / 2; ++a) v[a] = fmaf(tab[2 * a + 1], xs[0], tab[2 * a] * om);
        }
#pragma unroll
        for (int j = 1; j < K; ++j) {
#pragma unroll
            for (int a = 0; a < (L >> (j + 1)); ++a) v[a] = v[2 * a] + xs[j] * (v[2 * a + 1] - v[2 * a]);
        }
        yt[buf][lane][wave] = v[0];
    }
    __syncthreads();
    store(t1 - 1, buf ^ 1);
}

// gpart: as prob_bwd_t leaves it, or null where the block has the whole batch: it then writes graw itself
template <int K, int W>
__global__ __launch_bounds__(64 * PROB_ON) void prob_ordered_bwd(const float *__restrict__ x, const float *__restrict__ gy,
                                                                  const float *__restrict__ sig, ProbTemp T, float *__restrict__ gx,
                                                                  float *__restrict__ gpart, float *__restrict__ graw, int B, int N,
                                                                  int BT, int tiles_per_chunk) {
    constexpr int L = 1 << K;
    constexpr int KL = K / 2, KU = K - KL, LL = 1 << KL, LU = 1 << KU;
    typedef ProbPiece<K, W> Piece;
    __shared__ float xt[3][64][Piece::S], gturn[2][PROB_ON][65];
    const int lane = threadIdx.x & 63, wave = dl_uniform(threadIdx.x >> 6);
    const int n0 = blockIdx.x * PROB_ON, n = n0 + wave, M = N * K, cols = min(PROB_ON * K, M - n0 * K);
    const bool live = n < N;
    float tab[L];  // the table less a value of its own (prob_table_element)
    {
        const float s = live && lane < L ? sig[(size_t)n * L + lane] : 0.0f;
        const float first = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(s), 0)),
                    last = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(s), L - 1));
        prob_spread<L>(s - (L > 2 ? 0.5f * first + 0.5f * last : first), tab);
    }
    float acc[L];
#pragma unroll
    for (int a = 0; a < L; ++a) acc[a] = 0.0f;
    const int t0 = blockIdx.y * tiles_per_chunk, t1 = min(BT, t0 + tiles_per_chunk);
    Piece next;
    next.place(M, cols);
    float ng = 0.0f;
    const int trow = threadIdx.x / PROB_ON, tcol = threadIdx.x % PROB_ON;
    auto request = [&](int t) {
        next.request(Piece::tile(x + (size_t)t * 64 * M + n0 * K, M, n0 * K, B - t * 64));
        const int b = t * 64 + trow;
        ng = (b < B && n0 + tcol < N) ? gy[(size_t)b * N + n0 + tcol] : 0.0f;
    };
    auto store = [&](int t, int piece) { next.store(xt[piece], Piece::tile(gx + (size_t)t * 64 * M + n0 * K, M, n0 * K, B - t * 64)); };
    request(t0);
    int piece = 0, before = 2;
    for (int t = t0; t < t1; ++t) {
        const int buf = (t - t0) & 1;
        next.put(xt[piece]);
        gturn[buf][tcol][trow] = ng;
        __syncthreads();  // this piece is filled, the one before holds its gradient, the third has been stored
        if (t + 1 < t1) request(t + 1);
        if (gx && t > t0) store(t - 1, before);
        float xs[K], om[K];
#pragma unroll
        for (int j = 0; j < K; ++j) { xs[j] = xt[piece][lane][wave * K + j]; om[j] = 1.0f - xs[j]; }
        const float g = gturn[buf][wave][lane];
        float u[LL], w[LU], dx[K];
        prob_products<KL>(xs, om, u);
        prob_products<KU>(xs + KL, om + KL, w);
        if (gx) {
            if constexpr (KL > 0) {
                float V[LL];
#pragma unroll
                for (int lo = 0; lo < LL; ++lo) {
                    V[lo] = tab[lo] * w[0];
#pragma unroll
                    for (int hi = 1; hi < LU; ++hi) V[lo] = fmaf(tab[lo | (hi << KL)], w[hi], V[lo]);
                }
                prob_fold_gradient<KL>(V, xs, om, dx);
            }
            float Z[LU];
#pragma unroll
            for (int hi = 0; hi < LU; ++hi) {
                Z[hi] = tab[hi << KL] * u[0];
#pragma unroll
                for (int lo = 1; lo < LL; ++lo) Z[hi] = fmaf(tab[lo | (hi << KL)], u[lo], Z[hi]);
            }
            prob_fold_gradient<KU>(Z, xs + KL, om + KL, dx + KL);
#pragma unroll
            for (int j = 0; j < K; ++j) xt[piece][lane][wave * K + j] = g * dx[j];
        }
#pragma unroll
        for (int lo = 0; lo < LL; ++lo) {
            const float gu = g * u[lo];
#pragma unroll
            for (int hi = 0; hi < LU; ++hi) acc[lo | (hi << KL)] = fmaf(gu, w[hi], acc[lo | (hi << KL)]);
        }
        before = piece;
        piece = piece == 2 ? 0 : piece + 1;
    }
    if (gx) {
        __syncthreads();
        store(t1 - 1, before);
    }
    const float mine = prob_sum_lanes<K>(acc, lane);
    const int a = prob_sum_entry<K>(lane);
    if (!live || (lane & ((64 >> K) - 1)) != 0) return;
    if (gpart) {
        gpart[((size_t)blockIdx.y * N + n) * L + a] = mine;
    } else {
        const float s = sig[(size_t)n * L + a];
        graw[(size_t)n * L + a] = mine * s * (1.0f - s) * prob_inv_t_of(T, n);
    }
}

// graw[n,a,d] = sigmoid'(w/T)/T * sum over chunks of gpart[chunk][c][a];
// sig == null (hybrid node): the plain sum, kept in the table's own layout [c][a]
struct ProbReduce {  // the table-gradient reduction, also carried as extra blocks of the gather launch
    const float *gpart, *sig;
    ProbTemp T;
    float *graw;
    int N, L, O, chunks;
    bool flat = false;  // hybrid: the gradient of what the table is the sigmoid of, in the table's own layout
};
__device__ __forceinline__ void prob_reduce_element(const ProbReduce &R, long long e);
__global__ __launch_bounds__(256) void prob_reduce_weights(ProbReduce R) {
    prob_reduce_element(R, (long long)blockIdx.x * 256 + threadIdx.x);
}
__device__ __forceinline__ void prob_reduce_element(const ProbReduce &R, long long e) {
    const float *gpart = R.gpart, *sig = R.sig;
    float *graw = R.graw;
    const int N = R.N, L = R.L, O = R.O, chunks = R.chunks;
    const long long total = (long long)N * L * O;
    if (e >= total) return;
    float acc = 0.0f;
    int ch = 0;
    for (; ch + 8 <= chunks; ch += 8) {  // eight loads in flight, added in chunk order (one at a time: 0.2 us a chunk)
        float part[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) part[q] = gpart[(size_t)(ch + q) * total + e];
#pragma unroll
        for (int q = 0; q < 8; ++q) acc += part[q];
    }
    for (; ch < chunks; ++ch) acc += gpart[(size_t)ch * total + e];
    if (!sig) {
        graw[e] = acc;
        return;
    }
    const float s = sig[e];
    if (R.flat) {
        graw[e] = acc * s * (1.0f - s);
        return;
    }
    const int a = (int)(e % L);
    const long long c = e / L;
    const int n = (int)(c / O), d = (int)(c % O);
    graw[((size_t)n * L + a) * O + d] = acc * s * (1.0f - s) * prob_inv_t_of(R.T, n);
}

#define PROB_IS 64  // inputs per block of the gather
#define PROB_WI 16  // inputs per wavefront
#define PROB_EG 8   // entries requested together
// FAST (one output per node): the CSR entries of a wavefront's 16 inputs are held one per lane
// (row offset, local input) and replayed eight at a time with buffer loads whose offset travels
// in an SGPR, the next eight requested before the current ones are summed.
template <bool FAST, bool STREAM>
__global__ __launch_bounds__(256) void prob_gather_t(const float *__restrict__ gmT, const int *__restrict__ inv_ptr,
                                                      const int *__restrict__ inv_pos, float *__restrict__ gx, int B,
                                                      int I, int N, int K, int O, int BT, int gather_blocks, ProbReduce R) {
    __shared__ float tile[PROB_IS][65];  // [input][row]
    if ((int)blockIdx.x >= gather_blocks) {  // the blocks appended for the independent table-gradient reduction
        prob_reduce_element(R, (long long)(blockIdx.x - gather_blocks) * 256 + threadIdx.x);
        return;
    }
    int slab, t;
    if (!dl_xcd_map((I + PROB_IS - 1) / PROB_IS, BT, slab, t)) return;
    const int i0 = slab * PROB_IS;
    const int lane = threadIdx.x & 63;
    const int wave = dl_uniform(threadIdx.x >> 6);
    const int iend = min(PROB_IS, I - i0);
    const int wbeg = wave * PROB_WI;
    if (FAST) {
        const __amdgpu_buffer_rsrc_t rs =
            __builtin_amdgcn_make_buffer_rsrc((void *)(gmT + (size_t)t * N * K * 64), 0, N * K * 256, PROB_RSRC);
        const int lane4 = lane * 4;
        const int myptr = inv_ptr[min(i0 + wbeg + min(lane, PROB_WI), I)];
#pragma unroll
        for (int r = 0; r < PROB_WI; ++r) tile[wbeg + r][lane] = 0.0f;  // inputs nobody reads keep 0
        const int ebeg = __builtin_amdgcn_readlane(myptr, 0);
        const int eend = __builtin_amdgcn_readlane(myptr, PROB_WI);
        float acc = 0.0f;
        int cur = -1;
        for (int base = ebeg; base < eend; base += 64) {
            const int e = base + lane;
            const bool valid = e < eend;
            const int p = valid ? inv_pos[e] : 0;
            int ii = 0;  // local input of entry e
#pragma unroll
            for (int l = 1; l <= PROB_WI; ++l) ii += (__builtin_amdgcn_readlane(myptr, l) <= e) ? 1 : 0;
            const int rec = valid ? ((p << 8) | ii) : 0;  // row offset p * 256 in the upper bits
            const int cnt = min(64, eend - base);
            struct Group { int r[PROB_EG]; float g[PROB_EG]; };
            auto request = [&](int s0, Group &G) {
#pragma unroll
                for (int q = 0; q < PROB_EG; ++q) {
                    const int r = __builtin_amdgcn_readlane(rec, s0 + q);
                    G.r[q] = r;
                    G.g[q] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, lane4, r & ~255, STREAM ? PROB_NT : 0));
                }
            };
            auto sum_up = [&](const Group &G, int s0) {
#pragma unroll
                for (int q = 0; q < PROB_EG; ++q) {
                    if (s0 + q >= cnt) break;  // wave-uniform
                    const int ri = G.r[q] & 31;
                    if (ri != cur) {
                        if (cur >= 0) tile[wbeg + cur][lane] = acc;
                        acc = 0.0f;
                        cur = ri;
                    }
                    acc += G.g[q];
                }
            };
            const int m = (cnt + PROB_EG - 1) / PROB_EG;
            Group A, Bq;
            request(0, A);
            int gi = 0;
            for (; gi + 2 < m; gi += 2) {
                request((gi + 1) * PROB_EG, Bq);
                sum_up(A, gi * PROB_EG);
                request((gi + 2) * PROB_EG, A);
                sum_up(Bq, (gi + 1) * PROB_EG);
            }
            if (gi + 1 < m) {
                request((gi + 1) * PROB_EG, Bq);
                sum_up(A, gi * PROB_EG);
                sum_up(Bq, (gi + 1) * PROB_EG);
            } else {
                sum_up(A, gi * PROB_EG);
            }
        }
        if (cur >= 0) tile[wbeg + cur][lane] = acc;
    } else {
        const float *slabT = gmT + (size_t)t * N * O * K * 64 + lane;
        for (int r = 0; r < PROB_WI; ++r) {
            const int i = i0 + wbeg + r;
            float acc = 0.0f;
            if (i < I) {
                const int e0 = inv_ptr[i], e1 = inv_ptr[i + 1];  // wave-uniform
                for (int e = e0; e < e1; ++e) {
                    const int p = inv_pos[e];
                    const int n = p / K, j = p - n * K;
                    for (int d = 0; d < O; ++d) acc += slabT[(((size_t)n * O + d) * K + j) * 64];
                }
            }
            tile[wbeg + r][lane] = acc;
        }
    }
    __syncthreads();
    if (iend == PROB_IS && (I & 3) == 0 && ((uintptr_t)gx & 15) == 0) {
#pragma unroll
        for (int pass = 0; pass < 4; ++pass) {
            const int e = pass * 256 + threadIdx.x;
            const int r = e / (PROB_IS / 4), i4 = (e % (PROB_IS / 4)) * 4;
            const int b = t * 64 + r;
            const prob_f4 v = {tile[i4][r], tile[i4 + 1][r], tile[i4 + 2][r], tile[i4 + 3][r]};
            if (b >= B) continue;
            prob_f4 *at = reinterpret_cast<prob_f4 *>(&gx[(size_t)b * I + i0 + i4]);
            if constexpr (STREAM) __builtin_nontemporal_store(v, at);
            else *at = v;
        }
    } else {
        for (int e = threadIdx.x; e < 64 * PROB_IS; e += 256) {
            const int r = e / PROB_IS, ii = e % PROB_IS;
            const int b = t * 64 + r;
            if (b < B && ii < iend) gx[(size_t)b * I + i0 + ii] = tile[ii][r];
        }
    }
}

// the gather and the reduction of the table-gradient partials do not depend on each other: one launch, the
// reduction as extra blocks behind the gather's
static void prob_launch_gather_and_reduce(const float *gmT, const int *inv_ptr, const int *inv_pos, float *gx, int B, int I,
                                          int N, int k, int O, int BT, const ProbReduce &R, long long WT, hipStream_t s) {
    const int rblocks = dl_ceil_div(WT, 256);
    if (!gx) {
        DL_TIMED("prob_reduce_weights", s, (prob_reduce_weights<<<rblocks, 256, 0, s>>>(R)));
        return;
    }
    const int gblocks = dl_xcd_grid(dl_ceil_div(I, PROB_IS), BT);
#define GATHER(FAST, STREAM)                                                                                                  \
    DL_TIMED("prob_gather_t+reduce", s, (prob_gather_t<FAST, STREAM><<<gblocks + rblocks, 256, 0, s>>>(gmT, inv_ptr, inv_pos, gx, B, I, \
                                                                                                       N, k, O, BT, gblocks, R)))
    if (O != 1) GATHER(false, false);
    else if (prob_gm_stream(B, N, k, O)) GATHER(true, true);
    else GATHER(true, false);
#undef GATHER
}

// ---------------------------------------------------------------------------------
// Generic kernels, any k up to DL_MAX_K.
__global__ __launch_bounds__(256) void prob_generic_fwd(const float *__restrict__ x, const int *__restrict__ idx32,
                                                         const float *__restrict__ raw, ProbTemp T, float *__restrict__ y,
                                                         int B, int I, int N, int K, int O) {
    const long long gid = (long long)blockIdx.x * 256 + threadIdx.x;
    const long long NO = (long long)N * O;
    if (gid >= (long long)B * NO) return;
    const int b = (int)(gid / NO);
    const int n = (int)((gid % NO) / O), d = (int)((gid % NO) % O);
    const float inv_t = prob_inv_t_of(T, n);
    float xs[DL_MAX_K];
    for (int j = 0; j < K; ++j) xs[j] = x[(size_t)b * I + idx32[(size_t)n * K + j]];
    const int L = 1 << K;
    float acc = 0.0f;
    for (int a = 0; a < L; ++a) {
        float p = 1.0f;
        for (int j = 0; j < K; ++j) p *= ((a >> j) & 1) ? xs[j] : 1.0f - xs[j];
        acc += dl_sigmoid(raw[((size_t)n * L + a) * O + d] * inv_t) * p;
    }
    y[gid] = acc;
}

// hybrid: `raw` is the table itself in the layout [n][d][a] and the input gradient carries q / (q + 1e-8)
__global__ __launch_bounds__(256) void prob_generic_bwd(const float *__restrict__ x, const int *__restrict__ idx32,
                                                         const float *__restrict__ raw, ProbTemp T,
                                                         const float *__restrict__ gy, float *__restrict__ gx,
                                                         float *__restrict__ graw, int B, int I, int N, int K, int O,
                                                         int hybrid) {
    const long long gid = (long long)blockIdx.x * 256 + threadIdx.x;
    if (gid >= (long long)B * N) return;
    const int b = (int)(gid / N), n = (int)(gid % N);
    const float inv_t = prob_inv_t_of(T, n);
    float xs[DL_MAX_K], gxs[DL_MAX_K];
    for (int j = 0; j < K; ++j) { xs[j] = x[(size_t)b * I + idx32[(size_t)n * K + j]]; gxs[j] = 0.0f; }
    const int L = 1 << K;
    for (int d = 0; d < O; ++d) {
        const float g = gy[((size_t)b * N + n) * O + d];
        for (int a = 0; a < L; ++a) {
            const size_t w = hybrid ? ((size_t)n * O + d) * L + a : ((size_t)n * L + a) * O + d;
            const float s = hybrid ? raw[w] : dl_sigmoid(raw[w] * inv_t);
            float p = 1.0f;
            for (int j = 0; j < K; ++j) p *= ((a >> j) & 1) ? xs[j] : 1.0f - xs[j];
            atomicAdd(&graw[w], hybrid ? g * p : g * p * s * (1.0f - s) * inv_t);
            if (gx) {
                for (int j = 0; j < K; ++j) {
                    float q = 1.0f;
                    for (int m = 0; m < K; ++m)
                        if (m != j) q *= ((a >> m) & 1) ? xs[m] : 1.0f - xs[m];
                    gxs[j] += g * s * (((a >> j) & 1) ? q : -q);
                }
            }
        }
    }
    if (gx)
        for (int j = 0; j < K; ++j) {
            const float q = xs[j] * (1.0f - xs[j]);
            atomicAdd(&gx[(size_t)b * I + idx32[(size_t)n * K + j]], hybrid ? gxs[j] * q / (q + PROB_HYBRID_EPS) : gxs[j]);
        }
}

__global__ __launch_bounds__(256) void prob_eval_kernel(const float *__restrict__ x, const int *__restrict__ idx32,
                                                         const float *__restrict__ raw, ProbTemp T, float *__restrict__ y,
                                                         int B, int I, int N, int K, int O) {
    const long long gid = (long long)blockIdx.x * 256 + threadIdx.x;
    const long long NO = (long long)N * O;
    if (gid >= (long long)B * NO) return;
    const int b = (int)(gid / NO);
    const int n = (int)((gid % NO) / O), d = (int)((gid % NO) % O);
    const float inv_t = prob_inv_t_of(T, n);
    float s = 0.0f;
    for (int j = 0; j < K; ++j) s += x[(size_t)b * I + idx32[(size_t)n * K + j]] * (float)(1 << j);
    long long a = (long long)s;
    const int L = 1 << K;
    a = a < 0 ? 0 : (a > L - 1 ? L - 1 : a);
    y[gid] = dl_sigmoid(raw[((size_t)n * L + a) * O + d] * inv_t) >= 0.5f ? 1.0f : 0.0f;
}

__global__ __launch_bounds__(256) void prob_fill_zero(float *p, long long n) {
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i < n) p[i] = 0.0f;
}

// ---------------------------------------------------------------------------------
static int prob_check(int B, int I, int N, int k, int O) {
    if (B <= 0 || I <= 0 || N <= 0 || k <= 0 || O <= 0) return DL_ERR_SHAPE;
    if (k > DL_MAX_K) return DL_ERR_UNSUPPORTED;
    if (B > 4000000) return DL_ERR_UNSUPPORTED;  // batch tiles ride in grid.y (at most 65535 of them, extra rows included)
    return DL_OK;
}
// the tiled path addresses a batch tile of xT with 32-bit byte offsets (input * 256)
static inline bool prob_fast(int I, int N, int k, int O) {
    return k <= DL_MAX_FAST_K && I < (1 << 23) && (long long)N * O * k < (1 << 23);
}
// temperature.clamp(min=1e-6); with a per-node array the kernels take every node's own value
static inline ProbTemp prob_temp(float t, const float *t_n) { return ProbTemp{1.0f / (t > 1e-6f ? t : 1e-6f), t_n}; }
static inline int prob_bt(int B) { return (B + 63) / 64; }
static inline int prob_block_columns(long long NO) { return NO <= 12 ? 4 : 16; }
// Batch tiles per wavefront of prob_bwd_t.  Its blocks (16 or 4 columns x one chunk of tiles) share 256 CUs of 16 wavefronts:
// the fullest CU has so many rounds of them, a block spends about 2 (k <= 4), 4 or 6 (k = 6) tiles' time on its table and
// its sums over the lanes, and the sum over the chunks costs a twentieth of a tile's time each.  2000 x 3001 -> 5003 hybrid
// nodes of 4 inputs (313 blocks a chunk): one chunk 82 us, four 64; 1024 x 4096 -> 4096 nodes, where one chunk is 256 blocks,
// keep it (k = 5: 31.7 against 34.7 in more).  Few columns over many rows, with at most 16 chunks / as here, kernel and
// gather with the sum, us: 147456 rows x 32 columns, k = 6 243 + 42 / 52 + 46, k = 4 144 + 27 / 37 + 29; 65536 rows x 1 column, k = 6
// 67 + 7 / 11 + 11, x 64 columns, k = 4 57 + 17 / 26 + 17.
static inline int prob_tiles_per_chunk_of(int BT, long long columns, int W, int own) {
    const int resident = 256 * 16 / W;
    const long long blocks = dl_ceil_div(columns, W);
    int best = BT;
    double best_cost = 0.0;
    auto consider = [&](long long c) {
        if (c < 1 || c > BT) return;
        const int tpc = dl_ceil_div(BT, c), chunks = dl_ceil_div(BT, tpc);
        const long long all = blocks * chunks;
        const double cost = (all > resident ? (double)dl_ceil_div(all, resident) : 1.1) * (tpc + own) + 0.05 * chunks;
        if (best_cost == 0.0 || cost < best_cost) { best = tpc; best_cost = cost; }
    };
    for (int c = 1; c <= 16; ++c) consider(c);
    for (int c = 20; c <= BT; c += c / 4) consider(c);
    for (int rounds = 1; rounds <= 4; ++rounds) consider(rounds * resident / blocks);  // no CU idle in the last round
    return best;
}
static inline int prob_bwd_own_tiles(int k) { return k >= 6 ? 6 : (k == 5 ? 4 : 2); }
static inline int prob_tiles_per_chunk(int B, int N, int k, int O) {
    return prob_tiles_per_chunk_of(prob_bt(B), (long long)N * O, prob_block_columns((long long)N * O), prob_bwd_own_tiles(k));
}
static inline size_t prob_sig_bytes(int N, int k, int O) { return dl_align256((size_t)N * O * ((size_t)1 << k) * sizeof(float)); }
static inline size_t prob_xT_bytes(int B, int I) { return dl_align256((size_t)prob_bt(B) * I * 64 * sizeof(float)); }

// what the forward leaves for the backward: the sigmoid table, the re-tiled input and the table less a value per column
extern "C" size_t dl_prob_saved_bytes(int B, int I, int N, int k, int O) {
    if (B <= 0 || I <= 0 || N <= 0 || k <= 0 || O <= 0 || !prob_fast(I, N, k, O)) return 256;
    return 2 * prob_sig_bytes(N, k, O) + prob_xT_bytes(B, I);
}
// dL/d(mapped inputs) and the partial table gradients
static inline size_t prob_gm_bytes(int B, int N, int k, int O) {
    const size_t BT = prob_bt(B);
    const int chunks = dl_ceil_div(prob_bt(B), prob_tiles_per_chunk(B, N, k, O));
    return dl_align256(BT * N * O * k * 64 * sizeof(float)) + dl_align256((size_t)chunks * N * O * ((size_t)1 << k) * sizeof(float));
}
// of a backward that is handed what the forward left
extern "C" size_t dl_prob_bwd_saved_workspace_bytes(int B, int I, int N, int k, int O) {
    if (B <= 0 || I <= 0 || N <= 0 || k <= 0 || O <= 0 || !prob_fast(I, N, k, O)) return 256;
    return prob_gm_bytes(B, N, k, O);
}
// of one that makes it itself, with room for a whole [B, N O] array in the place of the table less a value per column
extern "C" size_t dl_prob_bwd_workspace_bytes(int B, int I, int N, int k, int O) {
    if (B <= 0 || I <= 0 || N <= 0 || k <= 0 || O <= 0 || !prob_fast(I, N, k, O)) return 256;
    return prob_sig_bytes(N, k, O) + prob_xT_bytes(B, I) + dl_align256((size_t)prob_bt(B) * N * O * 64 * sizeof(float)) +
           prob_gm_bytes(B, N, k, O);
}

#define PROB_DISPATCH(K, CALL) \
    switch (K) {               \
        case 1: CALL(1); break; case 2: CALL(2); break; case 3: CALL(3); break; \
        case 4: CALL(4); break; case 5: CALL(5); break; default: CALL(6); break; \
    }

static int prob_forward(const float *x, const int32_t *idx32, const float *raw_w, ProbTemp inv_t, float *y, void *saved,
                        size_t saved_bytes, int B, int I, int N, int k, int O, void *stream) {
    if (!x || !idx32 || !raw_w || !y) return DL_ERR_NULL;
    int rc = prob_check(B, I, N, k, O);
    if (rc) return rc;
    hipStream_t s = (hipStream_t)stream;
    if (!prob_fast(I, N, k, O)) {
        DL_TIMED("prob_generic_fwd", s, (prob_generic_fwd<<<dl_ceil_div((long long)B * N * O, 256), 256, 0, s>>>(x, idx32, raw_w, inv_t, y, B, I, N, k, O)));
        return dl_launch_status();
    }
    if (!saved) return DL_ERR_NULL;
    if (saved_bytes < dl_prob_saved_bytes(B, I, N, k, O)) return DL_ERR_WORKSPACE;
    const int BT = prob_bt(B), L = 1 << k;
    float *sig = (float *)saved;
    float *xT = (float *)((char *)saved + prob_sig_bytes(N, k, O));
    // x re-tiled and the tables built in one launch
    prob_launch_to_tiles("prob_to_tiles_x+sig_table", x, xT, B, I,
                         ProbTables{raw_w, nullptr, inv_t, sig, (float *)((char *)xT + prob_xT_bytes(B, I)), N, L, O}, s);
    const int grid = dl_xcd_grid(dl_ceil_div((long long)N * O, PROB_TC), BT);
#define CALL(KK) DL_TIMED("prob_fwd_t", s, (prob_fwd_t<KK><<<grid, 64 * PROB_FW, 0, s>>>(xT, idx32, sig, y, B, I, N, O, BT)))
    PROB_DISPATCH(k, CALL)
#undef CALL
    return dl_launch_status();
}

extern "C" int dl_prob_layer_fwd(const float *x, const int32_t *idx32, const float *raw_w, float temperature, float *y,
                                 void *saved, size_t saved_bytes, int B, int I, int N, int k, int O, void *stream) {
    return prob_forward(x, idx32, raw_w, prob_temp(temperature, nullptr), y, saved, saved_bytes, B, I, N, k, O, stream);
}
extern "C" int dl_prob_layer_fwd_nodes(const float *x, const int32_t *idx32, const float *raw_w, const float *temperature_n,
                                       float *y, void *saved, size_t saved_bytes, int B, int I, int N, int k, int O,
                                       void *stream) {
    if (!temperature_n) return DL_ERR_NULL;
    return prob_forward(x, idx32, raw_w, prob_temp(1.0f, temperature_n), y, saved, saved_bytes, B, I, N, k, O, stream);
}

template <bool HYB>
static void prob_launch_bwd(const char *name, const float *xT, const float *gy, const int32_t *idx32, const float *table,
                            float *gmT, float *gpart, int B, int I, int N, int k, int O, int tpc, bool want_gm, hipStream_t s) {
    const int BT = prob_bt(B), NO = N * O, W = prob_block_columns(NO);
    const dim3 grid(dl_ceil_div(NO, W), dl_ceil_div(BT, tpc));
#define CALL(KK)                                                                                                                  \
    do {                                                                                                                          \
        if (W == 4) DL_TIMED(name, s, (prob_bwd_t<KK, HYB, 4, false><<<grid, 256, 0, s>>>(xT, gy, idx32, table, gmT, gpart, I, N, \
                                                                                          O, BT, tpc, want_gm, B)));              \
        else if (O == 1 && prob_gm_stream(B, N, k, O))                                                                            \
            DL_TIMED(name, s, (prob_bwd_t<KK, HYB, 16, true><<<grid, 1024, 0, s>>>(xT, gy, idx32, table, gmT, gpart, I, N, O, BT, \
                                                                                   tpc, want_gm, B)));                            \
        else DL_TIMED(name, s, (prob_bwd_t<KK, HYB, 16, false><<<grid, 1024, 0, s>>>(xT, gy, idx32, table, gmT, gpart, I, N, O,   \
                                                                                     BT, tpc, want_gm, B)));                      \
    } while (0)
    PROB_DISPATCH(k, CALL)
#undef CALL
}

static int prob_backward(const float *x, const void *saved, const int32_t *idx32, const int32_t *inv_ptr,
                         const int32_t *inv_pos, const float *raw_w, ProbTemp inv_t, const float *gy, float *gx, float *graw,
                         void *ws, size_t ws_bytes, int B, int I, int N, int k, int O, void *stream) {
    if (!x || !idx32 || !raw_w || !gy || !graw) return DL_ERR_NULL;
    if (gx && (!inv_ptr || !inv_pos)) return DL_ERR_NULL;
    int rc = prob_check(B, I, N, k, O);
    if (rc) return rc;
    hipStream_t s = (hipStream_t)stream;
    const long long WT = (long long)N * ((long long)1 << k) * O;
    if (!prob_fast(I, N, k, O)) {
        DL_TIMED("prob_fill_zero", s, (prob_fill_zero<<<dl_ceil_div(WT, 256), 256, 0, s>>>(graw, WT)));
        if (gx) prob_fill_zero<<<dl_ceil_div((long long)B * I, 256), 256, 0, s>>>(gx, (long long)B * I);
        DL_TIMED("prob_generic_bwd", s, (prob_generic_bwd<<<dl_ceil_div((long long)B * N, 256), 256, 0, s>>>(x, idx32, raw_w, inv_t, gy, gx, graw, B, I, N,
                                                                          k, O, 0)));
        return dl_launch_status();
    }
    if (!ws) return DL_ERR_NULL;
    if (ws_bytes < (saved ? prob_gm_bytes(B, N, k, O) : dl_prob_bwd_workspace_bytes(B, I, N, k, O))) return DL_ERR_WORKSPACE;
    const int BT = prob_bt(B), L = 1 << k, NO = N * O;
    const int tpc = prob_tiles_per_chunk(B, N, k, O);
    const int chunks = dl_ceil_div(BT, tpc);
    char *w = (char *)ws;
    float *sig = (float *)saved;  // what the forward of the same x, raw_w and temperature left
    if (!saved) { sig = (float *)w; w += 2 * prob_sig_bytes(N, k, O) + prob_xT_bytes(B, I); }
    float *xT = (float *)((char *)sig + prob_sig_bytes(N, k, O)), *cen = (float *)((char *)xT + prob_xT_bytes(B, I));
    float *gmT = (float *)w; w += dl_align256((size_t)BT * NO * k * 64 * sizeof(float));
    float *gpart = (float *)w;
    if (!saved)
        prob_launch_to_tiles("prob_to_tiles_x+sig_table", x, xT, B, I, ProbTables{raw_w, nullptr, inv_t, sig, cen, N, L, O}, s);
    prob_launch_bwd<false>("prob_bwd_t", xT, gy, idx32, cen, gmT, gpart, B, I, N, k, O, tpc, gx != nullptr, s);
    const ProbReduce R = {gpart, sig, inv_t, graw, N, L, O, chunks};
    prob_launch_gather_and_reduce(gmT, inv_ptr, inv_pos, gx, B, I, N, k, O, BT, R, WT, s);
    return dl_launch_status();
}

extern "C" int dl_prob_layer_bwd(const float *x, const void *saved, const int32_t *idx32, const int32_t *inv_ptr,
                                 const int32_t *inv_pos,
                                 const float *raw_w, float temperature, const float *gy, float *gx, float *graw,
                                 void *ws, size_t ws_bytes, int B, int I, int N, int k, int O, void *stream) {
    return prob_backward(x, saved, idx32, inv_ptr, inv_pos, raw_w, prob_temp(temperature, nullptr), gy, gx, graw, ws, ws_bytes,
                         B, I, N, k, O, stream);
}
extern "C" int dl_prob_layer_bwd_nodes(const float *x, const void *saved, const int32_t *idx32, const int32_t *inv_ptr,
                                       const int32_t *inv_pos, const float *raw_w, const float *temperature_n,
                                       const float *gy, float *gx, float *graw, void *ws, size_t ws_bytes, int B, int I,
                                       int N, int k, int O, void *stream) {
    if (!temperature_n) return DL_ERR_NULL;
    return prob_backward(x, saved, idx32, inv_ptr, inv_pos, raw_w, prob_temp(1.0f, temperature_n), gy, gx, graw, ws, ws_bytes,
                         B, I, N, k, O, stream);
}

// Nodes that read their inputs in order (prob_ordered_*).
static inline int prob_ordered_check(int B, int N, int k) {
    const int rc = prob_check(B, 1, N, k, 1);
    if (rc) return rc;
    return k <= DL_MAX_FAST_K && (long long)N * k < (1 << 23) ? DL_OK : DL_ERR_UNSUPPORTED;
}
static inline int prob_ordered_bwd_tiles(int B, int N, int k) {
    return prob_tiles_per_chunk_of(prob_bt(B), N, PROB_ON, prob_bwd_own_tiles(k));
}
// values per access: the rows of x and gx have to start on multiples of that (and a block's columns to end there)
// (One at a time with six inputs means an x or gx off by four bytes; those two kernels spill 9 and 11 registers, forward and backward of 4096
// rows x 999 nodes 108 us where re-tiling takes 135, of 40 nodes 25 against 35.)
static inline int prob_ordered_wide(const float *x, const float *gx, int N, int k) {
    const uintptr_t at = (uintptr_t)x | (uintptr_t)gx;
    const long long M = (long long)N * k;
    return M % 4 == 0 && at % 16 == 0 ? 4 : M % 2 == 0 && at % 8 == 0 ? 2 : 1;
}
extern "C" size_t dl_prob_ordered_saved_bytes(int N, int k) {
    return N <= 0 || k <= 0 || k > DL_MAX_FAST_K ? 256 : prob_sig_bytes(N, k, 1);
}
extern "C" size_t dl_prob_ordered_bwd_workspace_bytes(int B, int N, int k) {
    if (B <= 0 || prob_ordered_check(B, N, k) != DL_OK) return 256;
    const int chunks = dl_ceil_div(prob_bt(B), prob_ordered_bwd_tiles(B, N, k));
    return chunks > 1 ? chunks * prob_sig_bytes(N, k, 1) : 256;
}
extern "C" int dl_prob_ordered_fwd(const float *x, const float *raw_w, float temperature, const float *temperature_n, float *y,
                                   void *saved, size_t saved_bytes, int B, int N, int k, void *stream) {
    if (!x || !raw_w || !y || !saved) return DL_ERR_NULL;
    const int rc = prob_ordered_check(B, N, k);
    if (rc) return rc;
    if (saved_bytes < dl_prob_ordered_saved_bytes(N, k)) return DL_ERR_WORKSPACE;
    hipStream_t s = (hipStream_t)stream;
    const ProbTemp T = prob_temp(temperature, temperature_n);
    const int BT = prob_bt(B), tpc = prob_tiles_per_chunk_of(BT, N, PROB_ON, 1);
    const dim3 grid(dl_ceil_div(N, PROB_ON), dl_ceil_div(BT, tpc));
    const int wide = prob_ordered_wide(x, nullptr, N, k);
#define CALL(KK)                                                                                                                \
    do {                                                                                                                        \
        if (wide == 4) DL_TIMED("prob_ordered_fwd", s, (prob_ordered_fwd<KK, 4><<<grid, 64 * PROB_ON, 0, s>>>(                  \
            x, raw_w, T, (float *)saved, y, B, N, BT, tpc)));                                                                   \
        else if (wide == 2) DL_TIMED("prob_ordered_fwd", s, (prob_ordered_fwd<KK, 2><<<grid, 64 * PROB_ON, 0, s>>>(             \
            x, raw_w, T, (float *)saved, y, B, N, BT, tpc)));                                                                   \
        else DL_TIMED("prob_ordered_fwd", s, (prob_ordered_fwd<KK, 1><<<grid, 64 * PROB_ON, 0, s>>>(                            \
            x, raw_w, T, (float *)saved, y, B, N, BT, tpc)));                                                                   \
    } while (0)
    PROB_DISPATCH(k, CALL)
#undef CALL
    return dl_launch_status();
}
extern "C" int dl_prob_ordered_bwd(const float *x, const void *saved, float temperature, const float *temperature_n, const float *gy,
                                   float *gx, float *graw, void *ws, size_t ws_bytes, int B, int N, int k, void *stream) {
    if (!x || !saved || !gy || !graw || !ws) return DL_ERR_NULL;
    const int rc = prob_ordered_check(B, N, k);
    if (rc) return rc;
    if (ws_bytes < dl_prob_ordered_bwd_workspace_bytes(B, N, k)) return DL_ERR_WORKSPACE;
    hipStream_t s = (hipStream_t)stream;
    const ProbTemp T = prob_temp(temperature, temperature_n);
    const int BT = prob_bt(B), tpc = prob_ordered_bwd_tiles(B, N, k), chunks = dl_ceil_div(BT, tpc), L = 1 << k;
    const dim3 grid(dl_ceil_div(N, PROB_ON), chunks);
    const float *sig = (const float *)saved;
    float *gpart = chunks > 1 ? (float *)ws : nullptr;
    const int wide = prob_ordered_wide(x, gx, N, k);
#define CALL(KK)                                                                                                                \
    do {                                                                                                                        \
        if (wide == 4) DL_TIMED("prob_ordered_bwd", s, (prob_ordered_bwd<KK, 4><<<grid, 64 * PROB_ON, 0, s>>>(                  \
            x, gy, sig, T, gx, gpart, graw, B, N, BT, tpc)));                                                                   \
        else if (wide == 2) DL_TIMED("prob_ordered_bwd", s, (prob_ordered_bwd<KK, 2><<<grid, 64 * PROB_ON, 0, s>>>(             \
            x, gy, sig, T, gx, gpart, graw, B, N, BT, tpc)));                                                                   \
        else DL_TIMED("prob_ordered_bwd", s, (prob_ordered_bwd<KK, 1><<<grid, 64 * PROB_ON, 0, s>>>(                            \
            x, gy, sig, T, gx, gpart, graw, B, N, BT, tpc)));                                                                   \
    } while (0)
    PROB_DISPATCH(k, CALL)
#undef CALL
    if (chunks > 1) {
        const ProbReduce R = {gpart, sig, T, graw, N, L, 1, chunks};
        DL_TIMED("prob_reduce_weights", s, (prob_reduce_weights<<<dl_ceil_div((long long)N * L, 256), 256, 0, s>>>(R)));
    }
    return dl_launch_status();
}

// Hybrid nodes: the forward is the DWN lookup; the backward is the probabilistic one on the table as given.
extern "C" size_t dl_hybrid_bwd_workspace_bytes(int B, int I, int N, int k, int O) {
    if (B <= 0 || I <= 0 || N <= 0 || k <= 0 || O <= 0 || !prob_fast(I, N, k, O)) return 256;
    return dl_prob_bwd_workspace_bytes(B, I, N, k, O) - prob_sig_bytes(N, k, O);
}

// The forward leaves x re-tiled for the backward where both take the tiled path.
static inline bool hybrid_tiled(int B, int I, int N, int k, int O) {
    return prob_check(B, I, N, k, O) == DL_OK && prob_fast(I, N, k, O);
}
extern "C" size_t dl_dwn_saved_bytes(int B, int I, int N, int k, int O);
extern "C" size_t dl_dwn_fwd_workspace_bytes(int B, int I, int N, int k, int O);
extern "C" size_t dl_dwn_planes_bytes(int B, int C);
extern "C" int dl_dwn_layer_fwd(const float *x, const int32_t *idx32, const float *luts, float *y, void *saved, void *ws,
                                size_t ws_bytes, int B, int I, int N, int k, int O, void *stream);
extern "C" int dl_dwn_layer_fwd_planes(const void *planes_in, const int32_t *idx32, const float *luts, float *y,
                                       void *planes_out, void *saved, int B, int I, int N, int k, int O, void *stream);
extern "C" size_t dl_hybrid_saved_bytes(int B, int I, int N, int k, int O) {
    return hybrid_tiled(B, I, N, k, O) ? prob_xT_bytes(B, I) + prob_sig_bytes(N, k, O) : 256;
}
// the lookup's addresses, which nothing reads afterwards, and its planes or workspace
extern "C" size_t dl_hybrid_fwd_workspace_bytes(int B, int I, int N, int k, int O) {
    if (B <= 0 || I <= 0 || N <= 0 || k <= 0 || O <= 0) return 256;
    const size_t planes = dl_align256(dl_dwn_planes_bytes(B, I)), own = dl_align256(dl_dwn_fwd_workspace_bytes(B, I, N, k, O));
    return dl_align256(dl_dwn_saved_bytes(B, I, N, k, O)) + (planes > own ? planes : own);
}
// raw (nullable): the tables are its sigmoid and written to `luts`, by the blocks that build the backward's
static int hybrid_forward(const float *x, const int32_t *idx32, const float *raw, float *luts, float *y, void *saved,
                          size_t saved_bytes, void *ws, size_t ws_bytes, int B, int I, int N, int k, int O, void *stream) {
    if (!x || !idx32 || !luts || !y || !saved || !ws) return DL_ERR_NULL;
    if (B <= 0 || I <= 0 || N <= 0 || k <= 0 || O <= 0) return DL_ERR_SHAPE;
    if (saved_bytes < dl_hybrid_saved_bytes(B, I, N, k, O) || ws_bytes < dl_hybrid_fwd_workspace_bytes(B, I, N, k, O))
        return DL_ERR_WORKSPACE;
    hipStream_t s = (hipStream_t)stream;
    const size_t addr_bytes = dl_align256(dl_dwn_saved_bytes(B, I, N, k, O));
    char *rest = (char *)ws + addr_bytes;
    if (raw && !hybrid_tiled(B, I, N, k, O)) return DL_ERR_UNSUPPORTED;
    if (hybrid_tiled(B, I, N, k, O)) {
        const ProbTables q{raw, raw ? nullptr : luts, ProbTemp{1.0f, nullptr}, raw ? luts : nullptr, (float *)((char *)saved + prob_xT_bytes(B, I)),
                           N, 1 << k, O, true};
        prob_launch_to_tiles<true>("hybrid_tiles+planes", x, (float *)saved, B, I, q, s, (unsigned long long *)rest);
        const int rc = dl_dwn_layer_fwd_planes(rest, idx32, luts, y, nullptr, ws, B, I, N, k, O, stream);
        if (rc != DL_ERR_UNSUPPORTED) return rc;
    }
    return dl_dwn_layer_fwd(x, idx32, luts, y, ws, rest, ws_bytes - addr_bytes, B, I, N, k, O, stream);
}
extern "C" int dl_hybrid_layer_fwd(const float *x, const int32_t *idx32, const float *luts, float *y, void *saved,
                                   size_t saved_bytes, void *ws, size_t ws_bytes, int B, int I, int N, int k, int O,
                                   void *stream) {
    return hybrid_forward(x, idx32, nullptr, const_cast<float *>(luts), y, saved, saved_bytes, ws, ws_bytes, B, I, N, k, O, stream);
}
extern "C" int dl_hybrid_raw_fwd(const float *x, const int32_t *idx32, const float *raw_luts, float *luts, float *y, void *saved,
                                 size_t saved_bytes, void *ws, size_t ws_bytes, int B, int I, int N, int k, int O, void *stream) {
    if (!raw_luts) return DL_ERR_NULL;
    return hybrid_forward(x, idx32, raw_luts, luts, y, saved, saved_bytes, ws, ws_bytes, B, I, N, k, O, stream);
}

static int hybrid_backward(const float *x, const void *saved, const int32_t *idx32, const int32_t *inv_ptr,
                           const int32_t *inv_pos, const float *luts, const float *gy, float *gx, float *gluts, void *ws,
                           size_t ws_bytes, size_t ws_needed, int B, int I, int N, int k, int O, void *stream, bool to_raw = false) {
    if (!idx32 || !luts || !gy || !gluts) return DL_ERR_NULL;
    if (!x && !(saved && hybrid_tiled(B, I, N, k, O))) return DL_ERR_NULL;
    if (gx && (!inv_ptr || !inv_pos)) return DL_ERR_NULL;
    int rc = prob_check(B, I, N, k, O);
    if (rc) return rc;
    hipStream_t s = (hipStream_t)stream;
    const long long WT = (long long)N * ((long long)1 << k) * O;
    if (!prob_fast(I, N, k, O)) {
        DL_TIMED("prob_fill_zero", s, (prob_fill_zero<<<dl_ceil_div(WT, 256), 256, 0, s>>>(gluts, WT)));
        if (gx) prob_fill_zero<<<dl_ceil_div((long long)B * I, 256), 256, 0, s>>>(gx, (long long)B * I);
        DL_TIMED("prob_generic_bwd", s, (prob_generic_bwd<<<dl_ceil_div((long long)B * N, 256), 256, 0, s>>>(
                                            x, idx32, luts, ProbTemp{1.0f, nullptr}, gy, gx, gluts, B, I, N, k, O, 1)));
        return dl_launch_status();
    }
    if (!ws) return DL_ERR_NULL;
    if (ws_bytes < ws_needed) return DL_ERR_WORKSPACE;
    const int BT = prob_bt(B), L = 1 << k, NO = N * O;
    const int tpc = prob_tiles_per_chunk(B, N, k, O);
    const int chunks = dl_ceil_div(BT, tpc);
    char *w = (char *)ws;
    const float *xT = (const float *)saved;  // what the forward of the same x and luts left
    if (!saved) {
        float *own = (float *)w; w += prob_xT_bytes(B, I) + prob_sig_bytes(N, k, O);
        prob_launch_to_tiles("prob_to_tiles_x", x, own, B, I,
                             ProbTables{nullptr, luts, ProbTemp{1.0f, nullptr}, nullptr, (float *)((char *)own + prob_xT_bytes(B, I)), N, L, O}, s);
        xT = own;
    }
    const float *cen = (const float *)((const char *)xT + prob_xT_bytes(B, I));
    float *gmT = (float *)w; w += dl_align256((size_t)BT * NO * k * 64 * sizeof(float));
    float *gpart = (float *)w;
    prob_launch_bwd<true>("hybrid_bwd_t", xT, gy, idx32, cen, gmT, gpart, B, I, N, k, O, tpc, gx != nullptr, s);
    const ProbReduce R = {gpart, to_raw ? luts : nullptr, ProbTemp{1.0f, nullptr}, gluts, N, L, O, chunks, true};
    prob_launch_gather_and_reduce(gmT, inv_ptr, inv_pos, gx, B, I, N, k, O, BT, R, WT, s);
    return dl_launch_status();
}

extern "C" int dl_hybrid_layer_bwd(const float *x, const int32_t *idx32, const int32_t *inv_ptr, const int32_t *inv_pos,
                                   const float *luts, const float *gy, float *gx, float *gluts, void *ws, size_t ws_bytes,
                                   int B, int I, int N, int k, int O, void *stream) {
    return hybrid_backward(x, nullptr, idx32, inv_ptr, inv_pos, luts, gy, gx, gluts, ws, ws_bytes,
                           dl_hybrid_bwd_workspace_bytes(B, I, N, k, O), B, I, N, k, O, stream);
}
extern "C" size_t dl_hybrid_bwd_saved_workspace_bytes(int B, int I, int N, int k, int O) {
    return hybrid_tiled(B, I, N, k, O) ? prob_gm_bytes(B, N, k, O) : 256;
}
extern "C" int dl_hybrid_layer_bwd_saved(const float *x, const void *saved, const int32_t *idx32, const int32_t *inv_ptr,
                                         const int32_t *inv_pos, const float *luts, const float *gy, float *gx, float *gluts,
                                         void *ws, size_t ws_bytes, int B, int I, int N, int k, int O, void *stream) {
    if (!saved) return DL_ERR_NULL;
    return hybrid_backward(x, saved, idx32, inv_ptr, inv_pos, luts, gy, gx, gluts, ws, ws_bytes,
                           dl_hybrid_bwd_saved_workspace_bytes(B, I, N, k, O), B, I, N, k, O, stream);
}

// of a forward that made the tables: gluts is the gradient of what they are the sigmoid of
extern "C" int dl_hybrid_raw_bwd(const void *saved, const int32_t *idx32, const int32_t *inv_ptr, const int32_t *inv_pos, const float *luts,
                                 const float *gy, float *gx, float *graw, void *ws, size_t ws_bytes, int B, int I, int N, int k, int O,
                                 void *stream) {
    if (!saved) return DL_ERR_NULL;
    if (B > 0 && I > 0 && N > 0 && k > 0 && O > 0 && !hybrid_tiled(B, I, N, k, O)) return DL_ERR_UNSUPPORTED;
    return hybrid_backward(nullptr, saved, idx32, inv_ptr, inv_pos, luts, gy, gx, graw, ws, ws_bytes,
                           dl_hybrid_bwd_saved_workspace_bytes(B, I, N, k, O), B, I, N, k, O, stream, true);
}

// Eval forward with a workspace: the binarised sigmoid table of every node is the table of a DWN layer, so the
// DWN eval path (bit-planes when every input is 0 or 1, the literal float address otherwise) answers.
extern "C" size_t dl_dwn_eval_workspace_bytes(int B, int I, int N, int k, int O);
extern "C" int dl_dwn_layer_eval_ws(const float *x, const int32_t *idx32, const float *luts, float *y, void *ws,
                                    size_t ws_bytes, int B, int I, int N, int k, int O, void *stream);
static inline size_t prob_eval_table_bytes(int N, int k, int O) { return dl_align256((size_t)N * O * ((size_t)1 << k) * 4); }
extern "C" size_t dl_prob_eval_workspace_bytes(int B, int I, int N, int k, int O) {
    if (B <= 0 || I <= 0 || N <= 0 || k <= 0 || O <= 0 || k > DL_MAX_FAST_K) return 256;
    return prob_eval_table_bytes(N, k, O) + dl_dwn_eval_workspace_bytes(B, I, N, k, O);
}
static int prob_eval_ws(const float *x, const int32_t *idx32, const float *raw_w, ProbTemp T, float *y, void *ws,
                        size_t ws_bytes, int B, int I, int N, int k, int O, void *stream) {
    if (!x || !idx32 || !raw_w || !y) return DL_ERR_NULL;
    int rc = prob_check(B, I, N, k, O);
    if (rc) return rc;
    hipStream_t s = (hipStream_t)stream;
    if (k > DL_MAX_FAST_K) {
        DL_TIMED("prob_eval_kernel", s, (prob_eval_kernel<<<dl_ceil_div((long long)B * N * O, 256), 256, 0, s>>>(
                                            x, idx32, raw_w, T, y, B, I, N, k, O)));
        return dl_launch_status();
    }
    if (!ws) return DL_ERR_NULL;
    if (ws_bytes < dl_prob_eval_workspace_bytes(B, I, N, k, O)) return DL_ERR_WORKSPACE;
    float *sig = (float *)ws;
    const int L = 1 << k;
    DL_TIMED("prob_sig_table", s, (prob_sig_table<<<dl_ceil_div((long long)N * L * O, 256), 256, 0, s>>>(
                                      raw_w, T, sig, N, L, O)));
    const size_t tb = prob_eval_table_bytes(N, k, O);
    return dl_dwn_layer_eval_ws(x, idx32, sig, y, (char *)ws + tb, ws_bytes - tb, B, I, N, k, O, stream);
}
extern "C" int dl_prob_layer_eval_ws(const float *x, const int32_t *idx32, const float *raw_w, float temperature, float *y,
                                     void *ws, size_t ws_bytes, int B, int I, int N, int k, int O, void *stream) {
    return prob_eval_ws(x, idx32, raw_w, prob_temp(temperature, nullptr), y, ws, ws_bytes, B, I, N, k, O, stream);
}
extern "C" int dl_prob_layer_eval_ws_nodes(const float *x, const int32_t *idx32, const float *raw_w,
                                           const float *temperature_n, float *y, void *ws, size_t ws_bytes, int B, int I,
                                           int N, int k, int O, void *stream) {
    if (!temperature_n) return DL_ERR_NULL;
    return prob_eval_ws(x, idx32, raw_w, prob_temp(1.0f, temperature_n), y, ws, ws_bytes, B, I, N, k, O, stream);
}

// The same for k <= 6 with the row of x staged in the LDS by persistent blocks of 1024 threads: a thread keeps the input
// indices of its (up to eight) columns and their binarised tables - bit a of a 64-bit mask = (sigmoid(w[a] / T) >= 0.5),
// taken with the expression of prob_eval_kernel - in registers over all its rows.
template <int K>
__global__ __launch_bounds__(1024) void prob_eval_lds(const float *__restrict__ x, const int *__restrict__ idx32,
                                                       const float *__restrict__ raw, ProbTemp T, float *__restrict__ y,
                                                       int B, int I, long long NO, int O, long long c_begin, long long c_end) {
    extern __shared__ float prob_eval_row[];
    float *row = prob_eval_row;
    constexpr int L = 1 << K, QC = 8;
    int ix[QC][K];
    unsigned long long mask[QC];
#pragma unroll
    for (int q = 0; q < QC; ++q) {
        const long long c = c_begin + threadIdx.x + 1024LL * q;
        mask[q] = 0ull;
#pragma unroll
        for (int j = 0; j < K; ++j) ix[q][j] = 0;
        if (c < c_end) {
            const int n = (int)(c / O), d = (int)(c % O);
            const float inv_t = prob_inv_t_of(T, n);
#pragma unroll
            for (int j = 0; j < K; ++j) ix[q][j] = idx32[(size_t)n * K + j];
            for (int a = 0; a < L; ++a)
                mask[q] |= (dl_sigmoid(raw[((size_t)n * L + a) * O + d] * inv_t) >= 0.5f ? 1ull : 0ull) << a;
        }
    }
    const bool vec = (I & 3) == 0 && (((uintptr_t)x) & 15) == 0;
    for (int b = blockIdx.x; b < B; b += gridDim.x) {
        const float *xrow = x + (size_t)b * I;
        __syncthreads();  // the readers of the row before are done
        if (vec) {
            for (int i = threadIdx.x * 4; i < I; i += 4096)
                *reinterpret_cast<float4 *>(row + i) = *reinterpret_cast<const float4 *>(xrow + i);
        } else {
            for (int i = threadIdx.x; i < I; i += 1024) row[i] = xrow[i];
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < QC; ++q) {
            const long long c = c_begin + threadIdx.x + 1024LL * q;
            if (c >= c_end) break;
            float sum = 0.0f;
#pragma unroll
            for (int j = 0; j < K; ++j) sum += row[ix[q][j]] * (float)(1 << j);  // the order of prob_eval_kernel's loop
            long long a = (long long)sum;
            a = a < 0 ? 0 : (a > L - 1 ? L - 1 : a);
            __builtin_nontemporal_store(((mask[q] >> a) & 1ull) ? 1.0f : 0.0f, y + (size_t)b * NO + c);
        }
    }
}

extern "C" int dl_prob_layer_eval(const float *x, const int32_t *idx32, const float *raw_w, float temperature, float *y,
                                  int B, int I, int N, int k, int O, void *stream) {
    if (!x || !idx32 || !raw_w || !y) return DL_ERR_NULL;
    int rc = prob_check(B, I, N, k, O);
    if (rc) return rc;
    const long long NO = (long long)N * O;
    if (k <= 6 && I <= 32768 && NO >= 1024) {
        hipStream_t s = (hipStream_t)stream;
        const size_t lds = (size_t)I * sizeof(float);
        const ProbTemp T = prob_temp(temperature, nullptr);
        for (long long c0 = 0; c0 < NO; c0 += 8192) {  // windows of 8192 columns: eight per thread
            const long long c1 = c0 + 8192 < NO ? c0 + 8192 : NO;
#define CALL(KK)                                                                                                       \
    do {                                                                                                               \
        if (lds > 64 * 1024) {                                                                                         \
            const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(&prob_eval_lds<KK>),               \
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);            \
            if (e != hipSuccess) return (int)e;                                                                        \
        }                                                                                                              \
        DL_TIMED("prob_eval_kernel", s,                                                                                \
                 (prob_eval_lds<KK><<<B < 256 ? B : 256, 1024, lds, s>>>(x, idx32, raw_w, T, y, B, I, NO, O, c0, c1))); \
    } while (0)
            PROB_DISPATCH(k, CALL)
#undef CALL
        }
        return dl_launch_status();
    }
    DL_TIMED("prob_eval_kernel", (hipStream_t)stream, (prob_eval_kernel<<<dl_ceil_div((long long)B * N * O, 256), 256, 0, (hipStream_t)stream>>>(
        x, idx32, raw_w, prob_temp(temperature, nullptr), y, B, I, N, k, O)));
    return dl_launch_status();
}
