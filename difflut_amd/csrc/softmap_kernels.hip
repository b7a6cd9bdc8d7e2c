// LearnableLayer soft connectivity on gfx950:  m = x * softmax(W / tau)^T  and its adjoint, on the
// 16-bit matrix cores with fp32 accumulation (v_mfma_f32_32x32x16_bf16, ..._f16).
//
//   forward   m[b,o]  = rs[o] * sum_i x[b,i] E[o,i]          E = exp((W - max)/tau), rs = 1 / row sum
//   backward  gx[b,i] = sum_o gs[b,o] E[o,i]                  gs = gm * rs
//             gW[o,i] = rs[o] E[o,i] (G[o,i] - r[o]) / tau    G = gm^T x, r[o] = sum_b gm[b,o] m[b,o]
//             (r is the row sum of G * S written through the saved forward output, so the M x I
//              matrix G never needs a second pass)
//
// Operands.  precision 1 rounds x, E, gs (for gx) and gm (for gW) to bf16 once (nearest even).  precision 0 keeps fp32 values:
// every operand, times 2^24, is the EXACT sum of three bf16 planes (8 + 8 + 8 significant bits, each the rounding of what
// the planes above left; the factor keeps the lowest plane of every fp32 value, denormal ones included, a normal number).
// A product is the six plane products hi*hi, hi*mid, mid*hi, mid*mid, hi*lo, lo*hi.  The three products left out are
// below 2^-26 of |a*b| (|mid| <= 2^-9 |a|, |lo| <= 2^-18 |a|), less than the 2^-24 by which one fp32 multiply-add rounds,
// and bf16 products are exact in fp32, so the result is an fp32 product sum, times 2^48.  Six bf16 products at
// 2.5 PFLOP/s are 417 TFLOP/s of fp32 work against 157 on the fp32 matrix cores.
// Where a sum of an operand's size could overflow with that factor, or as the sum before rs, while the result does not, and
// for infinities and NaN, which planes do not carry, the product is computed with fp32 multiply-adds instead
// (softmap_plain): the pack pass notes the largest magnitude (softmap_note_large).
// Pairs.  Large products of precision 0 (SM_PAIR_WORK) take half as many matrix operations: an operand, scaled by a power of two
// to below 2^15, is hi + 2^-11 lo with hi its rounding to fp16 and lo that of 2^11 times the rest, and a product is hi*hi +
// 2^-11 (hi*lo + lo*hi), the second part in a sum of its own.  From 2^-13 on - 2^-27 of the largest - a pair is within 2^-23 of
// its value (23 of 24 bits); below, within 2^-36 of itself, whatever is left of the value.  The product left out, lo*lo, is below 2^-22
// of |a*b| (|lo| <= 2^-11 of the value), 2^-25 on average.  So no value may lie below: a sum can be made of small ones alone, where
// zeros of the other operand take out the large ones.
//   E is scaled by its row maximum, which is one, x by its largest value; where a value of either that is not zero lies below
//   2^-27 of that, decided on the device, the products it is in take the planes (launches of either kind that are not to run
//   end at once): with W of N(0, 6) at tau 1, where E spans more, the forward and gx.
//   gs is scaled row by row and gm column by column, so that no output row answers for another's magnitude.  Ordinary gradients
//   have a few values below 2^-27 of those (58 of the 24.6 million of a learnable layer's step): the pack pass leaves up to SM_TINY_MOST of them
//   out and softmap_plain adds their terms; where there are more, the product takes the planes, gx with E's made from its pairs
//   (SoftmapArgs::tiny).
// Error against float64 (2-norm) of m / gx / gW, 512 x 3136 x 48000, W of N(0, 1.5), tau 1: 1.1e-7 / 1.7e-7 / 4.3e-7 with pairs,
// 5.3e-7 / 3.2e-7 / 11.8e-7 with planes, whose operands are exact but whose sums have twice as many additions and no groups of
// stages (below); short sums: SM_PAIR_CHUNK.
//
// Layout.  An MFMA lane wants 8 consecutive reduction steps of one row: a "unit" of 16 bytes.  Every operand is stored
// as [reduction / 8][rows] units, rows padded to whole tiles with zeros, by the pass that has it in registers anyway
// (row statistics for E, softmap_pack for x and gs).  A tile of a stage is then a few contiguous runs, goes to the
// LDS without passing through registers (global_load_lds, 16 bytes per lane) in the order in which the MFMAs
// read it, without bank conflicts, and the products have no ragged edges except in their stores.  E is stored once, in units
// of 8 ROWS o (what gx reduces over); the forward reduces over i and turns its tiles on the way out of the LDS
// (ds_read_b64_tr_b16), which costs two reads per fragment instead of one and saves writing E a second time.
#include <type_traits>

#include "dl_common.h"

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 halfx8 __attribute__((ext_vector_type(8)));
typedef _Float16 halfx2 __attribute__((ext_vector_type(2)));
typedef unsigned uintx4 __attribute__((ext_vector_type(4)));
typedef short shortx4 __attribute__((ext_vector_type(4)));
typedef short shortx8 __attribute__((ext_vector_type(8)));

#define SM_LOG2E 1.4426950408889634f
#define SM_TC 128  // columns of an output tile
#define SM_GX_STAGE 16 // reduction steps of a stage with three planes
#define SM_UNIT 16 // bytes of a unit

// exp((w - mx)/tau), with scale = log2(e)/tau: one subtract, one multiply, the hardware exp2.
// Relative error about |w - mx|/tau * 6e-8 plus one ulp of exp2.  The row sums are built with the same function, so
// rows of S sum to one to rounding.
__device__ __forceinline__ float softmap_e(float w, float mx, float scale) {
    return __builtin_amdgcn_exp2f((w - mx) * scale);
}
__device__ __forceinline__ unsigned softmap_pk_bf16(float lo, float hi) {
    const floatx2 v = {lo, hi};
    return __builtin_bit_cast(unsigned, __builtin_convertvector(v, bf16x2));
}
__device__ __forceinline__ float softmap_lo(unsigned p) { return __uint_as_float(p << 16); }
__device__ __forceinline__ float softmap_hi(unsigned p) { return __uint_as_float(p & 0xffff0000u); }

#define SM_SCALE 0x1p24f    // of an operand that is cut into planes
#define SM_UNSCALE 0x1p-48f // of a product of two
#define SM_LARGE 0x1p16f    // values below need no look at whether a product of theirs could overflow
#define SM_BOUND 0x1p78f    // times 2^48, and 1 % for the planes' rounding: below 2^127

// The next plane of eight values as a unit; v is replaced by what is left for the planes below.
__device__ __forceinline__ uint4 softmap_unit(float *v) {
    unsigned w[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        w[j] = softmap_pk_bf16(v[2 * j], v[2 * j + 1]);
        v[2 * j] -= softmap_lo(w[j]);
        v[2 * j + 1] -= softmap_hi(w[j]);
    }
    return make_uint4(w[0], w[1], w[2], w[3]);
}

// ---- pairs: eight values, scaled to below 2^15, as a unit of hi = fp16(v) and one of lo = fp16(2^11 (v - hi))
#define SM_PAIR_EXP 14          // exponent that an operand's largest value is scaled to
#define SM_PAIR_LO 0x1p11f
#define SM_PAIR_TURN 8          // stages of a group
#define SM_PAIR_RANGE 0x1p-27f  // of the largest: from there on a pair holds 23 bits of a value
#define SM_PAIR_LEAST 0x1p-13f  // the same of a scaled one
// Values below that are summed one by one, at most.  The backward at 512 x 3136 x 48000, us: none 1345, 400 of them scattered 1432,
// all in one column 1562, 600 (planes) 1918; without pairs 1922.
#define SM_TINY_MOST 512

__device__ __forceinline__ void softmap_pair(const float *v, uint4 &hi, uint4 &lo) {
    unsigned h[4], l[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const floatx2 a = {v[2 * j], v[2 * j + 1]};
        const halfx2 t = __builtin_convertvector(a, halfx2);
        const floatx2 r = {(v[2 * j] - (float)t[0]) * SM_PAIR_LO, (v[2 * j + 1] - (float)t[1]) * SM_PAIR_LO};
        h[j] = __builtin_bit_cast(unsigned, t);
        l[j] = __builtin_bit_cast(unsigned, __builtin_convertvector(r, halfx2));
    }
    hi = make_uint4(h[0], h[1], h[2], h[3]);
    lo = make_uint4(l[0], l[1], l[2], l[3]);
}
// power of two that takes values of up to this magnitude (its bits) below 2^15
__device__ __forceinline__ int softmap_pair_shift(unsigned largest) { return SM_PAIR_EXP + 127 - (int)(largest >> 23); }

// What the choice between pairs and planes rests on, kept with the statistics: magnitudes of x, as bits, and whether a row of
// E spans more than the pairs carry.
struct SoftmapRange {
    unsigned x_largest, x_smallest, e_wide;  // x_smallest: of the values that are not zero
};
__device__ __forceinline__ bool softmap_x_wide(const SoftmapRange *r) {
    // (an infinity or a NaN among x as well: both sides are positive, and bits of positive floats compare as they do)
    return !(__uint_as_float(r->x_smallest) >= __uint_as_float(r->x_largest) * SM_PAIR_RANGE);
}
__device__ __forceinline__ bool softmap_wide(const SoftmapRange *r) { return r->e_wide != 0 || softmap_x_wide(r); }

__global__ __launch_bounds__(256) void softmap_clear(SoftmapRange *range, unsigned *words, int n) {
    const int e = blockIdx.x * 256 + threadIdx.x;
    if (range && e == 0) { range->x_largest = 0; range->x_smallest = 0x7f7fffffu; range->e_wide = 0; }
    if (e < n) words[e] = 0;
}

// The range of x: 512 x 3136 in 11 us.
__global__ __launch_bounds__(256) void softmap_scan_x(const float *__restrict__ x, long long total, SoftmapRange *range) {
    unsigned big = 0, small = 0x7f7fffffu;
    // eight loads in flight; past the end the last value again
    for (long long e = (long long)blockIdx.x * 2048 + threadIdx.x; e < total; e += (long long)gridDim.x * 2048) {
        unsigned v[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) v[q] = __float_as_uint(x[e + 256 * q < total ? e + 256 * q : total - 1]) & 0x7fffffffu;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            big = max(big, v[q]);
            small = min(small, v[q] != 0 ? v[q] : small);
        }
    }
    for (int off = 32; off > 0; off >>= 1) {
        big = max(big, (unsigned)__shfl_xor((int)big, off));
        small = min(small, (unsigned)__shfl_xor((int)small, off));
    }
    __shared__ unsigned part[2][4];
    if ((threadIdx.x & 63) == 0) { part[0][threadIdx.x >> 6] = big; part[1][threadIdx.x >> 6] = small; }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int q = 1; q < 4; ++q) { big = max(big, part[0][q]); small = min(small, part[1][q]); }
        // (atomics on one word queue up: most blocks see that they change nothing)
        if (big > __hip_atomic_load(&range->x_largest, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(&range->x_largest, big);
        if (small < __hip_atomic_load(&range->x_smallest, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMin(&range->x_smallest, small);
    }
}

// Largest magnitudes, as bits: of every column of gm, of every row of gs = gm * rs, and of gm.  A wavefront has 16 rows of 64
// columns at a time and goes over SM_SCAN_TILES such tiles of its rows.  512 x 48000 in 40 us, 2.5 TB/s.
#define SM_SCAN_TILES 4
__global__ __launch_bounds__(256) void softmap_scan_grad(const float *__restrict__ gm, const float *__restrict__ rs,
                                                         unsigned *__restrict__ row_max, unsigned *__restrict__ col_max,
                                                         unsigned *__restrict__ largest, const SoftmapRange *__restrict__ range,
                                                         int R, int C, int strips) {
    if (softmap_x_wide(range)) return;  // then nothing of gm goes into pairs
    const int lane = threadIdx.x & 63, wave = dl_uniform(threadIdx.x >> 6);
    const int r0 = (int)(blockIdx.x / strips) * 64 + wave * 16, c_first = (int)(blockIdx.x % strips) * (64 * SM_SCAN_TILES) + lane;
    __shared__ unsigned cols[64 * SM_SCAN_TILES];
    cols[threadIdx.x] = 0;
    __syncthreads();
    unsigned rows[16], big = 0;
#pragma unroll
    for (int i = 0; i < 16; ++i) rows[i] = 0;
    // every load in flight at once; past the ends the last row or column again, whose maxima nobody reads there
    float v[SM_SCAN_TILES][16], f[SM_SCAN_TILES];
#pragma unroll
    for (int t = 0; t < SM_SCAN_TILES; ++t) {
        const int col = min(c_first + t * 64, C - 1);
        f[t] = rs[col];
#pragma unroll
        for (int i = 0; i < 16; ++i) v[t][i] = gm[(size_t)min(r0 + i, R - 1) * C + col];
    }
#pragma unroll
    for (int t = 0; t < SM_SCAN_TILES; ++t) {
        unsigned cb = 0;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            cb = max(cb, __float_as_uint(v[t][i]) & 0x7fffffffu);
            rows[i] = max(rows[i], __float_as_uint(v[t][i] * f[t]) & 0x7fffffffu);
        }
        atomicMax(&cols[t * 64 + lane], cb);
        big = max(big, cb);
    }
    // the maxima over the lanes, halving the rows a lane has at each of four steps: lane l ends with row l / 4
#pragma unroll
    for (int half = 8, off = 32; half > 0; half >>= 1, off >>= 1)
#pragma unroll
        for (int i = 0; i < half; ++i) {
            const bool up = (lane & off) != 0;
            const unsigned keep = up ? rows[i + half] : rows[i], give = up ? rows[i] : rows[i + half];
            rows[i] = max(keep, (unsigned)__shfl_xor((int)give, off));
        }
    rows[0] = max(rows[0], (unsigned)__shfl_xor((int)rows[0], 2));
    rows[0] = max(rows[0], (unsigned)__shfl_xor((int)rows[0], 1));
    if ((lane & 3) == 0 && rows[0] > __hip_atomic_load(row_max + r0 + (lane >> 2), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
        atomicMax(row_max + r0 + (lane >> 2), rows[0]);
    __syncthreads();
    if (cols[threadIdx.x] != 0) atomicMax(col_max + (int)(blockIdx.x % strips) * (64 * SM_SCAN_TILES) + threadIdx.x, cols[threadIdx.x]);
    for (int off = 32; off > 0; off >>= 1) big = max(big, (unsigned)__shfl_xor((int)big, off));
    if (lane == 0 && big > __hip_atomic_load(largest, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(largest, big);
}

// Largest magnitude of an operand, as bits (a NaN is larger than all); stays 0 while every value is below SM_LARGE, which is
// why the word is hardly ever written.  `big`: the bits of this thread's largest.
__device__ __forceinline__ void softmap_note_large(unsigned *largest, unsigned big) {
    if (__ballot(big >= __float_as_uint(SM_LARGE)) == 0) return;
    for (int off = 32; off > 0; off >>= 1) big = max(big, (unsigned)__shfl_xor((int)big, off));
    if ((threadIdx.x & 63) == 0 && big > __hip_atomic_load(largest, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
        atomicMax(largest, big);
}
__device__ __forceinline__ float softmap_largest(const unsigned *largest) {
    const unsigned big = *largest;
    return __uint_as_float(max(big, __float_as_uint(SM_LARGE)));
}

// ---------------------------------------------------------------------------------
// Row maxima, E and 1 / row sums of eight rows of W per block, E written as units of those eight rows.  Bound by HBM:
// W is read once and the planes written once (48000 x 3136: 602 MB in, 301 MB per plane out).  The rows stay in registers
// between the three steps (NQ values per row and thread), so T * NQ bounds the width; wider rows (NQ = 0) are read
// three times.  With one plane the sum is that of the rounded values.  Blocks past the last row and columns past I write zeros
// (the padding the products read).
// NP = 2: pairs; a block whose rows span more than pairs carry sets e_wide instead, and blocks that find it set, or x too wide,
// end.  NP = 3 with a range: the launch behind that one, which writes planes where it has come to that.
template <int NP, int T, int NQ>
__global__ __launch_bounds__(T, NQ == 8 ? 4 : 1) void softmap_rowstats(const float *__restrict__ W, float scale, float *__restrict__ mxs,
                                                      float *__restrict__ rss, char *__restrict__ E, size_t plane, int M,
                                                      int I, int Ip, unsigned *__restrict__ largest,
                                                      SoftmapRange *__restrict__ range) {
    constexpr int WV = T / 64;
    if (NP == 2 && softmap_x_wide(range)) return;
    if (NP == 3 && range && !softmap_wide(range)) return;
    __shared__ float red[2][8][WV];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    if (NP == 2) {  // read once for the block: another may set it meanwhile, and the barriers below are for all wavefronts or none
        __shared__ unsigned found_wide;
        if (tid == 0) found_wide = __hip_atomic_load(&range->e_wide, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        if (found_wide != 0) return;
    }
    const int o0 = blockIdx.x * 8;
    uint4 *out = reinterpret_cast<uint4 *>(E + (size_t)blockIdx.x * Ip * SM_UNIT);
    float v[NQ > 0 ? NQ : 1][8];
    float mx[8], sum[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) { mx[j] = -INFINITY; sum[j] = 0.0f; }
    auto load = [&](int i, int j) -> float { return i < I && o0 + j < M ? W[(size_t)(o0 + j) * I + i] : -INFINITY; };
    if (NQ > 0) {
#pragma unroll
        for (int q = 0; q < NQ; ++q)
#pragma unroll
            for (int j = 0; j < 8; ++j) v[q][j] = load(tid + T * q, j);
#pragma unroll
        for (int q = 0; q < NQ; ++q)
#pragma unroll
            for (int j = 0; j < 8; ++j) mx[j] = fmaxf(mx[j], v[q][j]);
    } else {
        for (int i = tid; i < I; i += T)
#pragma unroll
            for (int j = 0; j < 8; ++j) mx[j] = fmaxf(mx[j], load(i, j));
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        for (int off = 32; off > 0; off >>= 1) mx[j] = fmaxf(mx[j], __shfl_xor(mx[j], off));
        if (lane == 0) red[0][j][wave] = mx[j];
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        mx[j] = red[0][j][0];
#pragma unroll
        for (int q = 1; q < WV; ++q) mx[j] = fmaxf(mx[j], red[0][j][q]);
    }
    auto expo = [&](float w, int i, int j) -> float {
        const float e = i < I && o0 + j < M ? softmap_e(w, mx[j], scale) : 0.0f;
        return NP == 1 ? softmap_lo(softmap_pk_bf16(e, 0.0f)) : e;
    };
    bool bad = false;
    auto look = [&](const float *e) {  // (zeros are exact in both; a NaN is too wide)
#pragma unroll
        for (int j = 0; j < 8; ++j) bad |= !(e[j] >= SM_PAIR_RANGE) && e[j] != 0.0f;
    };
    auto store = [&](int i, float *e) {
        if (i < Ip) {
            if (NP == 2) {
                look(e);
#pragma unroll
                for (int j = 0; j < 8; ++j) e[j] *= (float)(1 << SM_PAIR_EXP);
                uint4 hi, lo;
                softmap_pair(e, hi, lo);
                *reinterpret_cast<uint4 *>(out + i) = hi;
                *reinterpret_cast<uint4 *>(reinterpret_cast<char *>(out + i) + plane) = lo;
                return;
            }
            if (NP > 1) {
#pragma unroll
                for (int j = 0; j < 8; ++j) e[j] *= SM_SCALE;
            }
#pragma unroll
            for (int p = 0; p < (NP == 1 ? 1 : 3); ++p)
                *reinterpret_cast<uint4 *>(reinterpret_cast<char *>(out + i) + p * plane) = softmap_unit(e);
        }
    };
    if (NQ > 0) {
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
#pragma unroll
            for (int j = 0; j < 8; ++j) { v[q][j] = expo(v[q][j], tid + T * q, j); sum[j] += v[q][j]; }
        }
#pragma unroll
        for (int q = 0; q < NQ; ++q) store(tid + T * q, v[q]);
    } else {
        for (int i = tid; i < Ip; i += T) {
            float e[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) { e[j] = expo(load(i, j), i, j); sum[j] += e[j]; }
            store(i, e);
        }
    }
    if (NP == 2 && __ballot(bad) != 0 && lane == 0) atomicOr(&range->e_wide, 1u);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        for (int off = 32; off > 0; off >>= 1) sum[j] += __shfl_xor(sum[j], off);
        if (lane == 0) red[1][j][wave] = sum[j];
    }
    __syncthreads();
    if (tid < 8) {
        float t = red[1][tid][0];
#pragma unroll
        for (int q = 1; q < WV; ++q) t += red[1][tid][q];
        float mj = red[0][tid][0];
#pragma unroll
        for (int q = 1; q < WV; ++q) mj = fmaxf(mj, red[0][tid][q]);
        mxs[o0 + tid] = o0 + tid < M ? mj : 0.0f;
        rss[o0 + tid] = o0 + tid < M ? 1.0f / t : 0.0f;
        if (largest && blockIdx.x == 0 && tid == 0) *largest = 0;  // of x, which is packed after this
    }
}

// ---------------------------------------------------------------------------------
// src [R][C] fp32 -> units along the rows [Rp/8][Cp] and / or along the columns [Cp/8][Rp], NP planes each, the latter scaled
// per column where `colscale` is given, padding zero; three planes are those of 2^24 times the value.  With `other`:
// dots[chunk][c] = sum of src * other over the 64 rows of the chunk (unscaled; the reader adds the chunks in order).
// Block = 64 columns x 64 rows: a thread has sixteen rows of a column, so units along the rows leave straight from registers;
// those along the columns go through the LDS (row stride 65 words, no conflicts).  `largest` (three planes; nullable): see
// softmap_note_large; `clear` (nullable): such a word that a later launch fills.  `alternate` (three planes): factor of
// every second group of SM_GX_STAGE columns in the units along the columns.
// NP = 2: pairs, or planes where `range` says so: units along the rows are gW's, which takes E from W and asks for x's range only.
// `row_max` (units along the columns) and `col_max` (units along the rows): the magnitudes that the pairs are scaled by, without
// them x_largest.  `tiny`: how many values the pairs along the columns ([0]) and along the rows ([1]) leave out.  With `tiny_at`
// this launch finds them and lists the first SM_TINY_MOST of each as (row of the product's result, step of its reduction); else
// they are counted already, and where there are more than that the units along the rows are planes, with `again` those along the
// columns too, and nothing else is written.
template <int NP>
__global__ __launch_bounds__(256) void softmap_pack(const float *__restrict__ src, const float *__restrict__ colscale,
                                                    const float *__restrict__ other, float *__restrict__ dots,
                                                    char *__restrict__ rows8, size_t rows_plane, char *__restrict__ cols8,
                                                    size_t cols_plane, int R, int C, int Rp, int Cp, float alternate, unsigned *__restrict__ largest,
                                                    unsigned *__restrict__ clear, const SoftmapRange *__restrict__ range,
                                                    const unsigned *__restrict__ row_max, const unsigned *__restrict__ col_max,
                                                    unsigned *__restrict__ tiny, int2 *__restrict__ tiny_at, bool again) {
    bool row_pairs = NP == 2 && !softmap_x_wide(range), col_pairs = NP == 2 && !softmap_wide(range);
    if (NP == 2 && tiny && !tiny_at) {
        const bool rows_many = row_pairs && tiny[1] > SM_TINY_MOST, cols_many = col_pairs && tiny[0] > SM_TINY_MOST;
        if (again && !rows_many) rows8 = nullptr;
        if (again && !cols_many) cols8 = nullptr;
        if (!rows8 && !cols8) return;
        row_pairs = row_pairs && !rows_many;
        col_pairs = col_pairs && !cols_many;
    }
    // (a grid of one dimension: the second holds 65535 blocks, 4.19 million rows)
    const int cb64 = Cp / 64, bx = blockIdx.x % cb64, by = blockIdx.x / cb64;
    if (clear && blockIdx.x == 0 && threadIdx.x == 0) *clear = 0;
    __shared__ float tile[64][65];
    __shared__ float part[4][64];
    const int c = threadIdx.x & 63, g = threadIdx.x >> 6;
    const int col = bx * 64 + c, r0 = by * 64;
    float v[16], dot = 0.0f;
    float f = colscale && col < C ? colscale[col] : 1.0f;
    if (NP > 1 && !col_pairs && (col / SM_GX_STAGE) % 2 != 0) f *= alternate;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int r = r0 + g * 16 + i;
        v[i] = r < R && col < C ? src[(size_t)r * C + col] : 0.0f;
    }
    if (other) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int r = r0 + g * 16 + i;
            dot += v[i] * (r < R && col < C ? other[(size_t)r * C + col] : 0.0f);
        }
        part[g][c] = dot;
    }
    if (NP > 1) {
        unsigned big = 0;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            big = max(big, __float_as_uint(v[i]) & 0x7fffffffu);
            if (NP == 3) v[i] *= SM_SCALE;
        }
        if (largest && !row_pairs) softmap_note_large(largest, big);
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) tile[g * 16 + i][c] = v[i] * f;
    __syncthreads();
    if (other && g == 0) dots[(size_t)by * Cp + col] = ((part[0][c] + part[1][c]) + part[2][c]) + part[3][c];
    // eight steps of the reduction, from `step` on, of row `row` of the result
    auto put_pairs = [&](float *w, unsigned biggest, char *d, size_t plane, int which, int row, int step) {
        const int shift = softmap_pair_shift(biggest);
        unsigned left_out = 0;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float scaled = __builtin_amdgcn_ldexpf(w[j], shift);
            const bool out = w[j] != 0.0f && fabsf(scaled) < SM_PAIR_LEAST;
            left_out |= out ? 1u << j : 0u;
            w[j] = out ? 0.0f : scaled;
        }
        if (tiny_at && left_out != 0 && __hip_atomic_load(tiny + which, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) <= SM_TINY_MOST) {
            // (past the limit nobody looks at the list, and the number no longer matters)
            unsigned at = atomicAdd(tiny + which, (unsigned)__popc(left_out));
            for (; left_out != 0 && at < SM_TINY_MOST; ++at, left_out &= left_out - 1)
                tiny_at[which * SM_TINY_MOST + at] = make_int2(row, step + __ffs(left_out) - 1);
        }
        uint4 hi, lo;
        softmap_pair(w, hi, lo);
        *reinterpret_cast<uint4 *>(d) = hi;
        *reinterpret_cast<uint4 *>(d + plane) = lo;
    };
    if (rows8) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int rb = (r0 >> 3) + g * 2 + h;
            if (8 * rb < Rp) {
                char *d = rows8 + ((size_t)rb * Cp + col) * SM_UNIT;
                if (row_pairs) {
                    put_pairs(v + 8 * h, col_max ? col_max[col] : range->x_largest, d, rows_plane, 1, col, rb * 8);
                    continue;
                }
                if (NP == 2) {
#pragma unroll
                    for (int j = 0; j < 8; ++j) v[8 * h + j] *= SM_SCALE;
                }
#pragma unroll
                for (int p = 0; p < (NP == 1 ? 1 : 3); ++p) *reinterpret_cast<uint4 *>(d + p * rows_plane) = softmap_unit(v + 8 * h);
            }
        }
    }
    if (cols8) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int cb = g * 2 + h, row = r0 + c;
            if (row < Rp) {
                float w[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) w[j] = tile[c][cb * 8 + j];
                char *d = cols8 + ((size_t)(bx * 8 + cb) * Rp + row) * SM_UNIT;
                if (col_pairs) {
                    put_pairs(w, row_max ? row_max[row] : range->x_largest, d, cols_plane, 0, row, (bx * 8 + cb) * 8);
                    continue;
                }
                if (NP == 2) {
#pragma unroll
                    for (int j = 0; j < 8; ++j) w[j] *= SM_SCALE;
                }
#pragma unroll
                for (int p = 0; p < (NP == 1 ? 1 : 3); ++p) *reinterpret_cast<uint4 *>(d + p * cols_plane) = softmap_unit(w);
            }
        }
    }
}

// out[e] = sum over chunks of part[chunk][e], fixed order; VEC = 4 when total is a multiple of 4.  Summed in double, so that the
// result is rounded once however many chunks there are (bound by the reads: no slower).
template <int VEC>
__global__ __launch_bounds__(256) void softmap_reduce_chunks(const float *__restrict__ part, float *__restrict__ out,
                                                              long long total, int chunks, const SoftmapRange *range, const unsigned *tiny,
                                                              int wide_chunks) {
    if (range && (softmap_wide(range) || (tiny && *tiny > SM_TINY_MOST))) chunks = wide_chunks;
    if (range && chunks == 1) return;  // it is in `out`
    const long long e = ((long long)blockIdx.x * 256 + threadIdx.x) * VEC;
    if (e >= total) return;
    if (VEC == 4) {
        double acc[4] = {0.0, 0.0, 0.0, 0.0};
        auto add = [&](const float4 &p) { acc[0] += p.x; acc[1] += p.y; acc[2] += p.z; acc[3] += p.w; };
        int c = 0;
        for (; c + 4 <= chunks; c += 4) {  // four independent loads in flight, added in chunk order
            const float4 p0 = *reinterpret_cast<const float4 *>(part + (size_t)c * total + e);
            const float4 p1 = *reinterpret_cast<const float4 *>(part + (size_t)(c + 1) * total + e);
            const float4 p2 = *reinterpret_cast<const float4 *>(part + (size_t)(c + 2) * total + e);
            const float4 p3 = *reinterpret_cast<const float4 *>(part + (size_t)(c + 3) * total + e);
            add(p0); add(p1); add(p2); add(p3);
        }
        for (; c < chunks; ++c) add(*reinterpret_cast<const float4 *>(part + (size_t)c * total + e));
        *reinterpret_cast<float4 *>(out + e) = make_float4((float)acc[0], (float)acc[1], (float)acc[2], (float)acc[3]);
    } else {
        double acc = 0.0;
        for (int c = 0; c < chunks; ++c) acc += part[(size_t)c * total + e];
        out[e] = (float)acc;
    }
}

// ---------------------------------------------------------------------------------
struct SoftmapArgs {
    const char *A, *Bm;       // operands, plane 0: A [k/8][lda] units; Bm [k/8][ldb] units, forward: E [o/8][ldb]
    size_t a_plane, b_plane;  // bytes from a plane to the next
    int lda, ldb;
    float *out;               // [chunks][R][C]
    int R, C;
    int stages, chunk_stages; // reduction stages in all and per chunk
    int inner_count, outer_count, col_tiles;
    const float *rs;          // forward, gW: 1 / row sum [M]
    // gW
    const float *dots;        // [parts][dot_ld] partial r
    int parts, dot_ld;
    const float *mx, *W;      // precision 0: E is rebuilt from W (4 bytes per entry instead of three planes)
    const char *E;            // precision 1: E itself, [o/8][lde] units
    int lde;
    float scale, inv_tau;
    bool vec_out;             // W and out start on 16-byte boundaries
    // pairs
    const SoftmapRange *range;
    const unsigned *row_max;  // magnitudes that the rows of A are scaled by; forward: none (x_largest)
    const unsigned *tiny;     // gx, gW: how many values the pairs of A leave out
};

// Loads that bypass the registers: lane l's 16 bytes at base + voff land at LDS address lds + 16 l.  The compiler does not
// count them; the stages below wait for them by number (they complete in order).
__device__ __forceinline__ void softmap_to_lds(unsigned lds, const char *base, unsigned voff) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(voff), "s"(base) : "memory", "m0");
}
// all of this wavefront's loads but the last N have landed, its LDS reads are done, and every wavefront has got here
template <int N>
__device__ __forceinline__ void softmap_stage_barrier() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

// gx with three planes sums the six products of a stage by themselves and adds them to the running sum in one rounding, because
// its reduction is the long one; and as the matrix cores round sums of bf16 products towards minus infinity, which would add up
// over thousands of stages, every second stage comes with the sign of gs turned (SM_GX_STAGE) and is subtracted.  Against
// float64 (2-norm), 512 x 3136 x 48000: 1.15e-6 with one running sum for everything, 0.50e-6 by stages, 0.32e-6 with turned
// signs as well; on the fp32 matrix cores 0.62e-6.  It costs 675 -> 725 us there.
//
// One product kernel, three operand modes.  At 512 x 3136 x 48000 (1.54e11 flop a product; before: 128 x 128 tiles staged
// through registers) forward / gx / gW take 161 / 151 / 264 us with bf16 operands (before 236 / 453 / 365) and 660 / 725 /
// 840 us with three planes (before, on the fp32 matrix cores, 1318 / 1494 / 1347): 1.0 and 1.27-1.40 PFLOP/s of bf16
// products, the latter what the matrix cores hold under power; gW adds 602 MB of stores and 301 (602) MB of reads.
// MODE 0: forward   rows=b cols=o red=i   A = x    B = E (turned)   out = C rs[o]
// MODE 1: gx        rows=b cols=i red=o   A = gs   B = E
// MODE 2: gW        rows=o cols=i red=b   A = gm   B = x            out = rs E (C - r) / tau
// Block = 256 threads = 2 x 2 wavefronts, tile 64 FA x 128, a wavefront FA x 2 MFMA tiles of 32 x 32.  FA = 4 (256 rows):
// per MFMA a block pulls 24 KB per 32 reduction steps (NP = 1), 48 bytes per clock and CU at the matrix peak where
// 128 x 128 tiles need 64, all that an L2 channel delivers.  Two or three blocks share a CU (accumulators 128 registers, 72 or 48 KB of LDS
// each), so one block's MFMAs run under the other's barriers and stores.  Stages are KC deep, NBUF of them in the LDS.
// Pairs (NP = 2): 128 x 128 tiles, because hi*hi and the rest have accumulators of their own (64 registers each) and the loop has
// no vector arithmetic but the sign below; three blocks share a CU for gW, whose epilogue is two thirds memory (575 us before its reads were asked for ahead, 510 so; 704 with
// two).  Forward and gx add the sums of SM_PAIR_TURN stages to running ones, signs turned from group to group for the reason
// given above, and have two blocks per CU.  The same sizes, forward / gx / gW: 475 / 448 / 510 us (planes 703 / 786 / 866).  Bound by the fills of the stages: a CU pulls 21-24 bytes
// a clock, 48-82 lines in flight of 300-470 clocks each, and the matrix cores are busy 49 / 56 / 46 % of a clock that is 1.8 GHz (with bf16 operands
// 2.15).  256 x 128 tiles with one accumulator, the
// rest's sum scaled and added by every stage: 514 / 560 / 668.  gx in
// 5, 10 or 15 chunks of the reduction: 445, 486 and 497 with their sum; 10 for the shorter running sums.
// NPB = 2 with NP = 3 (gx): gs in planes, E in pairs, whose planes - times 2^10, which makes their scale the planes' - are made on
// the way out of the LDS; for gradients that span too much where E does not.  The backward at 512 x 3136 x 48000 with such
// gradients 1651 us, 1782 with E in planes throughout.
// Stages in the LDS, and blocks per CU that the registers have to allow.  bf16 operands in 256 x 128 tiles: the forward and gx with two
// stages and three blocks (161 / 149 us; three stages and two blocks 178 / 154), gW, whose epilogue is most of its time, with three
// stages and two blocks (261; two and three 288).
static constexpr int softmap_stages(int mode, int np, int fa) { return fa == 4 && (np == 3 || (np == 1 && mode != 2)) ? 2 : 3; }
static constexpr int softmap_blocks(int mode, int np, int fa) {
    return (mode == 2 && np == 2) || (mode != 2 && np == 1 && fa == 4) ? 3 : 2;
}
template <int MODE, int NP, int FA, int NPB>
__global__ __launch_bounds__(256, softmap_blocks(MODE, NP, FA)) void softmap_mfma(SoftmapArgs g) {
    extern __shared__ __align__(16) char lds[];
    constexpr bool FROM_PAIRS = NP == 3 && NPB == 2;
    static_assert(NPB == NP || (FROM_PAIRS && MODE == 1), "only gx mixes planes and pairs");
    if (NP > 1 && g.range) {
        const bool wide = dl_uniform(MODE == 2 ? softmap_x_wide(g.range) : softmap_wide(g.range));
        const bool many = MODE != 0 && dl_uniform((int)(*g.tiny > SM_TINY_MOST));
        if (NP == 2 ? wide || many : FROM_PAIRS ? wide || !many : MODE == 1 ? !wide : !wide && !many) return;
    }
    constexpr int TR = 64 * FA, TC = SM_TC;
    constexpr int KC = NP == 1 ? 32 : SM_GX_STAGE, KB = KC / 8;
    constexpr int NBUF = softmap_stages(MODE, NP, FA), AHEAD = NBUF - 1;
    constexpr int A_BYTES = NP * TR * KC * 2, STAGE = (NP * TR + NPB * TC) * KC * 2;
    constexpr bool BY_STAGE = NP == 3 && MODE == 1;
    static_assert(NP != 2 || FA == 2, "pairs keep two sums per output");
    constexpr int NA = NP * KB * (TR / 64) / 4, NB = NPB * KB * (TC / 64) / 4;  // loads per wavefront and stage
    static_assert(NP * KB * (TR / 64) % 4 == 0 && NPB * KB * (TC / 64) % 4 == 0, "whole loads per wavefront");
    typedef __attribute__((address_space(3))) char lds_char;
    const unsigned lds_base = (unsigned)(uintptr_t)(lds_char *)lds;  // what softmap_to_lds counts from
    int inner, outer;
    if (!dl_xcd_map(g.inner_count, g.outer_count, inner, outer)) return;
    const int rt = MODE == 2 ? outer : inner;
    const int ct = MODE == 2 ? inner : outer % g.col_tiles;
    const int zc = MODE == 2 ? 0 : outer / g.col_tiles;
    const int r0 = rt * TR, c0 = ct * TC;
    const int s_begin = zc * g.chunk_stages, nst = min(g.stages - s_begin, g.chunk_stages);
    const int tid = threadIdx.x, lane = tid & 63, wave = dl_uniform(tid >> 6);
    const int wm = (wave >> 1) * (TR / 2), wn = (wave & 1) * 64;

    // ---- what a wavefront copies in a stage: 64 units (1 KB of LDS) per load
    const unsigned a_voff = lane * SM_UNIT;
    // forward: LDS unit (ob, i') of the E tile holds i = i' ^ 4 (ob & 3): the four o-blocks a turning read touches then
    // sit on different banks
    const unsigned b_voff = MODE == 0 ? ((unsigned)(lane / KC) * g.ldb + ((lane % KC) ^ (4 * ((KC == 16 ? lane / 16 : 2 * (wave & 1) + lane / 32) & 3)))) * SM_UNIT
                                      : lane * SM_UNIT;
    auto issue = [&](int st, int buf) __attribute__((always_inline)) {
        const unsigned base = lds_base + buf * STAGE;
        const int k8 = (s_begin + st) * KB;
#pragma unroll
        for (int j = 0; j < NA; ++j) {
            const int p = wave + 4 * j, rb = p % (TR / 64), kbp = p / (TR / 64);
            const int plane = kbp / KB, kb = kbp % KB;
            softmap_to_lds(base + p * 1024, g.A + plane * g.a_plane + ((size_t)(k8 + kb) * g.lda + r0 + rb * 64) * SM_UNIT, a_voff);
        }
#pragma unroll
        for (int j = 0; j < NB; ++j) {
            const int p = wave + 4 * j;
            const char *src;
            if (MODE == 0) {
                constexpr int PP = TC / 8 * KC / 64, OB = 64 / KC;  // loads per plane, o-blocks per load
                const int plane = p / PP, ob = (p % PP) * OB;
                src = g.Bm + plane * g.b_plane + ((size_t)(c0 / 8 + ob) * g.ldb + (size_t)(s_begin + st) * KC) * SM_UNIT;
            } else {
                const int cb = p % (TC / 64), kbp = p / (TC / 64);
                const int plane = kbp / KB, kb = kbp % KB;
                src = g.Bm + plane * g.b_plane + ((size_t)(k8 + kb) * g.ldb + c0 + cb * 64) * SM_UNIT;
            }
            softmap_to_lds(base + A_BYTES + p * 1024, src, b_voff);
        }
    };

    floatx16 acc[FA][2];
#pragma unroll
    for (int i = 0; i < FA; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;

    // pairs: the products with a lower half, times 2^11, and the sums of earlier groups of stages
    constexpr int FP = NP == 2 ? FA : 1;
    constexpr bool GROUPS = NP == 2 && MODE != 2;
    floatx16 low[FP][2], sum[GROUPS ? FP : 1][2];
    if (NP == 2) {
#pragma unroll
        for (int i = 0; i < FP; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    low[i][j][v] = 0.0f;
                    if (GROUPS) sum[i][j][v] = 0.0f;
                }
    }

    const int kh = lane >> 5, l32 = lane & 31;
    const unsigned a_rd = (kh * TR + wm + l32) * SM_UNIT;
    unsigned b_rd;
    if (MODE == 0) {
        const int q = lane & 15, oh = (lane >> 4) & 1, ob = wn / 8 + oh * 2 + ((q & 3) >> 1);
        const int i = kh * 8 + (q >> 2);
        b_rd = A_BYTES + (ob * KC + (i ^ (4 * (ob & 3)))) * SM_UNIT + (q & 1) * 8;
    } else {
        b_rd = A_BYTES + (kh * TC + wn + l32) * SM_UNIT;
    }
    auto compute = [&](int buf, float sign, unsigned turn) __attribute__((always_inline)) {
        const unsigned base = buf * STAGE;
#pragma unroll
        for (int kk = 0; kk < KC / 16; ++kk) {
            bf16x8 a[NP][FA], b[NP][2];
#pragma unroll
            for (int p = 0; p < NP; ++p) {
#pragma unroll
                for (int j = 0; p < NPB && j < 2; ++j) {
                    if (MODE == 0) {
                        typedef __attribute__((address_space(3))) shortx4 lds_shortx4;
                        const unsigned at = base + b_rd + (p * (TC / 8) * KC + j * 4 * KC + kk * 16) * SM_UNIT;
                        const shortx4 t0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_shortx4 *)(lds + at));
                        const shortx4 t1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_shortx4 *)(lds + (at ^ 64u)));
                        b[p][j] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(t0, t1, 0, 1, 2, 3, 4, 5, 6, 7));
                    } else {
                        b[p][j] = *reinterpret_cast<const bf16x8 *>(lds + base + b_rd + ((p * KB + kk * 2) * TC + j * 32) * SM_UNIT);
                    }
                }
#pragma unroll
                for (int i = 0; i < FA; ++i)
                    a[p][i] = *reinterpret_cast<const bf16x8 *>(lds + base + a_rd + ((p * KB + kk * 2) * TR + i * 32) * SM_UNIT);
            }
            if (FROM_PAIRS) {
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const halfx8 h = __builtin_bit_cast(halfx8, b[0][j]), l = __builtin_bit_cast(halfx8, b[1][j]);
                    float e[8];
#pragma unroll
                    for (int q = 0; q < 8; ++q) e[q] = fmaf((float)l[q], SM_SCALE / SM_PAIR_LO / (1 << SM_PAIR_EXP), (float)h[q] * (SM_SCALE / (1 << SM_PAIR_EXP)));
#pragma unroll
                    for (int p = 0; p < NP; ++p) b[p][j] = __builtin_bit_cast(bf16x8, softmap_unit(e));
                }
            }
            // small products first
            constexpr int PA[6] = {0, 2, 1, 0, 1, 0}, PB[6] = {2, 0, 1, 1, 0, 0};
            if (NP == 2) {
#pragma unroll
                for (int i = 0; i < FA; ++i) {
                    const uintx4 turned = __builtin_bit_cast(uintx4, a[0][i]) ^ (GROUPS ? turn : 0u);
#pragma unroll
                    for (int j = 0; j < 2; ++j) {
                        const halfx8 ah = __builtin_bit_cast(halfx8, a[0][i]), al = __builtin_bit_cast(halfx8, a[NP - 1][i]);
                        const halfx8 bh = __builtin_bit_cast(halfx8, b[0][j]), bl = __builtin_bit_cast(halfx8, b[NP - 1][j]);
                        floatx16 &c = low[i % FP][j];
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(halfx8, turned), bh, acc[i][j], 0, 0, 0);
                        c = __builtin_amdgcn_mfma_f32_32x32x16_f16(al, bh, c, 0, 0, 0);
                        c = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, bl, c, 0, 0, 0);
                    }
                }
            } else if (BY_STAGE) {
#pragma unroll
                for (int i = 0; i < FA; ++i) {
                    floatx16 step[2];
#pragma unroll
                    for (int j = 0; j < 2; ++j)
#pragma unroll
                        for (int v = 0; v < 16; ++v) step[j][v] = 0.0f;
#pragma unroll
                    for (int t = 0; t < 6; ++t)
#pragma unroll
                        for (int j = 0; j < 2; ++j)
                            step[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[PA[t] % NP][i], b[PB[t] % NP][j], step[j], 0, 0, 0);
#pragma unroll
                    for (int j = 0; j < 2; ++j)
#pragma unroll
                        for (int v = 0; v < 16; ++v) acc[i][j][v] = fmaf(sign, step[j][v], acc[i][j][v]);
                }
            } else {
#pragma unroll
                for (int t = NP == 3 ? 0 : 5; t < 6; ++t)
#pragma unroll
                    for (int i = 0; i < FA; ++i)
#pragma unroll
                        for (int j = 0; j < 2; ++j)
                            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[PA[t] % NP][i], b[PB[t] % NP][j], acc[i][j], 0, 0, 0);
            }
        }
    };

#pragma unroll
    for (int s = 0; s < AHEAD; ++s)
        if (s < nst) issue(s, s);
    // gW, of the tile's rows, for the epilogue and behind the stages in the LDS: r (its parts added in order), for E rebuilt from W the
    // maximum, rs / tau, and the pairs' shift.  Read while the first stages come, eight parts at a time: one after the other, and at the
    // end of the block, they were eight trips to memory that nothing ran beside.
    float *rr = reinterpret_cast<float *>(lds + NBUF * STAGE);
    if (MODE == 2 && tid < TR) {
        float t = 0.0f;
        for (int q = 0; q < g.parts; q += 8) {
            float v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = g.dots[(size_t)min(q + u, g.parts - 1) * g.dot_ld + r0 + tid];
#pragma unroll
            for (int u = 0; u < 8; ++u) t = q + u < g.parts ? t + v[u] : t;
        }
        rr[tid] = t;
        rr[TR + tid] = g.mx[r0 + tid];
        rr[2 * TR + tid] = g.rs[r0 + tid] * g.inv_tau;
        if (NP == 2) rr[3 * TR + tid] = __int_as_float(-(softmap_pair_shift(g.range->x_largest) + softmap_pair_shift(g.row_max[r0 + tid])));
    }
    // what the epilogue reads of E or W for 32 rows of the wavefront's tile is asked for before the rows ahead of them are stored, E's first
    // rows before the last stage: with the parts above, gW 316 -> 264 us (bf16 operands), 575 -> 510 (pairs)
    const int rrow = lane >> 4, c4 = (lane & 15) * 4, col4 = c0 + wn + c4;
    const bool vec = g.C % 4 == 0 && g.vec_out;
    uint2 e[2][NP == 1 ? 8 : 1];
    floatx4 w4[NP != 1 ? 8 : 1];
    auto ask = [&](int i, int at) __attribute__((always_inline)) {
        const int row0 = r0 + wm + i * 32;
        if (NP == 1) {  // E as units of 8 rows: half a unit is this lane's four rows of a column
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    e[at][NP == 1 ? j * 4 + q : 0] = *reinterpret_cast<const uint2 *>(
                        g.E + ((size_t)((row0 >> 3) + q) * g.lde + c0 + wn + j * 32 + l32) * SM_UNIT + kh * 8);
        } else if (vec) {
#pragma unroll
            for (int it = 0; it < 8; ++it) {
                const int row = row0 + it * 4 + rrow;
                if (row < g.R && col4 < g.C) w4[NP != 1 ? it : 0] = *reinterpret_cast<const floatx4 *>(g.W + (size_t)row * g.C + col4);
            }
        }
    };
    int buf = 0, nbuf = AHEAD % NBUF;
    unsigned turn = 0;  // pairs: sign of the group's sums
    auto add_group = [&]() __attribute__((always_inline)) {
        const float sign = turn ? -1.0f : 1.0f;
#pragma unroll
        for (int i = 0; i < FP; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    sum[GROUPS ? i : 0][j][v] = fmaf(sign, acc[i][j][v], sum[GROUPS ? i : 0][j][v]);
                    acc[i][j][v] = 0.0f;
                }
    };
    for (int s = 0; s < nst; ++s) {
        if (s + AHEAD <= nst) softmap_stage_barrier<(NA + NB) * (AHEAD - 1)>();
        else softmap_stage_barrier<0>();
        if (s + AHEAD < nst) issue(s + AHEAD, nbuf);
        if (MODE == 2 && NP == 1 && s + 1 == nst) ask(0, 0);
        if (GROUPS && s % SM_PAIR_TURN == 0 && s > 0) {
            add_group();
            turn ^= 0x80008000u;
        }
        compute(buf, (s_begin + s) % 2 ? -1.0f : 1.0f, turn);
        buf = buf + 1 == NBUF ? 0 : buf + 1;
        nbuf = nbuf + 1 == NBUF ? 0 : nbuf + 1;
    }

    if (NP == 2) {
        if (GROUPS) add_group();
#pragma unroll
        for (int i = 0; i < FP; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int v = 0; v < 16; ++v)
                    acc[i][j][v] = fmaf(1.0f / SM_PAIR_LO, low[i][j][v], GROUPS ? sum[GROUPS ? i : 0][j][v] : acc[i][j][v]);
    }
    // accumulator layout of a 32x32 tile: register v of lane l holds row 8*(v/4) + 4*(l/32) + v%4, column l%32:
    // a store instruction writes two whole 128-byte lines
    const int R = g.R, C = g.C;
    // pairs: shift of the other operand, to be undone with that of the row
    const int shift = NP != 2 ? 0 : MODE == 0 ? SM_PAIR_EXP + softmap_pair_shift(g.range->x_largest)
                                  : MODE == 1 ? SM_PAIR_EXP : softmap_pair_shift(g.range->x_largest);
    if (MODE != 2) {
        float *dst = g.out + (size_t)zc * R * C;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int col = c0 + wn + j * 32 + l32;
            const float f = (NP == 3 ? SM_UNSCALE : 1.0f) * (MODE == 0 ? g.rs[col] : 1.0f);
#pragma unroll
            for (int i = 0; i < FA; ++i)
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    const int row = r0 + wm + i * 32 + 8 * (v >> 2) + 4 * kh + (v & 3);
                    if (row < R && col < C) {
                        float o = acc[i][j][v] * f;
                        if (NP == 2) o = __builtin_amdgcn_ldexpf(o, -(shift + (MODE == 1 ? softmap_pair_shift(g.row_max[row]) : 0)));
                        dst[(size_t)row * C + col] = o;
                    }
                }
        }
    } else {
        softmap_stage_barrier<63>();  // (the stages' reads are done; what the epilogue has asked for may be on its way)
        // 32 rows x 64 columns at a time go through the wavefront's own corner of the LDS, so that a lane owns four consecutive
        // columns of a row: 16-byte stores in runs of 256 bytes
        constexpr int TS = 68;  // floats per staged row: 64 + 4 keeps 16-byte alignment
        float *stg = reinterpret_cast<float *>(lds) + wave * (32 * TS);
#pragma unroll
        for (int i = 0; i < FA; ++i) {
            const int lr0 = wm + i * 32, row0 = r0 + lr0;
            if (NP == 1 && i + 1 < FA) ask(i + 1, (i + 1) & 1);
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                if (NP != 1 && j == 1) ask(i, 0);  // (not earlier: the registers are the sums', and in front of j = 0 eight spill: 535 us)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const float4 rv = *reinterpret_cast<const float4 *>(rr + lr0 + 8 * q + 4 * kh);
                    constexpr float f = NP == 3 ? SM_UNSCALE : 1.0f;
                    float o[4] = {acc[i][j][4 * q] * f, acc[i][j][4 * q + 1] * f, acc[i][j][4 * q + 2] * f, acc[i][j][4 * q + 3] * f};
                    if (NP == 2) {
                        const int4 sv = *reinterpret_cast<const int4 *>(rr + 3 * TR + lr0 + 8 * q + 4 * kh);
                        o[0] = __builtin_amdgcn_ldexpf(o[0], sv.x); o[1] = __builtin_amdgcn_ldexpf(o[1], sv.y);
                        o[2] = __builtin_amdgcn_ldexpf(o[2], sv.z); o[3] = __builtin_amdgcn_ldexpf(o[3], sv.w);
                    }
                    o[0] -= rv.x; o[1] -= rv.y; o[2] -= rv.z; o[3] -= rv.w;
                    if (NP == 1) {
                        const float4 fv = *reinterpret_cast<const float4 *>(rr + 2 * TR + lr0 + 8 * q + 4 * kh);
                        const uint2 eq = e[i & 1][NP == 1 ? j * 4 + q : 0];
                        o[0] *= softmap_lo(eq.x) * fv.x; o[1] *= softmap_hi(eq.x) * fv.y;
                        o[2] *= softmap_lo(eq.y) * fv.z; o[3] *= softmap_hi(eq.y) * fv.w;
                    }
#pragma unroll
                    for (int n = 0; n < 4; ++n) stg[(8 * q + 4 * kh + n) * TS + j * 32 + l32] = o[n];
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int it = 0; it < 8; ++it) {
                const int lr = it * 4 + rrow, row = row0 + lr;
                float4 o = *reinterpret_cast<const float4 *>(stg + lr * TS + c4);
                const size_t at = (size_t)row * C + col4;
                if (vec) {
                    if (row < R && col4 < C) {
                        if (NP != 1) {
                            const floatx4 w = w4[NP != 1 ? it : 0];
                            const float mx = rr[TR + lr0 + lr], f = rr[2 * TR + lr0 + lr];
                            o.x *= softmap_e(w.x, mx, g.scale) * f; o.y *= softmap_e(w.y, mx, g.scale) * f;
                            o.z *= softmap_e(w.z, mx, g.scale) * f; o.w *= softmap_e(w.w, mx, g.scale) * f;
                        }
                        __builtin_nontemporal_store(__builtin_bit_cast(floatx4, o), reinterpret_cast<floatx4 *>(g.out + at));
                    }
                } else {
                    const float os[4] = {o.x, o.y, o.z, o.w};
#pragma unroll
                    for (int n = 0; n < 4; ++n)
                        if (row < R && col4 + n < C)
                            g.out[at + n] = NP != 1 ? os[n] * (softmap_e(g.W[at + n], rr[TR + lr0 + lr], g.scale) * rr[2 * TR + lr0 + lr]) : os[n];
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
    }
}

template <int MODE, int NP, int FA, int NPB = NP>
static void softmap_launch(const SoftmapArgs &g, hipStream_t s) {
    constexpr int KC = NP == 1 ? 32 : 16, NBUF = softmap_stages(MODE, NP, FA);
    constexpr int lds_bytes = NBUF * (NP * 64 * FA + NPB * SM_TC) * KC * 2 + (MODE == 2 ? 4 * 64 * FA * 4 : 0);
    if (lds_bytes > 65536)
        (void)hipFuncSetAttribute(reinterpret_cast<const void *>(&softmap_mfma<MODE, NP, FA, NPB>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes);
    softmap_mfma<MODE, NP, FA, NPB><<<dl_xcd_grid(g.inner_count, g.outer_count), 256, lds_bytes, s>>>(g);
}

// ---------------------------------------------------------------------------------
// The products of precision 0 on the fp32 matrix cores (v_mfma_f32_32x32x2_f32), for operands that the planes do not carry.
// Launched behind every product; where the largest magnitudes allow the planes, which is all but always, a block reads them
// and ends (6 us of launch).  Else: 128 x 128 outputs per block and step, 2 x 2 wavefronts of 2 x 2 MFMA tiles, 16 reduction
// steps through the LDS with the next 16 on their way; every 128 steps the sums go into a second set of registers, so that
// long reductions round less.  512 x 3136 x 48000 with one infinite input: forward 2.34 ms, gW 2.37 (1.26 and 1.31 when the fp32
// matrix cores carried every call; such a call is an exception now).
struct SoftmapPlain {
    const float *x, *W, *gm, *mx, *rs, *dots;
    float *m, *gx, *gW;
    const unsigned *x_largest, *gm_largest;
    int B, I, M, parts, dot_ld;
    float scale, inv_tau;
    const SoftmapRange *range;  // pairs: what decided between them and planes
    const unsigned *tiny;       // and the values of gs ([0]) and gm ([1]) that they leave out
    const int2 *tiny_at;
};
#define SM_PT 128  // edge of a tile
#define SM_PLD 132 // its row in the LDS
template <int MODE>
__device__ void softmap_plain_tile(const SoftmapPlain &p, float (&As)[16][SM_PLD], float (&Bs)[16][SM_PLD], int r0, int c0) {
    const int R = MODE == 2 ? p.M : p.B, C = MODE == 0 ? p.M : p.I, K = MODE == 0 ? p.I : MODE == 1 ? p.M : p.B;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, kh = lane >> 5, l32 = lane & 31;
    const int wm = (wave >> 1) * 64, wn = (wave & 1) * 64;
    auto softmax = [&](int o, int i) -> float {
        return softmap_e(p.W[(size_t)o * p.I + i], p.mx[o], p.scale) * p.rs[o];
    };
    // (rows and columns past the end repeat the last and are not stored)
    auto a_at = [&](int row, int k) -> float {
        row = min(row, R - 1);
        // the forward's halved: a sum of weights that round to more than one must not overflow on the way
        return MODE == 0 ? 0.5f * p.x[(size_t)row * p.I + k] : MODE == 1 ? p.gm[(size_t)row * p.M + k] : p.gm[(size_t)k * p.M + row];
    };
    auto b_at = [&](int col, int k) -> float {
        col = min(col, C - 1);
        return MODE == 0 ? softmax(col, k) : MODE == 1 ? softmax(k, col) : p.x[(size_t)k * p.I + col];
    };
    // neighbouring threads along what is contiguous in memory: the reduction, or rows / columns
    constexpr bool A_ALONG_K = MODE != 2, B_ALONG_K = MODE == 0;
    float na[8], nb[8];
    auto fetch_as = [&](int k0, auto whole) {
        int t = tid;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            // addresses are made anew, and for two elements at a time: all of them do not fit the registers
            if (q % 2 == 0) asm volatile("" : "+v"(t)::"memory");
            const int e = q * 256 + t;
            const int ka = k0 + (A_ALONG_K ? e & 15 : e >> 7), kb = k0 + (B_ALONG_K ? e & 15 : e >> 7);
            const int ra = r0 + (A_ALONG_K ? e >> 4 : e & 127), cb = c0 + (B_ALONG_K ? e >> 4 : e & 127);
            na[q] = decltype(whole)::value || ka < K ? a_at(ra, ka) : 0.0f;
            nb[q] = decltype(whole)::value || kb < K ? b_at(cb, kb) : 0.0f;
        }
    };
    auto fetch = [&](int k0) {
        if (k0 + 16 <= K) fetch_as(k0, std::true_type{});
        else fetch_as(k0, std::false_type{});
    };
    floatx16 acc[2][2], sum[2][2];
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[t >> 1][t & 1][v] = sum[t >> 1][t & 1][v] = 0.0f;
    fetch(0);
    for (int k0 = 0; k0 < K; k0 += 16) {
        __syncthreads();
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int e = q * 256 + tid;
            if (A_ALONG_K) As[e & 15][e >> 4] = na[q];
            else As[e >> 7][e & 127] = na[q];
            if (B_ALONG_K) Bs[e & 15][e >> 4] = nb[q];
            else Bs[e >> 7][e & 127] = nb[q];
        }
        __syncthreads();
        if (k0 + 16 < K) fetch(k0 + 16);
#pragma unroll
        for (int kk = 0; kk < 8; ++kk) {
            const int k = 2 * kk + kh;
            const float a0 = As[k][wm + l32], a1 = As[k][wm + 32 + l32], b0 = Bs[k][wn + l32], b1 = Bs[k][wn + 32 + l32];
            acc[0][0] = __builtin_amdgcn_mfma_f32_32x32x2f32(a0, b0, acc[0][0], 0, 0, 0);
            acc[0][1] = __builtin_amdgcn_mfma_f32_32x32x2f32(a0, b1, acc[0][1], 0, 0, 0);
            acc[1][0] = __builtin_amdgcn_mfma_f32_32x32x2f32(a1, b0, acc[1][0], 0, 0, 0);
            acc[1][1] = __builtin_amdgcn_mfma_f32_32x32x2f32(a1, b1, acc[1][1], 0, 0, 0);
        }
        if ((k0 & 127) == 112 || k0 + 16 >= K) {
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    sum[t >> 1][t & 1][v] += acc[t >> 1][t & 1][v];
                    acc[t >> 1][t & 1][v] = 0.0f;
                }
        }
    }
    if (MODE == 2) {  // of the tile's rows: r, the maximum and rs / tau
        __syncthreads();
        if (tid < SM_PT) {
            const int row = min(r0 + tid, R - 1);
            float r = 0.0f;
            for (int q = 0; q < p.parts; ++q) r += p.dots[(size_t)q * p.dot_ld + row];
            As[0][tid] = r;
            As[1][tid] = p.mx[row];
            As[2][tid] = p.rs[row] * p.inv_tau;
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const int lr = wm + i * 32 + 8 * (v >> 2) + 4 * kh + (v & 3), row = r0 + lr;
            if (row >= R) continue;
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const int col = c0 + wn + j * 32 + l32;
                if (col >= C) continue;
                float o = sum[i][j][v];
                if (MODE == 0) {  // a mean of finite values is no larger than they are
                    const bool finite = __builtin_isfinite(o);
                    o *= 2.0f;
                    if (finite) o = fminf(fmaxf(o, -3.402823466e38f), 3.402823466e38f);
                    p.m[(size_t)row * C + col] = o;
                } else if (MODE == 1) {
                    p.gx[(size_t)row * C + col] = o;
                } else {
                    const size_t at = (size_t)row * C + col;
                    p.gW[at] = (o - As[0][lr]) * (softmap_e(p.W[at], As[1][lr], p.scale) * As[2][lr]);
                }
            }
        }
}
// The terms of the values that the pairs leave out, added to gx (MODE 1) or gW (MODE 2): a block has a row of the result and
// 256 of its columns, and takes the row's values in order, so that the sums are the same every time.
template <int MODE>
__device__ void softmap_tiny_terms(const SoftmapPlain &p, const int2 *__restrict__ found, int count, int2 *list) {
    __syncthreads();  // (`list`, of twice SM_TINY_MOST, may hold the other result's)
    int2 *as_found = list + SM_TINY_MOST;
    for (int e = threadIdx.x; e < count; e += 256) as_found[e] = found[e];
    __syncthreads();
    for (int e = threadIdx.x; e < count; e += 256) {
        const int2 mine = as_found[e];
        int rank = 0;
        for (int q = 0; q < count; ++q) {
            const int2 v = as_found[q];
            rank += v.x < mine.x || (v.x == mine.x && v.y < mine.y) ? 1 : 0;
        }
        list[rank] = mine;
    }
    __syncthreads();
    const int strips = (p.I + 255) / 256;
    for (int it = blockIdx.x; it < count * strips; it += gridDim.x) {
        const int first = it / strips, i = it % strips * 256 + (int)threadIdx.x, row = list[first].x;
        if ((first > 0 && list[first - 1].x == row) || i >= p.I) continue;
        float sum = 0.0f;
        for (int e = first; e < count && list[e].x == row; ++e) {
            const int k = list[e].y;
            if (MODE == 1) sum = fmaf(p.gm[(size_t)row * p.M + k] * p.rs[k], softmap_e(p.W[(size_t)k * p.I + i], p.mx[k], p.scale), sum);
            else sum = fmaf(p.gm[(size_t)k * p.M + row], p.x[(size_t)k * p.I + i], sum);
        }
        const size_t at = (size_t)row * p.I + i;
        if (MODE == 1) p.gx[at] += sum;
        else p.gW[at] = fmaf(sum, softmap_e(p.W[at], p.mx[row], p.scale) * (p.rs[row] * p.inv_tau), p.gW[at]);
    }
}
template <bool BWD>
__global__ __launch_bounds__(256, 2) void softmap_plain(SoftmapPlain p) {
    __shared__ float As[16][SM_PLD], Bs[16][SM_PLD];
    const float x = softmap_largest(p.x_largest), gm = BWD ? softmap_largest(p.gm_largest) : 0.0f;
    const int bt = (p.B + SM_PT - 1) / SM_PT, it = (p.I + SM_PT - 1) / SM_PT, mt = (p.M + SM_PT - 1) / SM_PT;
    // the largest sums the planes' accumulators could see, without the factor (a NaN compares false)
    if (!BWD) {
        if (x * (float)p.I < SM_BOUND) return;
        for (long long t = blockIdx.x; t < (long long)bt * mt; t += gridDim.x)
            softmap_plain_tile<0>(p, As, Bs, (int)(t % bt) * SM_PT, (int)(t / bt) * SM_PT);
        return;
    }
    __shared__ int2 list[BWD ? 2 * SM_TINY_MOST : 1];
    // (values are left out where the pairs ran: not by planes, which they gave way to beyond SM_TINY_MOST)
    const int rows_tiny = p.range && !softmap_wide(p.range) && p.tiny[0] <= SM_TINY_MOST ? (int)p.tiny[0] : 0;
    const int cols_tiny = p.range && !softmap_x_wide(p.range) && p.tiny[1] <= SM_TINY_MOST ? (int)p.tiny[1] : 0;
    if (!(gm * (float)p.M < SM_BOUND)) {
        for (long long t = blockIdx.x; t < (long long)bt * it; t += gridDim.x)
            softmap_plain_tile<1>(p, As, Bs, (int)(t / it) * SM_PT, (int)(t % it) * SM_PT);
    } else if (rows_tiny > 0) {
        softmap_tiny_terms<1>(p, p.tiny_at, rows_tiny, list);
    }
    if (!(gm * (float)p.B * x < SM_BOUND)) {
        for (long long t = blockIdx.x; t < (long long)mt * it; t += gridDim.x)
            softmap_plain_tile<2>(p, As, Bs, (int)(t / it) * SM_PT, (int)(t % it) * SM_PT);
    } else if (cols_tiny > 0) {
        softmap_tiny_terms<2>(p, p.tiny_at + SM_TINY_MOST, cols_tiny, list);
    }
}
#define SM_PLAIN_BLOCKS 512  // two per CU

// ---------------------------------------------------------------------------------
static int softmap_check(int B, int I, int M, int precision) {
    if (B <= 0 || I <= 0 || M <= 0) return DL_ERR_SHAPE;
    if (precision != 0 && precision != 1) return DL_ERR_UNSUPPORTED;
    return DL_OK;
}

static inline int softmap_round(int v, int to) { return dl_ceil_div(v, to) * to; }

// Sizes of the padded operands: whole tiles of rows, columns and reduction stages on every side they are used on.
struct SoftmapShape {
    int B, I, M, np;
    int Bp, Ip, Mp;                                   // padded
    int fa;                                           // MFMA tiles of 32 batch rows per wavefront
    int depth;                                        // reduction steps per stage
    int row_tiles, fwd_col_tiles, gx_col_tiles;       // forward and gx
    int fwd_stages, fwd_chunk, fwd_chunks;            // reduction over I
    int gx_stages, gx_chunk, gx_chunks;               // reduction over M
    size_t e_plane, x_plane, g_plane;                 // bytes of a plane of E, of x, of gs
    bool pairs;                                       // precision 0: pairs where the values allow them
    int pair_row_tiles, pair_fwd_chunk, pair_fwd_chunks, pair_gx_chunk, pair_gx_chunks;
};

// A product whose tiles do not fill the card's 512 resident blocks (two per CU) cuts its reduction into chunks, whose
// partial results are added in order by a second launch.  gx at 512 x 3136 x 48000 (50 tiles): 10 chunks, one round of 500
// blocks.  A chunk keeps at least 8 stages, below which a block is mostly its own start and end.
static void softmap_chunks(int stages, long long tiles, long long blocks, int *chunk, int *chunks) {
    long long n = blocks / tiles;
    if (n > stages / 8) n = stages / 8;
    if (n < 1) n = 1;
    *chunk = dl_ceil_div(stages, n);
    *chunks = dl_ceil_div(stages, *chunk);
}
// Pairs cost a pass over x and one over gm and ten launches of about 5 us a step, six of which end at once.  Measured, forward +
// backward, planes against pairs: 512 x 512 x 24000 (6.3e9) 332 -> 322 us (planes all the same, see below), 64 x 3136 x 30000 (6.0e9) 716 -> 594, 300 x 1500 x 20000
// (9.0e9) 578 -> 468, 512 x 3136 x 48000 2659 -> 2562 where E spans too much; below, planes.
#define SM_PAIR_WORK 6e9
// gx in chunks of the reduction shorter than this many stages takes the planes, and with it the whole call, which has one form of
// E: a pair's 23 bits are seen there, where longer sums round more than that.  Error of gx against float64 (2-norm, units of 1e-7),
// planes / pairs, by the planes' stages per chunk, W of N(0, 1.5), gm of N(0, 1): 24 (512 x 512 x 24000) 1.28 / 1.42, 25 (512 x 3136 x 4000)
// 1.23 / 1.38, 32 1.29 / 1.36, 36 1.38 / 1.41, 39 1.37 / 1.35, 41 1.41 / 1.39, 47 1.49 / 1.40, 57 1.57 / 1.41, 104 2.03 / 1.50, 300
// (512 x 3136 x 48000) 3.18 / 1.73; the same with W of N(0, 0.1) and with gm a product of two N(0, 1).  m and gW are closer with pairs at
// all of these, by 0.2 to 0.7.
#define SM_PAIR_CHUNK 40
static SoftmapShape softmap_shape(int B, int I, int M, int precision) {
    SoftmapShape h;
    h.B = B; h.I = I; h.M = M;
    h.np = precision == 1 ? 1 : 3;
    h.pairs = h.np == 3 && (double)B * I * M >= SM_PAIR_WORK;
    h.fa = B > 128 ? 4 : 2;
    h.depth = h.np == 1 ? 32 : 16;
    h.Bp = softmap_round(B, 64 * h.fa);
    h.Ip = softmap_round(I, 128);
    h.Mp = softmap_round(M, 256);
    h.row_tiles = h.Bp / (64 * h.fa);
    h.fwd_col_tiles = dl_ceil_div(M, SM_TC);
    h.gx_col_tiles = h.Ip / SM_TC;
    h.fwd_stages = dl_ceil_div(I, h.depth);
    h.gx_stages = dl_ceil_div(M, h.depth);
    softmap_chunks(h.fwd_stages, (long long)h.row_tiles * h.fwd_col_tiles, 512, &h.fwd_chunk, &h.fwd_chunks);
    softmap_chunks(h.gx_stages, (long long)h.row_tiles * h.gx_col_tiles, 512, &h.gx_chunk, &h.gx_chunks);
    h.pairs = h.pairs && h.gx_chunk >= SM_PAIR_CHUNK;
    h.pair_row_tiles = h.Bp / 128;
    softmap_chunks(h.fwd_stages, (long long)h.pair_row_tiles * h.fwd_col_tiles, 512, &h.pair_fwd_chunk, &h.pair_fwd_chunks);
    softmap_chunks(h.gx_stages, (long long)h.pair_row_tiles * h.gx_col_tiles, 1024, &h.pair_gx_chunk, &h.pair_gx_chunks);
    h.e_plane = dl_align256((size_t)(h.Mp / 8) * h.Ip * SM_UNIT);
    h.x_plane = dl_align256((size_t)(h.Ip / 8) * h.Bp * SM_UNIT);
    h.g_plane = dl_align256((size_t)(h.Mp / 8) * h.Bp * SM_UNIT);
    return h;
}

// `stats`, kept for the backward: max [Mp], 1/sum [Mp], x in units along the inputs (the forward's operand), E, and with
// fp32 operands the range (its first word the largest magnitude of x)
static inline size_t softmap_vec_bytes(const SoftmapShape &h) { return dl_align256((size_t)h.Mp * sizeof(float)); }
extern "C" size_t dl_soft_map_saved_bytes(int B, int I, int M, int precision) {
    if (B <= 0 || I <= 0 || M <= 0) return 256;
    const SoftmapShape h = softmap_shape(B, I, M, precision);
    return 2 * softmap_vec_bytes(h) + h.np * (h.x_plane + h.e_plane) + (h.np > 1 ? 256 : 0);
}

// workspace: partial products of the forward or of gx, partial r, x and gm in units along the batch, gs along the rows of W, the
// largest magnitude of gm (and how many values of gs and gm the pairs leave out), those of the rows of gs and the columns of gm,
// where the values left out are
static inline size_t softmap_part_bytes(const SoftmapShape &h) {
    int nf = h.fwd_chunks, ng = h.gx_chunks;
    if (h.pairs && h.pair_fwd_chunks > nf) nf = h.pair_fwd_chunks;
    if (h.pairs && h.pair_gx_chunks > ng) ng = h.pair_gx_chunks;
    const size_t fwd = nf > 1 ? (size_t)nf * h.B * h.M : 0, gx = ng > 1 ? (size_t)ng * h.B * h.I : 0;
    return dl_align256((fwd > gx ? fwd : gx) * sizeof(float));
}
static inline size_t softmap_dots_bytes(const SoftmapShape &h) {
    return dl_align256((size_t)(h.Bp / 64) * h.Mp * sizeof(float));
}
extern "C" size_t dl_soft_map_workspace_bytes(int B, int I, int M, int precision) {
    if (B <= 0 || I <= 0 || M <= 0) return 256;
    const SoftmapShape h = softmap_shape(B, I, M, precision);
    return 256 + softmap_part_bytes(h) + softmap_dots_bytes(h) + h.np * (h.x_plane + 2 * h.g_plane) +
           (h.pairs ? dl_align256((size_t)(h.Bp + h.Mp) * sizeof(unsigned)) + 2 * SM_TINY_MOST * sizeof(int2) : 0);
}

template <int NP>
static void softmap_stats_launch(const SoftmapShape &h, const float *W, float scale, float *mx, float *rs, char *E,
                                 unsigned *largest, SoftmapRange *range, hipStream_t s) {
    const int grid = h.Mp / 8;
#define SM_STATS(T, NQ) \
    DL_TIMED("softmap_rowstats", s, (softmap_rowstats<NP, T, NQ><<<grid, T, 0, s>>>(W, scale, mx, rs, E, h.e_plane, h.M, h.I, h.Ip, largest, range)))
    if (h.Ip <= 256 * 4) SM_STATS(256, 4);
    else if (h.Ip <= 256 * 8) SM_STATS(256, 8);
    else if (h.Ip <= 512 * 8) SM_STATS(512, 8);
    else if (h.Ip <= 1024 * 8) SM_STATS(1024, 8);
    else SM_STATS(1024, 0);
#undef SM_STATS
}
static void softmap_pack_launch(int np, const float *src, const float *colscale, const float *other, float *dots, char *rows8,
                                size_t rows_plane, char *cols8, size_t cols_plane, int R, int C, int Rp, int Cp, float alternate,
                                unsigned *largest, unsigned *clear, const SoftmapRange *range, const unsigned *row_max,
                                const unsigned *col_max, unsigned *tiny, int2 *tiny_at, bool again, hipStream_t s) {
    const int grid = Cp / 64 * dl_ceil_div(Rp, 64);
#define SM_PACK(NP) \
    DL_TIMED("softmap_pack", s, (softmap_pack<NP><<<grid, 256, 0, s>>>(src, colscale, other, dots, rows8, rows_plane, cols8, cols_plane, R, C, Rp, Cp, alternate, largest, clear, range, row_max, col_max, tiny, tiny_at, again)))
    if (np == 1) SM_PACK(1);
    else if (range) SM_PACK(2);
    else SM_PACK(3);
#undef SM_PACK
}
static void softmap_reduce(const float *part, float *out, long long total, int chunks, const SoftmapRange *range, const unsigned *tiny,
                           int wide_chunks, hipStream_t s) {
    if (total % 4 == 0 && ((uintptr_t)out & 15) == 0)
        DL_TIMED("softmap_reduce_chunks", s,
                 (softmap_reduce_chunks<4><<<dl_ceil_div(total / 4, 256), 256, 0, s>>>(part, out, total, chunks, range, tiny, wide_chunks)));
    else
        DL_TIMED("softmap_reduce_chunks", s,
                 (softmap_reduce_chunks<1><<<dl_ceil_div(total, 256), 256, 0, s>>>(part, out, total, chunks, range, tiny, wide_chunks)));
}
template <int MODE>
static void softmap_product(const char *name, const SoftmapShape &h, int fa, const SoftmapArgs &g, hipStream_t s) {
    if (h.np == 1) {
        if (fa == 4) DL_TIMED(name, s, (softmap_launch<MODE, 1, 4>(g, s)));
        else DL_TIMED(name, s, (softmap_launch<MODE, 1, 2>(g, s)));
    } else {
        if (fa == 4) DL_TIMED(name, s, (softmap_launch<MODE, 3, 4>(g, s)));
        else DL_TIMED(name, s, (softmap_launch<MODE, 3, 2>(g, s)));
    }
}

static inline int softmap_plain_grid(long long tiles) { return tiles < SM_PLAIN_BLOCKS ? (int)tiles : SM_PLAIN_BLOCKS; }

extern "C" int dl_soft_map_fwd(const float *x, const float *W, float tau, float *m, float *stats, void *ws,
                               size_t ws_bytes, int B, int I, int M, int precision, void *stream) {
    if (!x || !W || !m || !stats) return DL_ERR_NULL;
    int rc = softmap_check(B, I, M, precision);
    if (rc) return rc;
    if (!(tau > 0.0f)) return DL_ERR_SHAPE;
    if (precision == 1 && !ws) return DL_ERR_NULL;
    if (precision == 1 && ws_bytes < dl_soft_map_workspace_bytes(B, I, M, precision)) return DL_ERR_WORKSPACE;
    hipStream_t s = (hipStream_t)stream;
    SoftmapShape h = softmap_shape(B, I, M, precision);
    if (!ws || ws_bytes < dl_soft_map_workspace_bytes(B, I, M, precision)) {
        h.fwd_chunk = h.pair_fwd_chunk = h.fwd_stages;
        h.fwd_chunks = h.pair_fwd_chunks = 1;
    }
    char *p = (char *)stats;
    float *mx = (float *)p, *rs = (float *)(p + softmap_vec_bytes(h));
    char *x8 = p + 2 * softmap_vec_bytes(h), *E = x8 + h.np * h.x_plane;
    unsigned *x_largest = h.np > 1 ? (unsigned *)(E + h.np * h.e_plane) : nullptr;
    SoftmapRange *range = h.pairs ? (SoftmapRange *)x_largest : nullptr;
    const float scale = SM_LOG2E / tau;
    if (h.np == 1) softmap_stats_launch<1>(h, W, scale, mx, rs, E, nullptr, nullptr, s);
    else if (!h.pairs) softmap_stats_launch<3>(h, W, scale, mx, rs, E, x_largest, nullptr, s);
    else {
        DL_TIMED("softmap_clear", s, (softmap_clear<<<1, 256, 0, s>>>(range, nullptr, 0)));
        const int grid = dl_ceil_div((long long)B * I, 256 * 8);
        DL_TIMED("softmap_scan", s, (softmap_scan_x<<<grid < 256 ? grid : 256, 256, 0, s>>>(x, (long long)B * I, range)));
        softmap_stats_launch<2>(h, W, scale, mx, rs, E, nullptr, range, s);
        softmap_stats_launch<3>(h, W, scale, mx, rs, E, nullptr, range, s);
    }
    softmap_pack_launch(h.np, x, nullptr, nullptr, nullptr, nullptr, 0, x8, h.x_plane, B, I, h.Bp, h.Ip, 1.0f, h.pairs ? nullptr : x_largest,
                        nullptr, range, nullptr, nullptr, nullptr, nullptr, false, s);
    SoftmapArgs g{};
    g.A = x8; g.a_plane = h.x_plane; g.lda = h.Bp;
    g.Bm = E; g.b_plane = h.e_plane; g.ldb = h.Ip;
    g.R = B; g.C = M;
    g.stages = h.fwd_stages;
    g.col_tiles = h.fwd_col_tiles;
    g.rs = rs; g.range = range;
    auto product = [&](int row_tiles, int chunk, int chunks) {
        g.out = chunks > 1 ? (float *)ws : m;
        g.chunk_stages = chunk;
        g.inner_count = row_tiles; g.outer_count = h.fwd_col_tiles * chunks;
    };
    if (h.pairs) {
        product(h.pair_row_tiles, h.pair_fwd_chunk, h.pair_fwd_chunks);
        DL_TIMED("softmap_fwd", s, (softmap_launch<0, 2, 2>(g, s)));
    }
    product(h.row_tiles, h.fwd_chunk, h.fwd_chunks);
    softmap_product<0>("softmap_fwd", h, h.fa, g, s);
    if (h.pairs ? h.pair_fwd_chunks > 1 || h.fwd_chunks > 1 : h.fwd_chunks > 1)
        softmap_reduce((const float *)ws, m, (long long)B * M, h.pairs ? h.pair_fwd_chunks : h.fwd_chunks, range, nullptr, h.fwd_chunks, s);
    if (h.np > 1) {
        SoftmapPlain q{};
        q.x = x; q.W = W; q.mx = mx; q.rs = rs; q.m = m; q.x_largest = x_largest;
        q.B = B; q.I = I; q.M = M; q.scale = SM_LOG2E / tau;
        const int grid = softmap_plain_grid((long long)dl_ceil_div(B, SM_PT) * dl_ceil_div(M, SM_PT));
        DL_TIMED("softmap_plain", s, (softmap_plain<false><<<grid, 256, 0, s>>>(q)));
    }
    return dl_launch_status();
}

extern "C" int dl_soft_map_bwd(const float *x, const float *W, float tau, const float *m, const float *stats,
                               const float *gm, float *gx, float *gW, void *ws, size_t ws_bytes, int B, int I, int M,
                               int precision, void *stream) {
    if (!x || !W || !m || !stats || !gm || !gx || !gW || !ws) return DL_ERR_NULL;
    int rc = softmap_check(B, I, M, precision);
    if (rc) return rc;
    if (!(tau > 0.0f)) return DL_ERR_SHAPE;
    if (ws_bytes < dl_soft_map_workspace_bytes(B, I, M, precision)) return DL_ERR_WORKSPACE;
    hipStream_t s = (hipStream_t)stream;
    const SoftmapShape h = softmap_shape(B, I, M, precision);
    const char *p = (const char *)stats;
    const float *mx = (const float *)p, *rs = (const float *)(p + softmap_vec_bytes(h));
    const char *E = p + 2 * softmap_vec_bytes(h) + h.np * h.x_plane;
    const unsigned *x_largest = h.np > 1 ? (const unsigned *)(E + h.np * h.e_plane) : nullptr;
    char *w = (char *)ws;
    float *part = (float *)w; w += softmap_part_bytes(h);
    float *dots = (float *)w; w += softmap_dots_bytes(h);
    char *xb = w; w += h.np * h.x_plane;     // x  [Bp/8][Ip]
    char *gb = w; w += h.np * h.g_plane;     // gm [Bp/8][Mp]
    char *go = w; w += h.np * h.g_plane;     // gs [Mp/8][Bp]
    unsigned *gm_largest = h.np > 1 ? (unsigned *)w : nullptr;
    const SoftmapRange *range = h.pairs ? (const SoftmapRange *)x_largest : nullptr;
    unsigned *row_max = h.pairs ? (unsigned *)(w + 256) : nullptr, *col_max = h.pairs ? row_max + h.Bp : nullptr;
    if (h.pairs) {
        const int words = 64 + h.Bp + h.Mp, strips = dl_ceil_div(M, 64 * SM_SCAN_TILES);
        DL_TIMED("softmap_clear", s, (softmap_clear<<<dl_ceil_div(words, 256), 256, 0, s>>>(nullptr, gm_largest, words)));
        DL_TIMED("softmap_scan", s, (softmap_scan_grad<<<(unsigned)strips * dl_ceil_div(B, 64), 256, 0, s>>>(gm, rs, row_max, col_max, gm_largest, range, B, M, strips)));
    }
    unsigned *tiny = h.pairs ? gm_largest + 2 : nullptr;
    int2 *tiny_at = h.pairs ? (int2 *)(w + 256 + dl_align256((size_t)(h.Bp + h.Mp) * sizeof(unsigned))) : nullptr;
    auto pack_x = [&]() {
        softmap_pack_launch(h.np, x, nullptr, nullptr, nullptr, xb, h.x_plane, nullptr, 0, B, I, h.Bp, h.Ip, 1.0f, nullptr,
                            h.pairs ? nullptr : gm_largest, range, nullptr, nullptr, tiny, nullptr, false, s);
    };
    if (!h.pairs) pack_x();  // which clears gm_largest for the next
    softmap_pack_launch(h.np, gm, rs, m, dots, gb, h.g_plane, go, h.g_plane, B, M, h.Bp, h.Mp, -1.0f, gm_largest, nullptr,
                        range, row_max, col_max, tiny, tiny_at, false, s);
    if (h.pairs) {
        softmap_pack_launch(h.np, gm, rs, nullptr, nullptr, gb, h.g_plane, go, h.g_plane, B, M, h.Bp, h.Mp, -1.0f, nullptr, nullptr,
                            range, row_max, col_max, tiny, nullptr, true, s);
        pack_x();
    }
    SoftmapArgs g{};
    g.A = go; g.a_plane = h.g_plane; g.lda = h.Bp;
    g.Bm = E; g.b_plane = h.e_plane; g.ldb = h.Ip;
    g.R = B; g.C = I;
    g.stages = h.gx_stages;
    g.col_tiles = h.gx_col_tiles;
    g.range = range; g.row_max = row_max; g.tiny = tiny;
    auto product = [&](int row_tiles, int chunk, int chunks) {
        g.out = chunks > 1 ? part : gx;
        g.chunk_stages = chunk;
        g.inner_count = row_tiles; g.outer_count = h.gx_col_tiles * chunks;
    };
    if (h.pairs) {
        product(h.pair_row_tiles, h.pair_gx_chunk, h.pair_gx_chunks);
        DL_TIMED("softmap_gx", s, (softmap_launch<1, 2, 2>(g, s)));
    }
    product(h.row_tiles, h.gx_chunk, h.gx_chunks);
    softmap_product<1>("softmap_gx", h, h.fa, g, s);
    if (h.pairs) {
        if (h.fa == 4) DL_TIMED("softmap_gx", s, (softmap_launch<1, 3, 4, 2>(g, s)));
        else DL_TIMED("softmap_gx", s, (softmap_launch<1, 3, 2, 2>(g, s)));
    }
    if (h.pairs ? h.pair_gx_chunks > 1 || h.gx_chunks > 1 : h.gx_chunks > 1)
        softmap_reduce(part, gx, (long long)B * I, h.pairs ? h.pair_gx_chunks : h.gx_chunks, range, tiny, h.gx_chunks, s);
    // gW: tiles of 256 rows of W where they fill the card, else of 128
    const int fa = (long long)(h.Mp / 256) * h.gx_col_tiles >= 512 ? 4 : 2;
    SoftmapArgs q{};
    q.A = gb; q.a_plane = h.g_plane; q.lda = h.Mp;
    q.Bm = xb; q.b_plane = h.x_plane; q.ldb = h.Ip;
    q.out = gW;
    q.R = M; q.C = I;
    q.stages = dl_ceil_div(B, h.depth); q.chunk_stages = q.stages;
    q.inner_count = h.gx_col_tiles; q.col_tiles = h.gx_col_tiles;
    q.rs = rs; q.dots = dots; q.parts = dl_ceil_div(B, 64); q.dot_ld = h.Mp;
    q.mx = mx; q.W = W; q.E = E; q.lde = h.Ip; q.scale = SM_LOG2E / tau; q.inv_tau = 1.0f / tau;
    q.range = range; q.row_max = col_max; q.tiny = h.pairs ? tiny + 1 : nullptr;
    q.vec_out = (((uintptr_t)W | (uintptr_t)gW) & 15) == 0;
    if (h.pairs) {
        q.outer_count = dl_ceil_div(M, 128);
        DL_TIMED("softmap_gw", s, (softmap_launch<2, 2, 2>(q, s)));
    }
    q.outer_count = dl_ceil_div(M, 64 * fa);
    softmap_product<2>("softmap_gw", h, fa, q, s);
    if (h.np > 1) {
        SoftmapPlain u{};
        u.x = x; u.W = W; u.gm = gm; u.mx = mx; u.rs = rs; u.dots = dots; u.gx = gx; u.gW = gW;
        u.x_largest = x_largest; u.gm_largest = gm_largest;
        u.range = range; u.tiny = tiny; u.tiny_at = tiny_at;
        u.B = B; u.I = I; u.M = M; u.parts = q.parts; u.dot_ld = q.dot_ld; u.scale = q.scale; u.inv_tau = q.inv_tau;
        const int grid = softmap_plain_grid((long long)(M > B ? dl_ceil_div(M, SM_PT) : dl_ceil_div(B, SM_PT)) * dl_ceil_div(I, SM_PT));
        DL_TIMED("softmap_plain", s, (softmap_plain<true><<<grid, 256, 0, s>>>(u)));
    }
    return dl_launch_status();
}
