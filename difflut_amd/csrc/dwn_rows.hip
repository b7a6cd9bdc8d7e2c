// A DWN layer on few rows, one launch whatever comes in and goes out.  Rows are taken eight at a time: a block turns the eight rows
// of its input into a byte per input in the LDS - bit r = row r, thresholded, or compared with a thermometer's thresholds, of which
// the code is then never written - or reads these bytes out of bit-planes.  A thread is a column: its k bytes hold the addresses of
// the eight rows, a table entry is read for each, and the results leave as rows of y, as a byte of the column's plane word, or summed
// over the columns of a group.  The addresses of a column's eight rows, for the backward, are eight bytes in a row.
// What bounds it is the chain of a launch (input, indices, table entries: three trips to memory) and, with more columns, the
// eight table entries at random places, 64 cycles of the texture addresser per load.  On many rows the kernels with a lane
// per row, which read a table once per 64 rows, are better: the rules where this is called say from where on.  k <= 6.
//   R = 1: fewer than eight rows of a model whose logits are asked for; inputs are read at their places.
#include "dwn_rows.h"

template <int K, bool PLANES, int R>
__global__ __launch_bounds__(1024) void dwn_rows(DwnRows a, int span) {
    constexpr int L = 1 << K;
    static_assert(R == 8 || R == 1, "a byte of rows, or one row");
    extern __shared__ uint8_t code[];  // [input], bit = row
    __shared__ float part[16][R];
    const int tid = threadIdx.x, b0 = blockIdx.y * R, rows = min(R, a.B - b0);
    const int NO = a.N * a.O, width = a.thr ? a.I / a.nbits : a.I;
    const int c_lo = blockIdx.x * span, c_hi = min(NO, c_lo + span);
    if (R == 8 && rows <= 0) {  // eight rows of the last tile that the batch does not have: zeros
        for (int c = c_lo + tid; c < c_hi; c += blockDim.x) {
            if (a.planes_out) a.planes_out[((size_t)(b0 >> 6) * NO + c) * 8 + ((b0 & 63) >> 3)] = 0;
            if (a.saved && c % a.O == 0)
                *reinterpret_cast<uint2 *>(a.saved + ((size_t)(b0 >> 6) * a.N + c / a.O) * 64 + (b0 & 63)) = make_uint2(0, 0);
        }
        return;
    }
    if constexpr (!PLANES && R == 8) {
        const float *from = a.x + (size_t)b0 * width;
        for (int f = tid; f < width; f += blockDim.x) {
            float v[8];
#pragma unroll
            for (int r = 0; r < 8; ++r) v[r] = from[(size_t)min(r, rows - 1) * width + f];
            if (a.thr) {
                for (int q = 0; q < a.nbits; ++q) {
                    const float limit = a.thr[f * a.nbits + q];
                    unsigned byte = 0;
#pragma unroll
                    for (int r = 0; r < 8; ++r) byte |= v[r] > limit ? 1u << r : 0u;
                    code[f * a.nbits + q] = (uint8_t)byte;
                }
            } else {
                unsigned byte = 0;
#pragma unroll
                for (int r = 0; r < 8; ++r) byte |= v[r] >= 0.5f ? 1u << r : 0u;
                code[f] = (uint8_t)byte;
            }
        }
        __syncthreads();
    }
    float sum[R];
#pragma unroll
    for (int r = 0; r < R; ++r) sum[r] = 0.0f;
    for (int c0 = c_lo; c0 < c_hi; c0 += blockDim.x) {
        const bool live = c0 + tid < c_hi;
        const int c = min(c0 + tid, c_hi - 1), n = c / a.O;
        int idx[K];
#pragma unroll
        for (int j = 0; j < K; ++j) idx[j] = a.idx32[(size_t)n * K + j];
        unsigned byte[K];
#pragma unroll
        for (int j = 0; j < K; ++j) {
            if constexpr (PLANES) {
                byte[j] = a.planes[((size_t)(b0 >> 6) * a.I + idx[j]) * 8 + ((b0 & 63) >> 3)] >> (b0 & 7);
            } else if constexpr (R == 8) {
                byte[j] = code[idx[j]];
            } else if (a.thr) {
                byte[j] = a.x[(size_t)b0 * width + (unsigned)idx[j] / (unsigned)a.nbits] > a.thr[idx[j]] ? 1u : 0u;
            } else {
                byte[j] = a.x[(size_t)b0 * width + idx[j]] >= 0.5f ? 1u : 0u;
            }
        }
        unsigned addr[R];
        float v[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            addr[r] = 0;
#pragma unroll
            for (int j = 0; j < K; ++j) addr[r] |= ((byte[j] >> r) & 1u) << j;
            v[r] = a.luts[(size_t)c * L + addr[r]];
        }
        unsigned ones = 0;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            ones |= r < rows && v[r] >= 0.5f ? 1u << r : 0u;
            if (!a.saved) v[r] = v[r] >= 0.5f ? 1.0f : 0.0f;
            sum[r] += live ? v[r] : 0.0f;
        }
        if (!live) continue;
        if (a.y) {
#pragma unroll
            for (int r = 0; r < R; ++r)
                if (r < rows) a.y[(size_t)(b0 + r) * NO + c] = v[r];
        }
        if constexpr (R == 8) {
            const int at = b0 & 63;
            if (a.planes_out) a.planes_out[((size_t)(b0 >> 6) * NO + c) * 8 + (at >> 3)] = (uint8_t)ones;
            if (a.saved && c == n * a.O) {
                unsigned lo = 0, hi = 0;
#pragma unroll
                for (int r = 0; r < 8; ++r)
                    if (r < rows) (r < 4 ? lo : hi) |= addr[r] << (8 * (r & 3));
                *reinterpret_cast<uint2 *>(a.saved + ((size_t)(b0 >> 6) * a.N + n) * 64 + at) = make_uint2(lo, hi);
            }
        }
    }
    if (!a.logits) return;
    // over the lanes, then over the wavefronts: a fixed order (of zeros and ones, any order gives the same)
#pragma unroll
    for (int r = 0; r < R; ++r)
        for (int off = 32; off > 0; off >>= 1) sum[r] += __shfl_xor(sum[r], off);
    if ((tid & 63) == 0) {
#pragma unroll
        for (int r = 0; r < R; ++r) part[tid >> 6][r] = sum[r];
    }
    __syncthreads();
    if (tid < rows) {
        float total = part[0][tid];
        for (int w = 1; w < (int)blockDim.x >> 6; ++w) total += part[w][tid];
        a.logits[(size_t)(b0 + tid) * a.groups + blockIdx.x] = total * a.inv_tau;
    }
}

struct DwnRowsGrid {
    int R, by, bx, threads, span, blocks;  // rows and columns of a block; blocks that have rows
};
// width: features or values that a block turns, 0 with planes; groups: of a head, else 0
static DwnRowsGrid dwn_rows_grid(int B, int width, int NO, int groups, bool planes_out, bool saved) {
    DwnRowsGrid q;
    q.R = groups && !saved && B < 8 ? 1 : 8;
    const int rows_by = dl_ceil_div(B, q.R);
    q.by = planes_out || saved ? (B + 63) / 64 * 8 : rows_by;
    // a thread per column, more where the input has more values to turn than that; blocks of 1024 share the columns as far as two
    // blocks per CU (of one group each: the groups)
    const int columns = groups ? (NO + groups - 1) / groups : NO;
    int threads = width == 0 || q.R == 1 || columns > width ? columns : width;
    if (groups && threads > 512 && (long long)groups * q.by > 256) threads = columns > 512 ? columns : 512;
    threads = q.threads = threads >= 1024 ? 1024 : (threads + 63) / 64 * 64;
    int bx = groups, span = columns;
    if (!groups) {
        bx = dl_ceil_div(NO, threads);
        if (bx > 1 && (long long)bx * q.by > 512) bx = q.by >= 512 ? 1 : dl_ceil_div(512, q.by) < bx ? dl_ceil_div(512, q.by) : bx;
        span = dl_ceil_div(dl_ceil_div(NO, bx), threads) * threads;
        bx = dl_ceil_div(NO, span);
    }
    q.bx = bx, q.span = span, q.blocks = bx * rows_by;
    return q;
}
// What the launch takes on the device as a layer under a head, us; the same arguments, width features or values of nbits columns each.  Terms:
// a launch and its blocks' threads; the turn of a block's eight rows (width 0: none) and its passes over the columns, as often as blocks
// follow one another on a CU; what all blocks read of x; outputs, and table entries, which of large tables come from further away.  Fitted to 16478 sizes (k = 2-6,
// 1-768 rows, 8-64512 inputs, 200-8000 columns in 1-20 groups, both modes), 7-9 % rms.
double dwn_rows_us(int B, int width, int nbits, int NO, int k, int groups, bool training) {
    const DwnRowsGrid q = dwn_rows_grid(B, width, NO, groups, false, training);
    const double passes = dl_ceil_div(q.span, q.threads), table = (1 << k) / 64.0, outputs = (double)B * NO * 1e-6, wide = q.threads / 1024.0;
    if (q.R == 1) return 1.9 + wide + passes * (0.35 + 0.18 * k + (width ? 0.3 : 0.0)) + 9.6 * outputs;
    const int in_lds = width ? (160 << 10) / (width * nbits + 512) : 32, per_cu = 2048 / q.threads < in_lds ? 2048 / q.threads : in_lds;
    double rounds = q.blocks / (256.0 * (per_cu > 0 ? per_cu : 1));
    if (rounds < 1.0) rounds = 1.0;
    const double fill = q.blocks / 256.0 * wide, turned = rounds * passes, entries = 1e-4 * NO * table;
    if (!width)
        return 0.59 + 2.98 * wide + turned * (2.54 + 0.35 * table + (training ? 0.32 : 0.0)) + 1.04 * outputs * table + 2.34 * fill + 0.85 * entries;
    return 1.54 + 2.38 * wide + rounds * dl_ceil_div(width, q.threads) * (0.34 + 0.1 * nbits) + turned * (1.62 + 0.09 * table + (training ? 0.43 : 0.0)) +
           0.64e-6 * q.blocks * width * nbits + outputs * (0.67 + 0.42 * table) + 1.22 * fill + 0.59 * entries;
}
// Whether it is the better launch for a layer that writes planes.  A first one: every block turns the whole input of its eight rows, so
// up to 8192 inputs, 1.5 million for all blocks and 256 blocks.  us on the device, code or packing and the layer / rows, nodes of six
// inputs, 3136 inputs: 4000 columns B = 64 10.6 / 8.2, 300 10.9 / 8.8, 768 11.4 / 15.2.  Of 6662 measured sizes it takes 1 % that are slower so and
// leaves 2 % that would be faster, by more than 5 %.  With planes in, hidden layers of one block's few columns: up to 384, in training 512.  Any B up to
// 768, k = 2-6, bit-sliced or looked up / rows: 64-150 columns 4.1 / 3.1 and 4.8 / 3.2, 320-384 4.1 / 3.75 and 4.8 / 3.9, 384-448 4.2 / 4.0, 448-512 4.1 / 4.2
// and 4.8 / 4.3, 600-1200 4.2 / 5.4 and 4.9 / 5.7.
bool dwn_rows_planes_pay(int B, int width, int nbits, int NO, bool training) {
    if (!width) return NO <= (training ? 512 : 384);
    const int blocks = dwn_rows_grid(B, width, NO, 0, true, training).blocks;
    return width * nbits <= 8192 && (double)blocks * width * nbits <= 1.5e6 && blocks <= 256;
}

template <int K>
static void dwn_rows_of(const DwnRows &a, hipStream_t s) {
    const DwnRowsGrid q = dwn_rows_grid(a.B, a.planes ? 0 : a.thr ? a.I / a.nbits : a.I, a.N * a.O, a.logits ? a.groups : 0,
                                        a.planes_out != nullptr, a.saved != nullptr);
    const int R = q.R, threads = q.threads, span = q.span;
    const size_t lds = a.planes || R == 1 ? 0 : (size_t)a.I;
    const dim3 grid(q.bx, q.by);
    if (a.planes && R == 8) DL_TIMED("dwn_rows", s, (dwn_rows<K, true, 8><<<grid, threads, 0, s>>>(a, span)));
    else if (a.planes) DL_TIMED("dwn_rows", s, (dwn_rows<K, true, 1><<<grid, threads, 0, s>>>(a, span)));
    else if (R == 8) DL_TIMED("dwn_rows", s, (dwn_rows<K, false, 8><<<grid, threads, lds, s>>>(a, span)));
    else DL_TIMED("dwn_rows", s, (dwn_rows<K, false, 1><<<grid, threads, 0, s>>>(a, span)));
}

void dwn_launch_rows(int k, const DwnRows &a, hipStream_t s) {
    switch (k) {
        case 1: dwn_rows_of<1>(a, s); break;
        case 2: dwn_rows_of<2>(a, s); break;
        case 3: dwn_rows_of<3>(a, s); break;
        case 4: dwn_rows_of<4>(a, s); break;
        case 5: dwn_rows_of<5>(a, s); break;
        default: dwn_rows_of<6>(a, s); break;
    }
}
