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

template <int K>
static void dwn_rows_of(const DwnRows &a, hipStream_t s) {
    const int NO = a.N * a.O, width = a.thr ? a.I / a.nbits : a.I;
    const int R = a.logits && !a.saved && a.B < 8 ? 1 : 8, by = a.planes_out || a.saved ? (a.B + 63) / 64 * 8 : dl_ceil_div(a.B, R);
    // a thread per column, more where the input has more values to turn than that; blocks of 1024 share the columns as far as two
    // blocks per CU (of one group each: the groups)
    const int columns = a.logits ? a.gsize : NO;
    int threads = a.planes || R == 1 || columns > width ? columns : width;
    if (a.logits && threads > 512 && (long long)a.groups * by > 256) threads = columns > 512 ? columns : 512;
    threads = threads >= 1024 ? 1024 : (threads + 63) / 64 * 64;
    int bx = a.groups, span = a.gsize;
    if (!a.logits) {
        bx = dl_ceil_div(NO, threads);
        if (bx > 1 && (long long)bx * by > 512) bx = by >= 512 ? 1 : dl_ceil_div(512, by) < bx ? dl_ceil_div(512, by) : bx;
        span = dl_ceil_div(dl_ceil_div(NO, bx), threads) * threads;
        bx = dl_ceil_div(NO, span);
    }
    const size_t lds = a.planes || R == 1 ? 0 : (size_t)a.I;
    const dim3 grid(bx, by);
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
