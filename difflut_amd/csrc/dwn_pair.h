// The input gradient of the first layer of a chain of DWN layers, taken together with its output gradient (dwn_pair.hip).
#pragma once
#include "dl_common.h"

#define DWN_PAIR_G 24      // nodes of the first layer per step
#define DWN_PAIR_I 128     // inputs at most
// what a step's connections are sorted into, by input: [I + 1] starts (padded), then G * k records: slot j in bits 0-2, the
// node's number in the step in bits 8-12, the byte offset of the slot's table row among the step's in bits 16-30
// [G] the second layer's connection (node << 3 | slot) that reads each of the step's nodes, -1 where there is not exactly one.
#define DWN_PAIR_STARTS 132
#define DWN_PAIR_STRIDE(k) (DWN_PAIR_STARTS + DWN_PAIR_G * ((k) + 1))
static inline int dwn_pair_groups(int N) { return dl_ceil_div(N, DWN_PAIR_G); }
static inline size_t dwn_pair_list_bytes(int N, int k) { return dl_align256((size_t)dwn_pair_groups(N) * DWN_PAIR_STRIDE(k) * sizeof(int)); }

// One step's connections by input, a block of 256 threads per step; inside an input they keep their order, so that a sum over
// the steps adds an input's terms in the order of the inverse mapping.
__device__ __forceinline__ void dwn_pair_list_block(const int *__restrict__ idx32, const int *__restrict__ inv_ptr1,
                                                    const int *__restrict__ inv_pos1, int *__restrict__ lists, int N, int K, int I,
                                                    int group) {
    __shared__ int in[DWN_PAIR_G * DL_MAX_FAST_K];
    const int first = group * DWN_PAIR_G;
    const int cnt = min(DWN_PAIR_G, N - first) * K;
    if ((int)threadIdx.x < cnt) in[threadIdx.x] = idx32[(size_t)first * K + threadIdx.x];
    __syncthreads();
    int *out = lists + (size_t)group * DWN_PAIR_STRIDE(K);
    if ((int)threadIdx.x < DWN_PAIR_G) {
        const int c = min(first + (int)threadIdx.x, N - 1), p0 = inv_ptr1[c];
        const int pos = inv_ptr1[c + 1] - p0 == 1 ? inv_pos1[p0] : -1;
        out[DWN_PAIR_STARTS + DWN_PAIR_G * K + threadIdx.x] = pos < 0 ? -1 : (pos / K << 3) | (pos % K);
    }
    if ((int)threadIdx.x <= I) {
        int before = 0;
        for (int q = 0; q < cnt; ++q) before += in[q] < (int)threadIdx.x ? 1 : 0;
        out[threadIdx.x] = before;
    }
    if ((int)threadIdx.x < cnt) {
        const int mine = in[threadIdx.x];
        int rank = 0;
        for (int q = 0; q < cnt; ++q) rank += (in[q] < mine || (in[q] == mine && q < (int)threadIdx.x)) ? 1 : 0;
        out[DWN_PAIR_STARTS + rank] = ((int)threadIdx.x << (16 + K + 1)) | ((int)threadIdx.x / K << 8) | ((int)threadIdx.x % K);
    } else if ((int)threadIdx.x < DWN_PAIR_G * K) {
        out[DWN_PAIR_STARTS + threadIdx.x] = 0;  // past the last node: a record all the same
    }
}

#define DWN_PAIR_T 4          // batch tiles per block
#define DWN_PAIR_ROUND 2048   // see dwn_pair_tiles
#define DWN_PAIR_LEAST 1100
int dwn_pair_tiles(int BT, int I, int N0, int k, int N1);
// gx [BT][I][64]: gy1, addr1, D1 (D form), inv_*: the second layer's; addr0, D0 (D form), lists: the first layer's
int dwn_pair_launch(const float *gy1, const uint8_t *addr1, const float *D1, const int *inv_ptr1, const int *inv_pos1, int N1,
                    const uint8_t *addr0, const float *D0, const int *lists, float *gx, int I, int N0, int k, int BT, hipStream_t s);
