// Input gradient of the first layer of a chain whose inputs are few and read many times (the patch columns of a
// convolution: 100 columns, 1152 nodes, 69 connections per column).
#include "dwn_pair.h"

// A block keeps four batch tiles - a lane four consecutive rows of one of them - and takes the first layer's nodes G at a time.
// Per step:
//   * the G nodes' output gradients are the second layer's input gradients, one term per connection: they are summed here
//     (dwn_bwd_gx_walk's sums) and put into the LDS, so the [B, N0] gradient is never stored;
//   * the nodes' addresses, times four, and their D-form rows (2^(k-1) floats per slot) go to the LDS as well;
//   * a wavefront owns `per` inputs, their sums in registers.  A connection costs a lane one read for its rows' addresses, one
//     for their gradients and a table value per row, all from the LDS.
// What a step needs from memory is asked for a step ahead.  An input's terms are added in the order of the inverse mapping:
// bit-equal to gathering from a stored output gradient.
// Bound by instruction issue and the LDS together: a connection of four rows per lane is 13 vector, 12 scalar and 6 LDS
// instructions of about 29 LDS clocks; four wavefronts per SIMD and 67 KB of LDS per block make two blocks per CU.  Gathering
// from the stored output gradient (dwn_bwd_gx_long) fetched 320 bytes per connection and tile from the L2, 17.5 clocks each,
// whatever the arithmetic (one lane read instead of two: 452 -> 431 us).  147456 rows, 100 columns, 1152 nodes of six inputs:
// 452 us and 262 for the second level's gather that stored the 680 MB -> 249 (of 2048 of the 2304 tiles) + 64 and 190; the layer's training
// step 961 -> 765.
typedef float dwn_f4 __attribute__((ext_vector_type(4)));
// Lane l's 16 bytes at base + voff land at LDS address lds + 16 l without passing through registers; waited for with vmcnt.
__device__ __forceinline__ void dwn_to_lds(unsigned lds, const char *base, unsigned voff) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(voff), "s"(base) : "memory", "m0");
}
__device__ __forceinline__ unsigned dwn_lds_offset(const void *p) {
    return (unsigned)(uintptr_t)(__attribute__((address_space(3))) const char *)(const char *)p;
}
template <typename T>
__device__ __forceinline__ __attribute__((address_space(3))) const T *dwn_lds(unsigned offset) {
    return (__attribute__((address_space(3))) const T *)offset;
}
// bits of a where mask is set, of b elsewhere; base + byte B of v: one instruction each
__device__ __forceinline__ unsigned dwn_bit_select(unsigned mask, unsigned a, unsigned b) {
    unsigned out;
    asm("v_bfi_b32 %0, %1, %2, %3" : "=v"(out) : "s"(mask), "v"(a), "v"(b));
    return out;
}
template <int B>
__device__ __forceinline__ unsigned dwn_add_byte(unsigned base, unsigned v) {
    unsigned out;
    asm("v_add_u32_sdwa %0, %1, %2 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:BYTE_%3" : "=v"(out) : "s"(base), "v"(v), "n"(B));
    return out;
}
template <int K, int WI>
__global__ __launch_bounds__(512, 4) void dwn_bwd_pair_gx(const float *__restrict__ gy1, const uint8_t *__restrict__ addr1,
                                                           const float *__restrict__ D1, const int *__restrict__ inv_ptr1,
                                                           const int *__restrict__ inv_pos1, int N1,
                                                           const uint8_t *__restrict__ addr0, const float *__restrict__ D0,
                                                           const int *__restrict__ lists, float *__restrict__ gx, int I, int N0,
                                                           int BT, int per) {
    constexpr int G = DWN_PAIR_G, Lh = 1 << (K - 1), W = 8, OWN = G / W;  // W wavefronts, OWN nodes of a step each
    constexpr int R = DWN_PAIR_T, TL = 64 / R;   // rows and tiles, lanes per tile
    constexpr int DB = G * K * Lh * 4;            // bytes of a step's table rows
    __shared__ __align__(16) float d_s[2][G * K * Lh];
    __shared__ __align__(16) float g_s[R][G][64];
    __shared__ __align__(16) uint32_t a_s[R][G][TL];
    const int lane = threadIdx.x & 63;
    const int wave = dl_uniform(threadIdx.x >> 6);
    const int t0 = blockIdx.x * R, sub = lane / TL, row0 = R * (lane % TL);  // my tile of the block's and my first row in it
    const int tile = min(t0 + sub, BT - 1);                                 // (tiles past the last repeat it and are not stored)
    const int wbeg = wave * per;
    const int mine = max(0, min(per, I - wbeg));  // my inputs: wbeg .. wbeg + mine - 1
    float acc[WI][R];
#pragma unroll
    for (int r = 0; r < WI; ++r)
#pragma unroll
        for (int u = 0; u < R; ++u) acc[r][u] = 0.0f;
    const int groups = (N0 + G - 1) / G;
    const unsigned d_lds = dwn_lds_offset(&d_s[0][0]);
    // my rows of tile `tile` in the arrays [B/64][nodes][64]
    const uint8_t *a0_t = addr0 + (size_t)tile * N0 * 64 + row0, *a1_t = addr1 + (size_t)tile * N1 * 64 + row0;
    const float *g1_t = gy1 + (size_t)tile * N1 * 64 + row0;
    // a step's table rows, into buffer `buf`
    auto fetch_tables = [&](int grp, int buf) {
        const unsigned bytes = (unsigned)min(G, N0 - grp * G) * (K * Lh * 4);
        const char *src = reinterpret_cast<const char *>(D0 + (size_t)grp * G * K * Lh);
#pragma unroll
        for (int p = 0; p < (DB + 8191) / 8192; ++p) {
            const unsigned chunk = (p * W + wave) * 1024u, off = chunk + lane * 16u;
            if (off < bytes) dwn_to_lds(d_lds + buf * DB + chunk, src, off);
        }
    };
    // my nodes of a step: their addresses, and what their output gradients are made of
    uint32_t a0[OWN], a1[OWN];
    dwn_f4 g1[OWN];
    float coef[OWN];
    auto fetch_nodes = [&](int grp, int rec) {
        const int c0 = grp * G, cnt = min(G, N0 - c0);
#pragma unroll
        for (int q = 0; q < OWN; ++q) {
            const int c = min(wave + q * W, cnt - 1);
            const int r = max(__builtin_amdgcn_readlane(rec, c), 0);
            a0[q] = *reinterpret_cast<const uint32_t *>(a0_t + (size_t)(c0 + c) * 64);
            a1[q] = *reinterpret_cast<const uint32_t *>(a1_t + (size_t)(r >> 3) * 64);
            g1[q] = *reinterpret_cast<const dwn_f4 *>(g1_t + (size_t)(r >> 3) * 64);
            coef[q] = D1[((size_t)(r >> 3) * K + (r & 7)) * Lh + (lane & (Lh - 1))];
        }
    };
    // what the lists say of a step, asked for ahead: the second layer's connections, where mine start by input, the first 64
    auto list_of = [&](int grp) { return lists + (size_t)min(grp, groups - 1) * DWN_PAIR_STRIDE(K); };
    auto recs_of = [&](int grp) { return list_of(grp)[DWN_PAIR_STARTS + G * K + min(lane, G - 1)]; };
    auto starts_of = [&](int grp) { return list_of(grp)[min(wbeg + min(lane, per), I)]; };
    int rec1 = recs_of(0);
    int my_start = starts_of(0);
    int my_rec = list_of(0)[DWN_PAIR_STARTS + min(__builtin_amdgcn_readlane(my_start, 0) + lane, G * K - 1)];
    fetch_tables(0, 0);
    fetch_nodes(0, rec1);
    int next_rec1 = recs_of(1);
    for (int grp = 0; grp < groups; ++grp) {
        const int c0 = grp * G, cnt = min(G, N0 - c0);
        const int s_begin = __builtin_amdgcn_readlane(my_start, 0), s_end = __builtin_amdgcn_readlane(my_start, per);
#pragma unroll
        for (int q = 0; q < OWN; ++q) {
            const int c = min(wave + q * W, cnt - 1);
            const int r = __builtin_amdgcn_readlane(rec1, c);
            const unsigned aw = a1[q];
            reinterpret_cast<uint32_t *>(&a_s[0][0][0])[(sub * G + c) * TL + lane % TL] = a0[q] << 2;
            dwn_f4 sum;
            if (r >= 0) {
                const unsigned low = (1u << (r & 7)) - 1u;
#pragma unroll
                for (int u = 0; u < R; ++u) {
                    const unsigned a = (aw >> (8 * u)) & 0xffu;
                    sum[u] = 0.0f + g1[q][u] * dl_lane_read(coef[q], (int)((a & low) | ((a >> 1) & ~low)));
                }
            } else {  // a node that is read by no connection of the second layer, or by several
#pragma unroll
                for (int u = 0; u < R; ++u) sum[u] = 0.0f;
                const int e0 = dl_uniform(inv_ptr1[c0 + c]), e1 = dl_uniform(inv_ptr1[c0 + c + 1]);
                for (int e = e0; e < e1; ++e) {
                    const int p = dl_uniform(inv_pos1[e]), n = p / K, j = p - n * K;
                    const float cf = D1[((size_t)n * K + j) * Lh + (lane & (Lh - 1))];
                    const dwn_f4 g = *reinterpret_cast<const dwn_f4 *>(g1_t + (size_t)n * 64);
                    const unsigned w = *reinterpret_cast<const uint32_t *>(a1_t + (size_t)n * 64), low = (1u << j) - 1u;
#pragma unroll
                    for (int u = 0; u < R; ++u) {
                        const unsigned a = (w >> (8 * u)) & 0xffu;
                        sum[u] += g[u] * dl_lane_read(cf, (int)((a & low) | ((a >> 1) & ~low)));
                    }
                }
            }
            *reinterpret_cast<dwn_f4 *>(&g_s[sub][c][row0]) = sum;
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the step's table rows have landed
        __syncthreads();
        if (grp + 1 < groups) {
            fetch_tables(grp + 1, (grp + 1) & 1);
            fetch_nodes(grp + 1, next_rec1);
        }
        rec1 = next_rec1;
        next_rec1 = recs_of(grp + 2);
        const int next_start = starts_of(grp + 1);
        // my connections one after the other, by input, the next one's address word under way
        const unsigned a_l = dwn_lds_offset(&a_s[0][0][0]) + sub * (G * 64) + row0, g_l = dwn_lds_offset(&g_s[0][0][0]) + sub * (G * 256) + row0 * 4;
        const unsigned d_l = d_lds + (grp & 1) * DB;
        for (int base = s_begin; base < s_end; base += 64) {
            // (every lane holds a record of the step; readlane takes the lane number modulo 64)
            const int rec = base == s_begin ? my_rec : list_of(grp)[DWN_PAIR_STARTS + min(base + lane, G * K - 1)];
            int q = __builtin_amdgcn_readlane(rec, 0), e = 0;
            unsigned w = *dwn_lds<uint32_t>(a_l + ((q & 0x1f00) >> 2));
#pragma unroll
            for (int r = 0; r < WI; ++r) {
                // (starts past my inputs repeat the last one: nothing to do there)
                const int hi = min(__builtin_amdgcn_readlane(my_start, r + 1) - base, 64);
                for (; e < hi; ++e) {
                    const int ahead = __builtin_amdgcn_readlane(rec, e + 1);
                    const unsigned w_ahead = *dwn_lds<uint32_t>(a_l + ((ahead & 0x1f00) >> 2));
                    const dwn_f4 g = *dwn_lds<dwn_f4>(g_l + (q & 0x1f00));
                    const unsigned ap = dwn_bit_select((0x04040404u << (q & 31)) - 0x01010101u, w, w >> 1);
                    const unsigned drow = d_l + ((unsigned)q >> 16);
                    float d[R];
                    d[0] = *dwn_lds<float>(dwn_add_byte<0>(drow, ap));
                    d[1] = *dwn_lds<float>(dwn_add_byte<1>(drow, ap));
                    d[2] = *dwn_lds<float>(dwn_add_byte<2>(drow, ap));
                    d[3] = *dwn_lds<float>(dwn_add_byte<3>(drow, ap));
#pragma unroll
                    for (int u = 0; u < R; ++u) acc[r][u] += g[u] * d[u];
                    q = ahead;
                    w = w_ahead;
                }
            }
        }
        my_start = next_start;
        my_rec = list_of(grp + 1)[DWN_PAIR_STARTS + min(__builtin_amdgcn_readlane(my_start, 0) + lane, G * K - 1)];
        __syncthreads();
    }
    if (t0 + sub < BT) {
#pragma unroll
        for (int r = 0; r < WI; ++r)
            if (r < mine) {
                dwn_f4 v;
#pragma unroll
                for (int u = 0; u < R; ++u) v[u] = acc[r][u];
                __builtin_nontemporal_store(v, reinterpret_cast<dwn_f4 *>(&gx[((size_t)tile * I + wbeg + r) * 64 + row0]));
            }
    }
}

template <int K>
static void dwn_pair_launch_k(const float *gy1, const uint8_t *addr1, const float *D1, const int *inv_ptr1, const int *inv_pos1,
                              int N1, const uint8_t *addr0, const float *D0, const int *lists, float *gx, int I, int N0, int BT,
                              hipStream_t s) {
    const int per = dl_ceil_div(I, 8), blocks = dl_ceil_div(BT, DWN_PAIR_T);
#define DWN_PAIR(WI_)                                                                                                  \
    DL_TIMED("dwn_bwd_pair_gx", s, (dwn_bwd_pair_gx<K, WI_><<<blocks, 512, 0, s>>>(gy1, addr1, D1, inv_ptr1, inv_pos1, N1, addr0, \
                                                                                    D0, lists, gx, I, N0, BT, per)))
    // registers for the sums of a wavefront's inputs: up to 40 inputs, up to 104 (5 x 5 patches of four channels), 128
    if (per <= 5) DWN_PAIR(5);
    else if (per <= 13) DWN_PAIR(13);
    else DWN_PAIR(16);
#undef DWN_PAIR
}

// The tiles it takes of BT (the first ones; 0 = none): all blocks of a round of DWN_PAIR_ROUND tiles - two blocks per CU - run
// at once and take 249 us together, 199 where there are only half as many of them, so a last round that is too empty is left
// to the gather from a stored output gradient, which goes by the tile.  Kernels of this path with setup against that one's,
// us, 100 columns, 1152 nodes: 769 tiles 280 / 269, 1026 344 / 350, 1530 387 / 501, 2052 (of which 4 in a second round) 445 / 654.
// The whole training step with this path and without, us, by inputs x nodes of the first level (k = 6; 512: k = 4), at about
// 1110, 1300, 2040 and 2300 tiles: 16 x 576 322 / 334, 326 / 368, 389 / 494, 479 / 534; 16 x 512 289 / 291, 298 / 318, 357 / 435,
// 421 / 461; 36 x 576 326 / 320, 335 / 353, 430 / 497, 458 / 538; 75 x 576 347 / 340, 354 / 371, 435 / 534, 487 / 572; 100 x 1152
// 535 / 544, 557 / 602, 675 / 849, 780 / 946; 128 x 1152 561 / 567, 588 / 625, 696 / 871, 799 / 964: at the least it loses 2 % at
// worst, from 1300 on it wins everywhere.
// Fewer than 16 inputs leave wavefronts without one; lists shorter than 32 take the gather that fills the table gradient in
// front, which reads a node's rows seldom enough.
int dwn_pair_tiles(int BT, int I, int N0, int k, int N1) {
    if (I < 16 || I > DWN_PAIR_I || (long long)N1 * k != N0 || (long long)N0 * k < 32LL * I) return 0;
    const int full = BT / DWN_PAIR_ROUND * DWN_PAIR_ROUND;
    return BT - full >= DWN_PAIR_LEAST ? BT : full;
}

int dwn_pair_launch(const float *gy1, const uint8_t *addr1, const float *D1, const int *inv_ptr1, const int *inv_pos1, int N1,
                    const uint8_t *addr0, const float *D0, const int *lists, float *gx, int I, int N0, int k, int BT, hipStream_t s) {
    switch (k) {
#define DWN_PAIR_K(K_) \
    case K_: dwn_pair_launch_k<K_>(gy1, addr1, D1, inv_ptr1, inv_pos1, N1, addr0, D0, lists, gx, I, N0, BT, s); break
        DWN_PAIR_K(1);
        DWN_PAIR_K(2);
        DWN_PAIR_K(3);
        DWN_PAIR_K(4);
        DWN_PAIR_K(5);
        default: dwn_pair_launch_k<6>(gy1, addr1, D1, inv_ptr1, inv_pos1, N1, addr0, D0, lists, gx, I, N0, BT, s); break;
#undef DWN_PAIR_K
    }
    return dl_launch_status();
}
