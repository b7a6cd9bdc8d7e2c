// Patch extraction of the convolutional LUT layer and its adjoint.
//   rows    r = (image b, output position oy, ox), row-major: r = (b * OH + oy) * OW + ox
//   columns c = (channel ch, dy, dx):                          c = (ch * KH + dy) * KW + dx
//   patches[r][c] = x[b, ch, oy*SH + dy - PH, ox*SW + dx - PW], 0 outside the image
// Neighbouring rows are neighbouring output positions, so with lane = row the loads of one column
// are (stride SW) contiguous in x and a 64-row tile of a column is 256 contiguous bytes tile-major.
#include "dl_common.h"

struct ConvGeom {
    int B, C, H, W, KH, KW, SH, SW, PH, PW, OH, OW;
};

#define CONV_MAX_COLS 4096  // columns whose offsets fit the per-block table

// per-column offset inside an image (ch*H*W + dy*W + dx) and (dy, dx) packed, built once per block
__device__ __forceinline__ void conv_fill_columns(const ConvGeom &g, int cols, int *off, int *dydx) {
    for (int c = threadIdx.x; c < cols; c += blockDim.x) {
        const int dx = c % g.KW, dy = (c / g.KW) % g.KH, ch = c / (g.KW * g.KH);
        off[c] = (ch * g.H + dy) * g.W + dx;
        dydx[c] = (dy << 16) | dx;
    }
}

// grid = ceil(rows / 64) blocks of 256 threads; block t writes rows 64 t .. 64 t + 63 (all columns), coalesced.
// flip (nullable, [rows][cols] bytes): bit-flip augmentation of the patch matrix, v -> v + (1 - 2 v) where set
// (base_layer.py:149-264 applied to the patches, convolutional.py:205-207).
__global__ __launch_bounds__(256) void conv_unfold_rows(const float *__restrict__ x, float *__restrict__ patches, ConvGeom g,
                                                         long long rows, int cols, const uint8_t *__restrict__ flip) {
    __shared__ int off[CONV_MAX_COLS], dydx[CONV_MAX_COLS];
    __shared__ long long base[64];
    __shared__ int y0s[64], x0s[64];
    conv_fill_columns(g, cols, off, dydx);
    if (threadIdx.x < 64) {
        const long long r = (long long)blockIdx.x * 64 + threadIdx.x;
        const long long rr = r < rows ? r : rows - 1;
        const int ox = (int)(rr % g.OW), oy = (int)((rr / g.OW) % g.OH);
        const long long b = rr / ((long long)g.OW * g.OH);
        const int y0 = oy * g.SH - g.PH, x0 = ox * g.SW - g.PW;
        y0s[threadIdx.x] = y0;
        x0s[threadIdx.x] = x0;
        base[threadIdx.x] = (b * g.C * g.H + y0) * (long long)g.W + x0;
    }
    __syncthreads();
    const long long r0 = (long long)blockIdx.x * 64;
    const int live = (int)min((long long)64, rows - r0);
    float *out = patches + r0 * cols;
    for (int e = threadIdx.x; e < live * cols; e += 256) {
        const int r = e / cols, c = e - r * cols;
        const int y = y0s[r] + (dydx[c] >> 16), xx = x0s[r] + (dydx[c] & 0xffff);
        const bool in = y >= 0 && y < g.H && xx >= 0 && xx < g.W;
        float v = in ? x[base[r] + off[c]] : 0.0f;
        if (flip && flip[r0 * cols + e]) v = v + (1.0f - 2.0f * v);
        out[e] = v;
    }
}

// The same patches as the bit-planes a DWN layer reads: word (t, c) holds in bit r (patches[64 t + r][c] >= 0.5).
// grid = ceil(rows / 64) blocks of 256 threads; lane = row, the four wavefronts share the columns.
__global__ __launch_bounds__(256) void conv_unfold_planes(const float *__restrict__ x, unsigned long long *__restrict__ planes,
                                                           ConvGeom g, long long rows, int cols,
                                                           const uint8_t *__restrict__ flip) {
    __shared__ int off[CONV_MAX_COLS], dydx[CONV_MAX_COLS];
    conv_fill_columns(g, cols, off, dydx);
    __syncthreads();
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const long long r = (long long)blockIdx.x * 64 + lane;
    const bool live = r < rows;
    const long long rr = live ? r : rows - 1;
    const int ox = (int)(rr % g.OW), oy = (int)((rr / g.OW) % g.OH);
    const long long b = rr / ((long long)g.OW * g.OH);
    const int y0 = oy * g.SH - g.PH, x0 = ox * g.SW - g.PW;
    const float *img = x + (b * g.C * g.H + y0) * (long long)g.W + x0;
    unsigned long long *out = planes + (size_t)blockIdx.x * cols;
    const int per = (cols + 3) / 4;
    const int c0 = w * per, c1 = min(cols, c0 + per);
    for (int cb = c0; cb < c1; cb += 64) {  // a lane keeps word cb + lane; 64 consecutive words leave together
        unsigned long long mine = 0;
        const int cnt = min(64, c1 - cb);
        for (int q = 0; q < cnt; ++q) {
            const int c = cb + q;
            const int y = y0 + (dydx[c] >> 16), xx = x0 + (dydx[c] & 0xffff);
            const bool in = live && y >= 0 && y < g.H && xx >= 0 && xx < g.W;
            float v = in ? img[off[c]] : 0.0f;
            if (flip && live && flip[r * cols + c]) v = v + (1.0f - 2.0f * v);  // the value the reference thresholds
            const unsigned long long mask = __ballot(live && v >= 0.5f);
            if (q == lane) mine = mask;
        }
        if (lane < cnt) out[cb + lane] = mine;
    }
}

// The same words at stride 1 without a mask, from the thresholded image as bits: a wavefront's ballot over 64 consecutive values of
// an image is a word of them in the LDS, a row of the image any W bits in a row.  The rows of a tile are pieces of lines of output
// positions (b, oy), and a column's bits over a piece are OW bits of image row oy + dy - PH from position dx - PW on: a shift
// per line in the place of a load, a comparison and a vote per position.  A block has `tiles` tiles and the images they are from.
// 256 images of 4 x 28 x 28, 5 x 5 patches (147456 x 100): 30 -> 12 us.
#define CONV_BIT_WORDS 4096  // of LDS
#define CONV_BIT_WAVES 16    // a trip to memory per block, not four: 20 us with four wavefronts
__global__ __launch_bounds__(64 * CONV_BIT_WAVES) void conv_unfold_bits(const float *__restrict__ x, unsigned long long *__restrict__ planes,
                                                         ConvGeom g, long long rows, int cols, int tiles, int words) {
    extern __shared__ unsigned long long bits[];  // [image][word]
    const int P = g.OH * g.OW, values = g.C * g.H * g.W, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const long long r0 = (long long)blockIdx.x * tiles * 64, r1 = min(rows, r0 + (long long)tiles * 64);
    const long long b0 = r0 / P;
    const int images = (int)((r1 - 1) / P - b0) + 1;
    const int all = images * words;
    for (int w0 = wave; w0 < all; w0 += CONV_BIT_WAVES * 8) {  // eight loads in flight
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int w = min(w0 + CONV_BIT_WAVES * u, all - 1), img = w / words, e = (w - img * words) * 64 + lane;
            v[u] = e < values ? x[(b0 + img) * values + e] : 0.0f;
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const unsigned long long mask = __ballot(v[u] >= 0.5f);
            if (lane == 0 && w0 + CONV_BIT_WAVES * u < all) bits[w0 + CONV_BIT_WAVES * u] = mask;
        }
    }
    __syncthreads();
    const unsigned long long line_mask = g.OW == 64 ? ~0ull : (1ull << g.OW) - 1ull;
    const unsigned long long row_mask = g.W == 64 ? ~0ull : (1ull << g.W) - 1ull;
    const int total = (int)(r1 - r0), off = (int)(r0 - b0 * P);
    for (int e = threadIdx.x; e < (total + 63) / 64 * cols; e += 64 * CONV_BIT_WAVES) {
        const int t = e / cols, c = e - t * cols, patch = c / g.KW, dx = c - patch * g.KW, ch = patch / g.KH, dy = patch - ch * g.KH;
        const int end = min(64, total - 64 * t);
        int line = (off + 64 * t) / g.OW, at = line * g.OW - off - 64 * t;  // its first position, from the tile's first row
        int img = line / g.OH, oy = line - img * g.OH;
        unsigned long long word = 0;
        for (; at < end; at += g.OW) {
            const int y = oy + dy - g.PH;
            if (y >= 0 && y < g.H) {
                const int first = (ch * g.H + y) * g.W, sh = first & 63;
                const unsigned long long *from = bits + img * words + (first >> 6);
                unsigned long long piece = from[0] >> sh;
                if (sh + g.W > 64) piece |= from[1] << (64 - sh);  // (sh > 0 here)
                piece = (((piece & row_mask) << g.PW) >> dx) & line_mask;
                word |= at >= 0 ? piece << at : piece >> -at;
            }
            if (++oy == g.OH) { oy = 0; ++img; }
        }
        planes[((size_t)(r0 >> 6) + t) * cols + c] = word;  // (past the last row there are no lines)
    }
}
// Whether the words come sooner that way.  A block stages its images, 2.4 us per 128 words, before it makes a word, and then takes a turn of
// 1024 words line by line; the votes take 0.19 us a word of a wavefront and nothing in front.  So few words, patches of one or two
// columns and many channels on many blocks are better voted on, and few rows of many columns, where the votes have few wavefronts, are not.
// The terms are fitted to 2269 sizes (1-64 channels, 5-60 pixels, fields of 1-7, 1-256 images, both kernels; 11 and 9 % rms): 2 % of them are slower by bits
// by more than 5 % where the rule takes them (1.24 times at most), 3 % would be faster where it does not, and on the average it is 1 % above the better one.
// us, votes / bits: 256 images of 4 x 28 x 28, field 5 30 / 12, field 1 7.7 / 9.7; 16 images of 3 x 16 x 16, field 3 5.2 / 6.9; 16 of 64 x 28 x 28, field
// 2 18 / 41, field 5 90 / 65; 64 of 64 x 7 x 7, field 4 55 / 79; one of 32 x 8 x 8, field 7 81 / 7.6; 5 of 64 x 8 x 8, field 5 83 / 21.
static inline bool conv_bits_pay(const ConvGeom &g, long long rows, int cols, int words, int tiles) {
    const int P = g.OH * g.OW, BT = dl_ceil_div(rows, 64), held = tiles < BT ? tiles : BT, span = 64 * held;
    const int images = (span - 1) / P + 1 + (P % span != 0 && span % P != 0), blocks = dl_ceil_div(rows, 64LL * tiles);
    const double rounds = blocks > 512 ? blocks / 512.0 : 1.0, trips = dl_ceil_div((long long)(images < g.B ? images : g.B) * words, 128);
    const double turns = dl_ceil_div((long long)held * cols, 64 * CONV_BIT_WAVES), lines = turns * (64.0 / g.OW + (64 % g.OW != 0));
    const double bits = 2.0 + rounds * (2.44 * trips + 1.7 * turns + 0.068 * lines) + blocks * (0.0042 * trips + 0.00048 * lines);
    const double votes = 3.35 + cols * (0.048 + 0.000038 * BT + 0.000062 * (BT > 2048 ? BT - 2048 : 0)) + 0.00077 * BT;
    return bits < 0.95 * votes;
}
// tiles per block, 0: not by bits
static int conv_bit_tiles(const ConvGeom &g, long long rows, int cols, int words) {
    if (g.SH != 1 || g.SW != 1 || g.W + 2 * g.PW > 64) return 0;
    for (int tiles = 8; tiles > 0; tiles /= 2)
        if (((long long)tiles * 64 / ((long long)g.OH * g.OW) + 2) * words <= CONV_BIT_WORDS)
            return conv_bits_pay(g, rows, cols, words, tiles) ? tiles : 0;
    return 0;
}

// Adjoint: gx[b,ch,y,xx] = sum over (dy,dx) of gpatches[(b,oy,ox)][(ch,dy,dx)] with oy*SH + dy - PH = y,
// ox*SW + dx - PW = xx.  One thread per pixel, terms added in (dy, dx) order.  gpatches row-major
// [rows][cols] or (tiled) tile-major [rows/64][cols][64].
__global__ __launch_bounds__(256) void conv_fold(const float *__restrict__ gp, float *__restrict__ gx, ConvGeom g, int cols,
                                                  int tiled) {
    const long long total = (long long)g.B * g.C * g.H * g.W;
    const long long e = (long long)blockIdx.x * 256 + threadIdx.x;
    if (e >= total) return;
    const int xx = (int)(e % g.W), y = (int)((e / g.W) % g.H);
    const int ch = (int)((e / ((long long)g.W * g.H)) % g.C);
    const long long b = e / ((long long)g.W * g.H * g.C);
    float acc = 0.0f;
    for (int dy = 0; dy < g.KH; ++dy) {
        const int ny = y + g.PH - dy;
        if (ny < 0 || ny % g.SH) continue;
        const int oy = ny / g.SH;
        if (oy >= g.OH) continue;
        for (int dx = 0; dx < g.KW; ++dx) {
            const int nx = xx + g.PW - dx;
            if (nx < 0 || nx % g.SW) continue;
            const int ox = nx / g.SW;
            if (ox >= g.OW) continue;
            const long long r = (b * g.OH + oy) * g.OW + ox;
            const int c = (ch * g.KH + dy) * g.KW + dx;
            acc += tiled ? gp[((r >> 6) * cols + c) * 64 + (r & 63)] : gp[r * cols + c];
        }
    }
    gx[e] = acc;
}

// The tile-major form at stride 1, patches KW wide: the positions of a line lie together, so the KW values of a line are asked for at
// once; 32-bit arithmetic.  Bound by the reads of the gradient, each value once.  256 images of 4 x 28 x 28, fields of 1 to 7, us, a thread
// that walks the patch / so: 7.2 / 5.2, 11 / 6.1, 18 / 8.0, 25 / 10, 34 / 13, 44 / 17, 56 / 20; wider ones, whose values would take more
// registers than a thread that is alone with them should, keep the walk.
template <int KW>
__global__ __launch_bounds__(256) void conv_fold_lines(const float *__restrict__ gp, float *__restrict__ gx, ConvGeom g, int cols) {
    const int e = blockIdx.x * 256 + threadIdx.x;
    if (e >= g.B * g.C * g.H * g.W) return;
    const int line = e / g.W, xx = e - line * g.W, plane = line / g.H, y = line - plane * g.H, b = plane / g.C, ch = plane - b * g.C;
    float acc = 0.0f;
    for (int dy = 0; dy < g.KH; ++dy) {
        const int oy = y + g.PH - dy;
        if (oy < 0 || oy >= g.OH) continue;
        const int r0 = (b * g.OH + oy) * g.OW, c0 = (ch * g.KH + dy) * KW;
        float v[KW];
#pragma unroll
        for (int dx = 0; dx < KW; ++dx) {
            const int ox = xx + g.PW - dx, r = r0 + ox;
            v[dx] = ox >= 0 && ox < g.OW ? gp[((size_t)(r >> 6) * cols + c0 + dx) * 64 + (r & 63)] : 0.0f;
        }
#pragma unroll
        for (int dx = 0; dx < KW; ++dx) acc += v[dx];
    }
    gx[e] = acc;
}

static int conv_geom(ConvGeom &g, int B, int C, int H, int W, int KH, int KW, int SH, int SW, int PH, int PW) {
    if (B <= 0 || C <= 0 || H <= 0 || W <= 0 || KH <= 0 || KW <= 0 || SH <= 0 || SW <= 0 || PH < 0 || PW < 0)
        return DL_ERR_SHAPE;
    if (H + 2 * PH < KH || W + 2 * PW < KW) return DL_ERR_SHAPE;
    if (KH > 0xffff || KW > 0xffff || (long long)C * KH * KW > CONV_MAX_COLS) return DL_ERR_UNSUPPORTED;
    if ((long long)C * H * W > 0x7fffffffLL) return DL_ERR_UNSUPPORTED;
    g = {B, C, H, W, KH, KW, SH, SW, PH, PW, (H + 2 * PH - KH) / SH + 1, (W + 2 * PW - KW) / SW + 1};
    if ((long long)B * g.OH * g.OW > 0x7fffffffLL * 64) return DL_ERR_UNSUPPORTED;
    return DL_OK;
}

extern "C" long long dl_unfold_rows(int B, int H, int W, int KH, int KW, int SH, int SW, int PH, int PW) {
    ConvGeom g;
    if (conv_geom(g, B, 1, H, W, KH, KW, SH, SW, PH, PW)) return 0;
    return (long long)B * g.OH * g.OW;
}

extern "C" int dl_unfold_flip(const float *x, const uint8_t *flip, float *patches, void *planes, int B, int C, int H, int W,
                              int KH, int KW, int SH, int SW, int PH, int PW, void *stream);
extern "C" int dl_unfold(const float *x, float *patches, void *planes, int B, int C, int H, int W, int KH, int KW, int SH,
                         int SW, int PH, int PW, void *stream) {
    return dl_unfold_flip(x, nullptr, patches, planes, B, C, H, W, KH, KW, SH, SW, PH, PW, stream);
}

extern "C" int dl_unfold_flip(const float *x, const uint8_t *flip, float *patches, void *planes, int B, int C, int H, int W,
                              int KH, int KW, int SH, int SW, int PH, int PW, void *stream) {
    if (!x || (!patches && !planes)) return DL_ERR_NULL;
    ConvGeom g;
    int rc = conv_geom(g, B, C, H, W, KH, KW, SH, SW, PH, PW);
    if (rc) return rc;
    hipStream_t s = (hipStream_t)stream;
    const long long rows = (long long)B * g.OH * g.OW;
    const int cols = C * KH * KW, grid = dl_ceil_div(rows, 64);
    if (patches) DL_TIMED("conv_unfold_rows", s, (conv_unfold_rows<<<grid, 256, 0, s>>>(x, patches, g, rows, cols, flip)));
    const int words = dl_ceil_div((long long)C * H * W, 64), tiles = planes && !flip ? conv_bit_tiles(g, rows, cols, words) : 0;
    if (tiles) {
        const size_t lds = ((size_t)tiles * 64 / ((size_t)g.OH * g.OW) + 2) * words * sizeof(unsigned long long);
        DL_TIMED("conv_unfold_bits", s, (conv_unfold_bits<<<dl_ceil_div(rows, 64LL * tiles), 64 * CONV_BIT_WAVES, lds, s>>>(
                                              x, (unsigned long long *)planes, g, rows, cols, tiles, words)));
    } else if (planes)
        DL_TIMED("conv_unfold_planes", s,
                 (conv_unfold_planes<<<grid, 256, 0, s>>>(x, (unsigned long long *)planes, g, rows, cols, flip)));
    return dl_launch_status();
}

extern "C" int dl_fold(const float *gpatches, int tiled, float *gx, int B, int C, int H, int W, int KH, int KW, int SH,
                       int SW, int PH, int PW, void *stream) {
    if (!gpatches || !gx) return DL_ERR_NULL;
    ConvGeom g;
    int rc = conv_geom(g, B, C, H, W, KH, KW, SH, SW, PH, PW);
    if (rc) return rc;
    hipStream_t s = (hipStream_t)stream;
    const long long total = (long long)B * C * H * W;
    if (tiled && SH == 1 && SW == 1 && total <= 0x7fffffffLL - 256 && (long long)B * g.OH * g.OW <= 0x7fffffffLL && KW <= 7) {
#define CONV_FOLD(KW_) \
    case KW_: DL_TIMED("conv_fold", s, (conv_fold_lines<KW_><<<dl_ceil_div(total, 256), 256, 0, s>>>(gpatches, gx, g, C * KH * KW_))); break
        switch (KW) {
            CONV_FOLD(1);
            CONV_FOLD(2);
            CONV_FOLD(3);
            CONV_FOLD(4);
            CONV_FOLD(5);
            CONV_FOLD(6);
            CONV_FOLD(7);
        }
#undef CONV_FOLD
        return dl_launch_status();
    }
    DL_TIMED("conv_fold", s, (conv_fold<<<dl_ceil_div(total, 256), 256, 0, s>>>(gpatches, gx, g, C * KH * KW, tiled)));
    return dl_launch_status();
}
