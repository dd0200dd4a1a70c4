// Learned wave surrogate: BF16 MFMA kernels for gfx950 (MI355X) and the
// encoder-decoder that uses them, forward, backward and Adam, all on the
// device.  No counterpart in the reference: the surrogate stands in for the
// wave action solve (wavestep, Wavestep.cu:755-1167) between full-solver
// checkpoints and predicts the wave-group-averaged fields the flow and
// sediment steps read from it (H, wave and roller dissipation, Fx, Fy).
//
// Tensors are NHWC.  Activations and their gradients are BF16, weights are
// kept as FP32 masters (Adam) with BF16 copies for the matrix cores, and
// every product accumulates in FP32 (v_mfma_f32_16x16x32_bf16).
//
// Convolutions are implicit GEMMs (pixels x output channels, K = taps x
// input channels):
//   k_conv        forward (also the data gradient, through the flipped and
//                 transposed weights: dX = conv(dZ, W')), with pooling,
//                 activation masks and the output head in its epilogue
//   k_conv_wgrad  weight gradient (output x input channels, K = pixels),
//                 split over pixel ranges into FP32 partials that
//                 k_reduce_parts sums in a fixed order
// A 16 x 16 x 32 MFMA takes from each lane 8 consecutive K values of one A
// row (lane % 16) and of one B column (lane % 16), the lanes' K slices
// being lane / 16; it leaves in each lane four rows 4*(lane/16)+r of column
// lane % 16 of the 16 x 16 result.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

#include "../../include/xbg.h"

namespace {

typedef __bf16 bf16;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4 mfma16(bf16x8 a, bf16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ bf16 to_bf16(float x) { return (bf16)x; }

constexpr int KB = 32;        // input channels per K block
constexpr int LROW = KB + 8;  // LDS row (pixel) stride in bf16: 80 B, keeps 16-B reads aligned and spread

// ---------------------------------------------------------------------------
// Convolution, 'same' padding (TAPS 9: 3x3, TAPS 1: 1x1), forward and data
// gradient, with the elementwise passes around it folded into its staging
// and its epilogue.
//
// Workgroup: 4 waves, TW pixels along x times 64 MB / TW rows (64 MB pixels)
// and BN output channels; wave w computes MB blocks of 16 pixels (pixels
// 64 m + 16 w + 0..15 of the tile, m < MB) x BN channels.  Per block of 32
// input channels the input tile (+1-pixel halo for 3x3) and the block's
// weights are staged in LDS; the next block's values are in flight from
// memory, in registers, while this one is multiplied.  The weights are the
// MFMA's A operand, so a lane holds four consecutive output channels of one
// pixel.  With 64-pixel rows a pixel fragment serves the three taps of its
// column that read it from three output rows: 54 LDS reads per 144 MFMAs
// instead of 72, under the LDS rate that a read per operand would reach.
// The sum over channel blocks and taps runs in the same order for any tile.
//
// Source (CSrc): a plain tensor; a decoder's concatenation read from its two
// parts (the coarse tensor at half resolution, the skip); or the network's
// 8 input channels, the other 24 being zero.  Epilogue (EPI): the tile goes
// through LDS as BF16, so that its values leave as 16-byte stores and
// neighbouring pixels can be combined:
//   E_STORE   store, 0 where mask <= 0 when a mask is given
//   E_POOL    store, and the 2x2 average pool of the stored values
//   E_HEAD    store, and the output head on the stored values
//   E_UPSUM   data gradient of a concatenation: channels below c1 summed over
//             the 2x2 cells of the upsampled part, the others stored as they are
//   E_UNPOOL  data gradient of a pooled tensor: a quarter of the value added
//             to the skip's gradient at the four fine pixels, then the mask
// Every value is rounded to BF16 where a pass of its own stored it, so the
// results are those of separate passes bit for bit.
//
// Bound at 64 x 256 x 256: memory at 32 channels (read 268 MB, write 268 MB),
// the LDS and matrix rates at 64 and more.  With the elementwise passes as
// kernels of their own (one value per thread) a backward of that size took
// 19.9 ms, 14.5 ms this way; inference at 512 x 1024 756 and 546 us.
// Requires Cin % 32 == 0, Cout % BN == 0, W % TW == 0, H % (64 MB / TW) == 0;
// E_POOL and E_UPSUM TW = 64, MB = 4; E_HEAD BN = Cout = 32.
// ---------------------------------------------------------------------------
enum { E_STORE, E_POOL, E_HEAD, E_UPSUM, E_UNPOOL };
struct CSrc {
    const bf16* a;  // channels 0 .. ca-1
    const bf16* b;  // channels ca .. (nullptr: none, they are zero)
    int ca, up;     // up: a is at half resolution
};
struct CEpi {
    bf16* y;           // E_UPSUM: the coarse part's gradient
    bf16* y2;          // E_POOL: pooled; E_UPSUM: the skip's gradient
    const bf16* mask;  // nullptr: none
    const bf16* skip;  // E_UNPOOL
    int c1;            // E_UPSUM
    const float *wh, *bh;
    float* head;       // E_HEAD: [pixel][HK]
};
constexpr int HK = 5;  // channels of the output head

__device__ __forceinline__ bf16x8 masked(bf16x8 v, bf16x8 m) {
#pragma unroll
    for (int e = 0; e < 8; e++)
        if (!((float)m[e] > 0.0f)) v[e] = to_bf16(0.0f);
    return v;
}

template <int TAPS, int TW, int BN, int MB, bool RELU, int EPI>
__global__ __launch_bounds__(256, 2) void k_conv(CSrc X, const bf16* __restrict__ Wt, const float* __restrict__ bias,
                                                 CEpi E, int H, int W, int Cin, int Cout) {
    constexpr int TR = 64 * MB / TW;  // rows per tile
    constexpr int HALO = TAPS == 9 ? 1 : 0;
    constexpr int SR = TR + 2 * HALO, SC = TW + 2 * HALO;
    constexpr int XB = SR * SC * LROW, WB = TAPS * BN * LROW, LO = BN + 8, OB = 64 * MB * LO;
    constexpr int NX = (SR * SC * 4 + 255) / 256, NW = (TAPS * BN * 4 + 255) / 256;
    constexpr int CH = BN / 8;  // 16-byte chunks of a pixel's output channels
    __shared__ __attribute__((aligned(16))) bf16 sm[XB + WB > OB ? XB + WB : OB];
    bf16 *sX = sm, *sW = sm + XB;
    const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63, l16 = lane & 15, s = lane >> 4;
    const int ntx = W / TW;
    const int xt = blockIdx.x % ntx, cb = blockIdx.x / ntx;
    const int x0 = xt * TW, y0 = blockIdx.y * TR, n = blockIdx.z;
    const int co0 = cb * BN;
    f32x4 acc[MB][BN / 16];
#pragma unroll
    for (int m = 0; m < MB; m++)
#pragma unroll
        for (int j = 0; j < BN / 16; j++) acc[m][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    // the next channel block's values, 16-byte chunks of 8 channels
    bf16x8 rx[NX], rw[NW];
    auto load = [&](int c0) {
        const bool second = c0 >= X.ca && X.b;
        const int up = second ? 0 : X.up, C = second ? Cin - X.ca : X.ca, cc = second ? c0 - X.ca : c0;
        const bf16* src = (second ? X.b : X.a) + (size_t)n * (H >> up) * (W >> up) * C + cc;
#pragma unroll
        for (int it = 0; it < NX; it++) {
            const int k = tid + it * 256, ch = k & 3, pix = k >> 2;
            const int yy = y0 + pix / SC - HALO, xx = x0 + pix % SC - HALO;
            bf16x8 v = {};
            if (pix < SR * SC && yy >= 0 && yy < H && xx >= 0 && xx < W && cc + ch * 8 < C)
                v = *(const bf16x8*)(src + ((size_t)(yy >> up) * (W >> up) + (xx >> up)) * C + ch * 8);
            rx[it] = v;
        }
#pragma unroll
        for (int it = 0; it < NW; it++) {
            const int k = tid + it * 256, ch = k & 3, row = k >> 2;  // row = tap * BN + j
            const int tap = row / BN, j = row % BN;
            if (row < TAPS * BN) rw[it] = *(const bf16x8*)(Wt + ((size_t)tap * Cout + co0 + j) * Cin + c0 + ch * 8);
        }
    };
    load(0);
    for (int c0 = 0; c0 < Cin; c0 += KB) {
        __syncthreads();
#pragma unroll
        for (int it = 0; it < NX; it++) {
            const int k = tid + it * 256;
            if (k < SR * SC * 4) *(bf16x8*)(sX + (k >> 2) * LROW + (k & 3) * 8) = rx[it];
        }
#pragma unroll
        for (int it = 0; it < NW; it++) {
            const int k = tid + it * 256;
            if (k < TAPS * BN * 4) *(bf16x8*)(sW + (k >> 2) * LROW + (k & 3) * 8) = rw[it];
        }
        __syncthreads();
        if (c0 + KB < Cin) load(c0 + KB);
        auto wfrag = [&](int tap, int j) { return *(const bf16x8*)(sW + (tap * BN + 16 * j + l16) * LROW + s * 8); };
        auto xfrag = [&](int r, int c) { return *(const bf16x8*)(sX + (r * SC + c) * LROW + s * 8); };
        if (TAPS == 9 && TW == 64) {
            // the fragments of MB consecutive rows, row r in slot r % MB
            bf16x8 xf[3][MB];
#pragma unroll
            for (int dx = 0; dx < 3; dx++)
#pragma unroll
                for (int m = 0; m < MB; m++) xf[dx][m] = xfrag(m, 16 * w + l16 + dx);
#pragma unroll
            for (int dy = 0; dy < 3; dy++) {
                if (dy > 0) {
#pragma unroll
                    for (int dx = 0; dx < 3; dx++) xf[dx][(dy - 1) % MB] = xfrag(MB - 1 + dy, 16 * w + l16 + dx);
                }
#pragma unroll
                for (int dx = 0; dx < 3; dx++)
#pragma unroll
                    for (int j = 0; j < BN / 16; j++) {
                        const bf16x8 b = wfrag(dy * 3 + dx, j);
#pragma unroll
                        for (int m = 0; m < MB; m++) acc[m][j] = mfma16(b, xf[dx][(m + dy) % MB], acc[m][j]);
                    }
            }
        } else {
#pragma unroll
            for (int tap = 0; tap < TAPS; tap++) {
                const int dy = TAPS == 9 ? tap / 3 : 0, dx = TAPS == 9 ? tap % 3 : 0;
                bf16x8 a[MB];
#pragma unroll
                for (int m = 0; m < MB; m++) {
                    const int q = 64 * m + 16 * w + l16;  // this lane's pixel within the tile
                    a[m] = xfrag(q / TW + dy, q % TW + dx);
                }
#pragma unroll
                for (int j = 0; j < BN / 16; j++) {
                    const bf16x8 b = wfrag(tap, j);
#pragma unroll
                    for (int m = 0; m < MB; m++) acc[m][j] = mfma16(b, a[m], acc[m][j]);
                }
            }
        }
    }
    // the tile as BF16 in LDS: the lane holds channels 16 j + 4 s + 0..3 of
    // pixel 64 m + 16 w + l16
    __syncthreads();
#pragma unroll
    for (int j = 0; j < BN / 16; j++) {
        const int c = 16 * j + 4 * s;
        f32x4 bv = f32x4{0.f, 0.f, 0.f, 0.f};
        if (bias) {
#pragma unroll
            for (int r = 0; r < 4; r++) bv[r] = bias[co0 + c + r];
        }
#pragma unroll
        for (int m = 0; m < MB; m++) {
            bf16x4 o;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                float v = acc[m][j][r] + bv[r];
                if (RELU) v = v > 0.0f ? v : 0.0f;
                o[r] = to_bf16(v);
            }
            *(bf16x4*)(sm + (64 * m + 16 * w + l16) * LO + c) = o;
        }
    }
    __syncthreads();
    const size_t img = (size_t)n * H * W;
    auto at = [&](int px, int ch) { return *(const bf16x8*)(sm + px * LO + ch * 8); };
    auto pixel = [&](int px) { return img + (size_t)(y0 + px / TW) * W + x0 + px % TW; };
    if (EPI == E_STORE || EPI == E_POOL || EPI == E_HEAD) {
#pragma unroll
        for (int it = 0; it < 64 * MB * CH / 256; it++) {
            const int i = tid + it * 256, px = i / CH, ch = i % CH;
            const size_t o = pixel(px) * Cout + co0 + ch * 8;
            bf16x8 v = at(px, ch);
            if (EPI == E_STORE && E.mask) v = masked(v, *(const bf16x8*)(E.mask + o));
            *(bf16x8*)(E.y + o) = v;
        }
    }
    if (EPI == E_POOL || EPI == E_UPSUM) {
        // 2x2 cells of the tile: 2 x 32 of them
        for (int i = tid; i < 16 * MB * CH; i += 256) {
            const int pp = i / CH, ch = i % CH, py = pp / 32, pxx = pp % 32, q = 2 * py * TW + 2 * pxx;
            if (EPI == E_UPSUM && co0 + ch * 8 >= E.c1) continue;
            const bf16x8 v00 = at(q, ch), v01 = at(q + 1, ch), v10 = at(q + TW, ch), v11 = at(q + TW + 1, ch);
            bf16x8 o;
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const float t = (float)v00[e] + (float)v01[e] + (float)v10[e] + (float)v11[e];
                o[e] = to_bf16(EPI == E_POOL ? 0.25f * t : t);
            }
            const int Co = EPI == E_POOL ? Cout : E.c1;
            *(bf16x8*)((EPI == E_POOL ? E.y2 : E.y) +
                       (((size_t)n * (H / 2) + y0 / 2 + py) * (W / 2) + x0 / 2 + pxx) * Co + co0 + ch * 8) = o;
        }
    }
    if (EPI == E_UPSUM) {
        for (int i = tid; i < 64 * MB * CH; i += 256) {
            const int px = i / CH, ch = i % CH;
            if (co0 + ch * 8 < E.c1) continue;
            *(bf16x8*)(E.y2 + pixel(px) * (Cout - E.c1) + co0 + ch * 8 - E.c1) = at(px, ch);
        }
    }
    if (EPI == E_UNPOOL) {
        for (int i = tid; i < 64 * MB * CH; i += 256) {
            const int px = i / CH, ch = i % CH;
            const bf16x8 v = at(px, ch);
            const size_t o0 = (((size_t)n * H + y0 + px / TW) * 4 * W + 2 * (x0 + px % TW)) * Cout + co0 + ch * 8;
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const size_t o = o0 + ((size_t)(q >> 1) * 2 * W + (q & 1)) * Cout;
                const bf16x8 sk = *(const bf16x8*)(E.skip + o);
                bf16x8 g;
#pragma unroll
                for (int e = 0; e < 8; e++) g[e] = to_bf16(0.25f * (float)v[e] + (float)sk[e]);
                *(bf16x8*)(E.y + o) = masked(g, *(const bf16x8*)(E.mask + o));
            }
        }
    }
    if (EPI == E_HEAD) {
        // Y[p][k] = b[k] + sum_c X[p][c] W[k][c] in FP32, one pixel per thread
        for (int px = tid; px < 64 * MB; px += 256) {
            float a[HK];
#pragma unroll
            for (int k = 0; k < HK; k++) a[k] = E.bh[k];
#pragma unroll
            for (int ch = 0; ch < CH; ch++) {
                const bf16x8 v = at(px, ch);
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    const float x = (float)v[e];
#pragma unroll
                    for (int k = 0; k < HK; k++) a[k] += x * E.wh[k * BN + ch * 8 + e];
                }
            }
            float* o = E.head + pixel(px) * HK;
#pragma unroll
            for (int k = 0; k < HK; k++) o[k] = a[k];
        }
    }
}

// ---------------------------------------------------------------------------
// Weight and bias gradient of a convolution: dW[tap][co][ci] = sum over
// pixels of dZ[p][co] * X[p + tap offset][ci], db[co] = sum of dZ[p][co].
//
// Pixels are the K index of the products, channels the contiguous index in
// memory: rows of both tensors are staged as they lie, and the transposed
// LDS read (four pixels of one channel per lane and read) makes the
// fragments, so each value is staged once instead of once per shift, without
// a transpose through registers.  A wave holds a 32 x 32 block of (co, ci)
// for all taps (144 accumulators of 256 registers) and takes two rows of dZ
// at a time, so that a fragment of an X row serves both (28 fragment reads
// per 72 products).  A workgroup takes a CBO x CBI block; where that is
// fewer than four such blocks, the waves share the pixels of a stage (the
// two 32-pixel halves of a segment, then row pairs) and add their sums at
// the end.  It walks down a range of rows of SEG-pixel strips, keeping the
// rows that the next rows' taps need in a ring, the following rows in flight
// in registers.  The bias sums are products with a block of ones.
// Partials go to part[split][taps*Cout*Cin + Cout] (FP32).
//
// Bound by the LDS reads and the matrix rate at 64 channels, by memory at 32.
// At 64 x 256 x 256 the 17 layers' weight and bias gradients and their
// reductions take 1.9 ms, and took 8.2 ms before (one copy of X per shift,
// transposed in registers, every X row read three times; bias sums in a pass
// of their own).
// Requires Cout % CBO == 0, Cin % CBI == 0; W % SEG == 0 unless RAGGED, whose
// pixels past W have zero gradients; the column before them is taken out of
// their products, where an infinite input would give NaN (0 x inf).
// ---------------------------------------------------------------------------
typedef short s16x4 __attribute__((ext_vector_type(4)));
// Lane l of a wave gets channel l % 16 at the eight pixels 8 (l / 16) + 0..7
// of the block whose first pixel's channels are at q, pixels PS apart.
template <int PS>
__device__ __forceinline__ bf16x8 tr_frag(const bf16* q, int lane) {
    const bf16* a = q + (8 * (lane >> 4) + ((lane & 15) >> 2)) * PS + (lane & 3) * 4;
    typedef __attribute__((address_space(3))) s16x4* lds_ptr;
    const bf16x4 u = __builtin_bit_cast(bf16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)a));
    const bf16x4 v = __builtin_bit_cast(bf16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(a + 4 * PS)));
    return __builtin_shufflevector(u, v, 0, 1, 2, 3, 4, 5, 6, 7);
}

template <int CBO, int CBI, int SEG>
struct WShape {
    static constexpr int NS = (CBO / 32) * (CBI / 32), WK = 4 / NS;  // 32 x 32 blocks; waves that share one
    static constexpr int KC = SEG / 32, KG = WK < KC ? WK : KC;      // 32-pixel chunks of a row; chunk groups
    static constexpr int RW = 2, RS = (WK / KG) * RW;                // rows per wave and per stage
};

template <int TAPS, int CBO, int CBI, int SEG, bool RAGGED>
__global__ __launch_bounds__(256, 2) void k_conv_wgrad(CSrc X, const bf16* __restrict__ dZ, float* __restrict__ part,
                                                       int N, int H, int W, int Cin, int Cout, int rows_per_split) {
    using S = WShape<CBO, CBI, SEG>;
    constexpr int HALO = TAPS == 9 ? 1 : 0, NDX = 2 * HALO + 1;
    constexpr int RS = S::RS, RW = S::RW, NRX = RS + 2 * HALO, XP = SEG + 2 * HALO;
    // pixel strides that spread the four pixel rows of a transposed read over the banks
    constexpr int PX = CBI == 64 ? 72 : 48, PD = CBO == 64 ? 72 : 48;
    constexpr int XROW = XP * PX, DROW = SEG * PD;
    constexpr int CX = CBI / 8, CD = CBO / 8;  // 16-byte chunks of a pixel
    constexpr int NX = (RS * XP * CX + 255) / 256, ND = (RS * SEG * CD + 255) / 256;
    constexpr int TG = TAPS == 9 ? 3 : 1;                         // taps added per round of the waves' final sum
    constexpr int RED = (S::WK - 1) * S::NS * (TG * 4 + 2) * 256 * 2;  // in bf16 units
    constexpr int LDS = NRX * XROW + RS * DROW;
    __shared__ __attribute__((aligned(16))) bf16 sm[LDS > RED ? LDS : RED];
    bf16 *sX = sm, *sD = sm + NRX * XROW;
    const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63, s = lane >> 4, l16 = lane & 15;
    const int cob = blockIdx.x % (Cout / CBO), cib = blockIdx.x / (Cout / CBO);
    const int co0 = cob * CBO, ci0 = cib * CBI, split = blockIdx.y;
    const int sub = w % S::NS, kg = w / S::NS;
    const int cs = (sub % (CBO / 32)) * 32, is = (sub / (CBO / 32)) * 32;  // the wave's block
    const int kc0 = kg % S::KG, row0 = (kg / S::KG) * RW;                  // its chunk and its first row of a stage
    const bool bias = cib == 0 && is == 0;
    f32x4 acc[TAPS][2][2], accb[2];
#pragma unroll
    for (int t = 0; t < TAPS; t++)
#pragma unroll
        for (int q = 0; q < 4; q++) acc[t][q >> 1][q & 1] = f32x4{0.f, 0.f, 0.f, 0.f};
    accb[0] = accb[1] = f32x4{0.f, 0.f, 0.f, 0.f};
    bf16x8 ones;
#pragma unroll
    for (int e = 0; e < 8; e++) ones[e] = to_bf16(1.0f);
    const int nseg = (W + SEG - 1) / SEG;
    const int r1 = min(N * nseg * H, (split + 1) * rows_per_split);
    int n = 0, x0 = 0, yend = 0;
    // 16-byte chunks of X (rows yb.., nothing past the run's last tap row)
    // and of dZ (rows yb.. of the run)
    auto ldx = [&](int k, int yb) {
        const int c = ci0 + (k % CX) * 8, px = (k / CX) % XP, y = yb + k / (CX * XP), x = x0 + px - HALO;
        const bool second = c >= X.ca && X.b;
        const int up = second ? 0 : X.up, C = second ? Cin - X.ca : X.ca, cc = second ? c - X.ca : c;
        bf16x8 v = {};
        if (y >= 0 && y < min(H, yend + HALO) && x >= 0 && x < W && cc < C)
            v = *(const bf16x8*)((second ? X.b : X.a) + (((size_t)n * (H >> up) + (y >> up)) * (W >> up) + (x >> up)) * C + cc);
        return v;
    };
    auto ldd = [&](int k, int yb) {
        const int c = co0 + (k % CD) * 8, px = (k / CD) % SEG, y = yb + k / (CD * SEG), x = x0 + px;
        bf16x8 v = {};
        if (y < yend && x < W) v = *(const bf16x8*)(dZ + (((size_t)n * H + y) * W + x) * Cout + c);
        return v;
    };
    for (int r = split * rows_per_split; r < r1;) {
        const int strip = r / H, y0 = r % H;
        n = strip / nseg;
        x0 = (strip % nseg) * SEG;
        yend = min(H, y0 + r1 - r);
        r += yend - y0;
        int base = 0;  // ring slot of row yy - HALO
        __syncthreads();
        for (int k = tid; k < NRX * XP * CX; k += 256)
            *(bf16x8*)(sX + (k / CX) * PX + (k % CX) * 8) = ldx(k, y0 - HALO);
        for (int k = tid; k < RS * SEG * CD; k += 256)
            *(bf16x8*)(sD + (k / CD) * PD + (k % CD) * 8) = ldd(k, y0);
        __syncthreads();
        for (int yy = y0; yy < yend; yy += RS) {
            const bool more = yy + RS < yend;
            bf16x8 rx[NX], rd[ND];
            if (more) {
#pragma unroll
                for (int it = 0; it < NX; it++) rx[it] = ldx(tid + it * 256, yy + RS + HALO);
#pragma unroll
                for (int it = 0; it < ND; it++) rd[it] = ldd(tid + it * 256, yy + RS);
            }
#pragma unroll
            for (int kc = 0; kc < S::KC / S::KG; kc++) {
                const int p0 = (kc0 + kc * S::KG) * 32;
                bf16x8 a[RW][2];
#pragma unroll
                for (int z = 0; z < RW; z++)
#pragma unroll
                    for (int t = 0; t < 2; t++) a[z][t] = tr_frag<PD>(sD + (row0 + z) * DROW + p0 * PD + cs + 16 * t, lane);
                if (bias) {
#pragma unroll
                    for (int z = 0; z < RW; z++)
#pragma unroll
                        for (int t = 0; t < 2; t++) accb[t] = mfma16(a[z][t], ones, accb[t]);
                }
#pragma unroll
                for (int xr = 0; xr < RW + 2 * HALO; xr++) {
                    int slot = base + row0 + xr;
                    if (slot >= NRX) slot -= NRX;
#pragma unroll
                    for (int dx = 0; dx < NDX; dx++) {
                        bf16x8 b[2];
#pragma unroll
                        for (int u = 0; u < 2; u++) {
                            b[u] = tr_frag<PX>(sX + slot * XROW + (p0 + dx) * PX + is + 16 * u, lane);
                            if (RAGGED && dx == 0) {
#pragma unroll
                                for (int e = 0; e < 8; e++)
                                    if (x0 + p0 + 8 * s + e >= W) b[u][e] = to_bf16(0.0f);
                            }
                        }
#pragma unroll
                        for (int z = 0; z < RW; z++) {
                            const int dy = xr - z;
                            if (dy < 0 || dy >= NDX || yy + row0 + z >= yend) continue;
#pragma unroll
                            for (int t = 0; t < 2; t++)
#pragma unroll
                                for (int u = 0; u < 2; u++)
                                    acc[dy * NDX + dx][t][u] = mfma16(a[z][t], b[u], acc[dy * NDX + dx][t][u]);
                        }
                    }
                }
            }
            if (more) {
                __syncthreads();
                // the oldest RS rows of the ring give way
#pragma unroll
                for (int it = 0; it < NX; it++) {
                    const int k = tid + it * 256;
                    if (k < RS * XP * CX) {
                        int slot = base + k / (CX * XP);
                        if (slot >= NRX) slot -= NRX;
                        *(bf16x8*)(sX + slot * XROW + ((k / CX) % XP) * PX + (k % CX) * 8) = rx[it];
                    }
                }
#pragma unroll
                for (int it = 0; it < ND; it++) {
                    const int k = tid + it * 256;
                    if (k < RS * SEG * CD) *(bf16x8*)(sD + (k / CD) * PD + (k % CD) * 8) = rd[it];
                }
                base += RS;
                if (base >= NRX) base -= NRX;
                __syncthreads();
            }
        }
    }
    // the waves that share a block add their sums, in wave order
    if constexpr (S::WK > 1) {
        f32x4* red = (f32x4*)sm;
        constexpr int SL = TG * 4 + 2;
#pragma unroll
        for (int g = 0; g < TAPS / TG; g++) {
            __syncthreads();
            if (kg > 0) {
                f32x4* o = red + ((kg - 1) * S::NS + sub) * SL * 64 + lane;
#pragma unroll
                for (int t = 0; t < TG; t++)
#pragma unroll
                    for (int q = 0; q < 4; q++) o[(t * 4 + q) * 64] = acc[g * TG + t][q >> 1][q & 1];
                if (g == 0) {
                    o[TG * 4 * 64] = accb[0];
                    o[(TG * 4 + 1) * 64] = accb[1];
                }
            }
            __syncthreads();
            if (kg == 0) {
#pragma unroll
                for (int j = 0; j < S::WK - 1; j++) {
                    const f32x4* o = red + (j * S::NS + sub) * SL * 64 + lane;
#pragma unroll
                    for (int t = 0; t < TG; t++)
#pragma unroll
                        for (int q = 0; q < 4; q++) acc[g * TG + t][q >> 1][q & 1] += o[(t * 4 + q) * 64];
                    if (g == 0) {
                        accb[0] += o[TG * 4 * 64];
                        accb[1] += o[(TG * 4 + 1) * 64];
                    }
                }
            }
        }
        if (kg > 0) return;
    }
    // lane holds rows (co) 4 s + r of tile t, column (ci) l16 of tile u
    float* o = part + (size_t)split * ((size_t)TAPS * Cout * Cin + Cout);
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int co = co0 + cs + 16 * t + 4 * s + r;
#pragma unroll
            for (int tap = 0; tap < TAPS; tap++)
#pragma unroll
                for (int u = 0; u < 2; u++)
                    o[((size_t)tap * Cout + co) * Cin + ci0 + is + 16 * u + l16] = acc[tap][t][u][r];
            if (bias && l16 == 0) o[(size_t)TAPS * Cout * Cin + co] = accb[t][r];
        }
}

// Sums over splits: job j sums part[s*n + i] over its splits into out[i]
// (i < nw) or outb[i - nw] (unless NULL).  Four threads take every fourth
// split in order, their sums are added in order.  64 values per workgroup:
// the loads of a wavefront are contiguous, and a short vector still spreads
// over many workgroups.  One launch serves as many layers as the partials
// buffer holds (18 launches of 5 us each on small batches before).
constexpr int NLAYER = 18;
struct SumJob {
    const float* part;
    float *out, *outb;
    int nsplit, blk0;  // first workgroup of the job
    unsigned n, nw;
};
struct SumJobs {
    int count, blocks;
    SumJob j[NLAYER];
};
__global__ __launch_bounds__(256) void k_reduce_parts(SumJobs J) {
    __shared__ float red[4][64];
    int k = 0;
    while (k + 1 < J.count && (int)blockIdx.x >= J.j[k + 1].blk0) k++;
    const SumJob q = J.j[k];
    const int l = threadIdx.x & 63, g = threadIdx.x >> 6;
    const size_t i = (size_t)(blockIdx.x - q.blk0) * 64 + l;
    float a = 0.0f;
    if (i < q.n) {
#pragma unroll 8
        for (int sp = g; sp < q.nsplit; sp += 4) a += q.part[(size_t)sp * q.n + i];
    }
    red[g][l] = a;
    __syncthreads();
    if (g == 0 && i < q.n) {
        a = ((red[0][l] + red[1][l]) + red[2][l]) + red[3][l];
        if (i < q.nw) q.out[i] = a;
        else if (q.outb) q.outb[i - q.nw] = a;
    }
}

// Flipped, transposed weights for the data gradients: per layer
// Wd[tap][ci][co] = W[taps-1-tap][co][ci] (the 180-degree rotation of a 3x3
// kernel), at the layer's offset w.  All layers in one launch.
struct FlipJob {
    size_t w;
    int taps, cout, cin, blk0;
};
struct FlipJobs {
    int count, blocks;
    FlipJob j[NLAYER];
};
__global__ __launch_bounds__(256) void k_flip_weights(const bf16* __restrict__ Wt, bf16* __restrict__ Wd, FlipJobs J) {
    int k = 0;
    while (k + 1 < J.count && (int)blockIdx.x >= J.j[k + 1].blk0) k++;
    const FlipJob q = J.j[k];
    const size_t i = (size_t)(blockIdx.x - q.blk0) * 256 + threadIdx.x;  // a layer may have 2^31 weights or more
    if (i >= (size_t)q.taps * q.cout * q.cin) return;
    const size_t r = i / q.cin;
    const int ci = i % q.cin, co = r % q.cout, tap = r / q.cout;
    Wd[q.w + ((size_t)(q.taps - 1 - tap) * q.cin + ci) * q.cout + co] = Wt[q.w + i];
}

// Backward of the output head (a 1x1 convolution of HC channels to HK in
// FP32; its forward is the E_HEAD epilogue): from the gradient dY[p][k] of
// its outputs, dX[p][c] = sum_k dY[p][k] W[k][c] where X > 0 (the ReLU that
// made X), and the partials of dW[k][c] = sum_p dY[p][k] X[p][c] and
// db[k] = sum_p dY[p][k]: part[blk][HK*HC + HK].  Four threads of eight
// channels take a pixel.  Bound by memory (148 B a pixel).
constexpr int HC = 32;
__global__ __launch_bounds__(256) void k_head_bwd(const float* __restrict__ dY, const float* __restrict__ Wh,
                                                  const bf16* __restrict__ X, bf16* __restrict__ dX, size_t P, int ppb,
                                                  float* __restrict__ part) {
    __shared__ float red[4][HK * HC + HK];
    const int tid = threadIdx.x, c = (tid & 3) * 8;
    const size_t p0 = (size_t)blockIdx.x * ppb, p1 = p0 + ppb < P ? p0 + ppb : P;
    float w[HK][8], a[HK][8], b[HK];
#pragma unroll
    for (int k = 0; k < HK; k++) {
        b[k] = 0.0f;
#pragma unroll
        for (int e = 0; e < 8; e++) {
            w[k][e] = Wh[k * HC + c + e];
            a[k][e] = 0.0f;
        }
    }
#pragma unroll 2
    for (size_t p = p0 + (tid >> 2); p < p1; p += 64) {
        const bf16x8 x = *(const bf16x8*)(X + p * HC + c);
        float d[HK];
#pragma unroll
        for (int k = 0; k < HK; k++) d[k] = dY[p * HK + k];
        bf16x8 o;
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const float xe = (float)x[e];
            float g = 0.0f;
#pragma unroll
            for (int k = 0; k < HK; k++) {
                g += d[k] * w[k][e];
                a[k][e] += d[k] * xe;
            }
            o[e] = to_bf16(xe > 0.0f ? g : 0.0f);
        }
        *(bf16x8*)(dX + p * HC + c) = o;
#pragma unroll
        for (int k = 0; k < HK; k++) b[k] += d[k];
    }
    // over the 16 pixels of a wavefront, then over the four wavefronts
#pragma unroll
    for (int k = 0; k < HK; k++) {
#pragma unroll
        for (int o = 4; o < 64; o <<= 1) {
            b[k] += __shfl_xor(b[k], o, 64);
#pragma unroll
            for (int e = 0; e < 8; e++) a[k][e] += __shfl_xor(a[k][e], o, 64);
        }
        if ((tid & 63) < 4) {
#pragma unroll
            for (int e = 0; e < 8; e++) red[tid >> 6][k * HC + c + e] = a[k][e];
            if ((tid & 3) == 0) red[tid >> 6][HK * HC + k] = b[k];
        }
    }
    __syncthreads();
    for (int i = tid; i < HK * HC + HK; i += 256)
        part[(size_t)blockIdx.x * (HK * HC + HK) + i] = red[0][i] + red[1][i] + red[2][i] + red[3][i];
}

// Mean squared error over the normalised targets: per-workgroup partial
// sums of (y - t)^2 (double) and, with G, the gradient g = 2 (y - t) / n.
// n is a multiple of 4.
__global__ __launch_bounds__(256) void k_mse(const float* __restrict__ Y, const bf16* __restrict__ T, size_t n,
                                             float* __restrict__ G, double* __restrict__ part) {
    __shared__ double red[256];
    double e = 0.0;
#pragma unroll 2
    for (size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * 4; i < n; i += (size_t)gridDim.x * 1024) {
        const f32x4 y = *(const f32x4*)(Y + i);
        const bf16x4 t = *(const bf16x4*)(T + i);
        f32x4 g;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const float d = y[k] - (float)t[k];
            g[k] = 2.0f * d / (float)n;
            e += (double)(d * d);
        }
        if (G) *(f32x4*)(G + i) = g;
    }
    red[threadIdx.x] = e;
    __syncthreads();
    for (int st = 128; st > 0; st >>= 1) {
        if ((int)threadIdx.x < st) red[threadIdx.x] += red[threadIdx.x + st];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}
// out = sum of part[0..n-1] / cnt, by one workgroup
__global__ __launch_bounds__(256) void k_mean(const double* __restrict__ part, int n, double cnt,
                                              double* __restrict__ out) {
    __shared__ double red[256];
    double e = 0.0;
    for (int i = threadIdx.x; i < n; i += 256) e += part[i];
    red[threadIdx.x] = e;
    __syncthreads();
    for (int st = 128; st > 0; st >>= 1) {
        if ((int)threadIdx.x < st) red[threadIdx.x] += red[threadIdx.x + st];
        __syncthreads();
    }
    if (threadIdx.x == 0) *out = red[0] / cnt;
}

// Adam (Kingma and Ba 2015) on FP32 masters; the BF16 copy (may be NULL)
// follows the update.  bc1 = 1 - beta1^t, bc2 = 1 - beta2^t.
__global__ __launch_bounds__(256) void k_adam(float* __restrict__ w, bf16* __restrict__ w16,
                                              const float* __restrict__ g, float* __restrict__ m,
                                              float* __restrict__ v, size_t n, float lr, float b1, float b2,
                                              float eps, float bc1, float bc2) {
    size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    float gi = g[i];
    float mi = b1 * m[i] + (1.0f - b1) * gi;
    float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    float mh = mi / bc1, vh = vi / bc2;
    float wi = w[i] - lr * mh / (sqrtf(vh) + eps);
    w[i] = wi;
    if (w16) w16[i] = to_bf16(wi);
}

__global__ __launch_bounds__(256) void k_f32_to_bf16(const float* __restrict__ a, bf16* __restrict__ b, size_t n) {
    size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) b[i] = to_bf16(a[i]);
}

}  // namespace

// ===========================================================================
// The network: a 4-level convolutional encoder-decoder (U-Net shape)
//   level 0 (H x W):       32 ch   conv3 x2          skip0
//   level 1 (H/2 x W/2):   64 ch   pool, conv3 x2    skip1
//   level 2 (H/4 x W/4):  128 ch   pool, conv3 x2    skip2
//   level 3 (H/8 x W/8):  256 ch   pool, conv3 x2
//   decoder: conv1 (halve channels) at the coarse level, nearest 2x
//   upsampling, concatenation with the skip, conv3 x2; head conv1 32 -> 5
// ReLU after every 3x3 convolution; the 1x1 convolutions are linear.
// Inputs: 8 channels (zb, zs, uu, vv, Hm0, Tp, dir, 0) of the first
// convolution's 32; outputs: 5 channels (H, Dw, Dr, Fx, Fy), normalised.
// 1.8 M parameters.  H must be even and W/8 either 32 or a multiple of 64.
// ===========================================================================
namespace {

struct ConvL {
    int cin, cout, taps, relu;
    size_t w, b;  // offsets of weights [taps][cout][cin] and bias [cout] in the parameter vector
};

}  // namespace

struct xbg_sur {
    int nmax = 0, H = 0, W = 0;
    hipStream_t st = nullptr;
    std::vector<ConvL> L;  // 17 convolutions, then the head (index 17)
    size_t nparam = 0;
    float *P = nullptr, *G = nullptr, *M = nullptr, *V = nullptr;  // FP32 params, grads, Adam moments
    bf16* P16 = nullptr;                                           // BF16 copy of the parameter vector
    bf16* Wd = nullptr;                                            // flipped weights for the data gradients
    float* part = nullptr;                                         // split-K / reduction partials
    size_t npart = 0, upart = 0;                                   // size, and how much the queued sums use
    SumJobs sums{};                                                // sums queued for the next launch
    double* lossp = nullptr;                                       // loss partials, then the loss
    double* hloss = nullptr;                                       // the loss on the host (pinned)
    hipEvent_t loss_done = nullptr;
    int adam_t = 0;
    // the batch, activations (A) and their gradients (D), by name
    std::vector<void*> allocs;
    bf16 *x8, *e0a, *e0, *p1, *e1a, *e1, *p2, *e2a, *e2, *p3, *b3a, *b3, *u2, *d2a, *d2, *u1, *d1a, *d1,
        *u0, *d0a, *d0;
    bf16 *g_e0a, *g_e0, *g_e1a, *g_e1, *g_e2a, *g_e2, *g_b3a, *g_b3, *g_u2, *g_d2a,
        *g_d2, *g_u1, *g_d1a, *g_d1, *g_u0, *g_d0a, *g_d0;
    float *y = nullptr, *gy = nullptr;
    std::string err;
};

namespace {

thread_local std::string g_sur_error;

int sfail(xbg_sur* s, int code, const std::string& m) {
    if (s) s->err = m;
    else g_sur_error = m;
    return code;
}
#define SHIP(s, call)                                                                            \
    do {                                                                                         \
        hipError_t e_ = (call);                                                                  \
        if (e_ != hipSuccess) return sfail(s, XBG_E_HIP, std::string(#call) + ": " + hipGetErrorString(e_)); \
    } while (0)

inline unsigned nblk(size_t n) { return (unsigned)((n + 255) / 256); }

// k_conv for any supported shape; the fused epilogues run at the sizes the
// network gives them (E_POOL, E_UPSUM: rows of 64 pixels in fours)
template <int EPI, bool RELU>
int conv(hipStream_t st, CSrc X, const bf16* Wt, const float* bias, const CEpi& E, int n, int H, int W, int Cin,
         int Cout, int taps) {
    if (Cin % 32 || Cout % 32 || !(taps == 1 || taps == 9)) return XBG_E_ARG;
    const int TW = W % 64 == 0 ? 64 : (W == 32 ? 32 : 0);
    if (!TW || H % (64 / TW)) return XBG_E_ARG;
    const int BN = Cout % 64 == 0 ? 64 : 32;
    // four 16-pixel blocks per wave where the rows divide, else one
    const int MB = H % (4 * 64 / TW) == 0 ? 4 : 1;
    const dim3 g((W / TW) * (Cout / BN), H / (MB * 64 / TW), n);
    constexpr bool CELLS = EPI == E_POOL || EPI == E_UPSUM;
    if (CELLS && (TW != 64 || MB != 4)) return XBG_E_ARG;
    if (EPI == E_HEAD && (Cout != 32 || TW != 64 || taps != 9)) return XBG_E_ARG;
#define CF(T_, TW_, BN_, MB_) k_conv<T_, TW_, BN_, MB_, RELU, EPI><<<g, dim3(256), 0, st>>>(X, Wt, bias, E, H, W, Cin, Cout)
#define CF_MB(T_, TW_, BN_)                                   \
    do {                                                      \
        if constexpr (CELLS) CF(T_, TW_, BN_, 4);             \
        else if (MB == 4) CF(T_, TW_, BN_, 4);                \
        else CF(T_, TW_, BN_, 1);                             \
    } while (0)
#define CF_BN(T_, TW_)                                        \
    do {                                                      \
        if constexpr (EPI == E_HEAD) CF_MB(T_, TW_, 32);      \
        else if (BN == 64) CF_MB(T_, TW_, 64);                \
        else CF_MB(T_, TW_, 32);                              \
    } while (0)
#define CF_TW(T_)                                             \
    do {                                                      \
        if constexpr (CELLS || EPI == E_HEAD) CF_BN(T_, 64);  \
        else if (TW == 64) CF_BN(T_, 64);                     \
        else CF_BN(T_, 32);                                   \
    } while (0)
    if constexpr (EPI != E_STORE) {
        if (taps != 9) return XBG_E_ARG;
        CF_TW(9);
    } else {
        if (taps == 9) CF_TW(9);
        else CF_TW(1);
    }
#undef CF
#undef CF_MB
#undef CF_BN
#undef CF_TW
    return hipGetLastError() == hipSuccess ? 0 : XBG_E_HIP;
}

// a tensor of c channels; the network's input has 8 and its convolution 32,
// the others being zero
CSrc plain(const bf16* x, int c) { return CSrc{x, nullptr, c, 0}; }
// the concatenation of a tensor of c channels at half resolution, each pixel
// standing for 2 x 2, and a skip of the other channels
CSrc concat(const bf16* u, const bf16* e, int c) { return CSrc{u, e, c, 1}; }

constexpr int MSE_PARTS = 1024;

// sums queued over part[nsplit][n]: nw values into out, the rest into outb
void queue_sum(SumJobs& J, const float* part, int nsplit, size_t n, size_t nw, float* out, float* outb) {
    J.j[J.count++] = SumJob{part, out, outb, nsplit, J.blocks, (unsigned)n, (unsigned)nw};
    J.blocks += (int)((n + 63) / 64);
}
void run_sums(hipStream_t st, SumJobs& J) {
    if (J.count) k_reduce_parts<<<J.blocks, dim3(256), 0, st>>>(J);
    J.count = J.blocks = 0;
}

// rows of one stage of k_conv_wgrad (WShape::RS)
int wgrad_stage_rows(int CBO, int CBI, int SEG) {
    const int wk = 4 / ((CBO / 32) * (CBI / 32)), kg = wk < SEG / 32 ? wk : SEG / 32;
    return 2 * (wk / kg);
}

// dW (FP32, [taps][Cout][Cin]) and db (Cout, may be NULL) of one convolution
// from its input X and the gradient dZ of its pre-activation output: partials
// behind the *used floats of part (npart) that queued sums hold, their sum
// queued; queued sums run first where the buffer or the table is full
int conv_wgrad(hipStream_t st, CSrc X, const bf16* dZ, float* dW, float* db, float* part, size_t npart, size_t* used,
               SumJobs& J, int n, int H, int W, int Cin, int Cout, int taps) {
    if (Cin % 32 || Cout % 32 || !(taps == 1 || taps == 9)) return XBG_E_ARG;
    const int CBO = Cout % 64 == 0 ? 64 : 32, CBI = Cin % 64 == 0 ? 64 : 32;
    const int gx = (Cout / CBO) * (Cin / CBI);
    const size_t per = (size_t)taps * Cout * Cin, np = per + Cout;
    // strips of 64 pixels, of 32 where rows are not a multiple of 64
    const int SEG = W % 64 == 0 ? 64 : 32;
    const int rows = n * ((W + SEG - 1) / SEG) * H;
    // two workgroups per CU, each of at least two stages (a small batch is
    // bound by the walk down the rows, about 3 us a stage: 16 rows each made
    // the 3 x 48 x 256 gradients 0.28 ms at 64 channels), within the buffer
    const int rs = wgrad_stage_rows(CBO, CBI, SEG);
    int want = 512 / gx;
    if (want < 1) want = 1;
    if (npart / np < (size_t)want) want = (int)(npart / np);
    if (want < 1) return XBG_E_ARG;
    int rps = (rows + want - 1) / want;
    if (rps < 2 * rs) rps = 2 * rs;
    rps = (rps + rs - 1) / rs * rs;
    const dim3 g(gx, (rows + rps - 1) / rps);
    if (J.count == NLAYER || *used + g.y * np > npart) {
        run_sums(st, J);
        *used = 0;
    }
    part += *used;
#define CWK(T_, O_, I_, S_, R_) k_conv_wgrad<T_, O_, I_, S_, R_><<<g, dim3(256), 0, st>>>(X, dZ, part, n, H, W, Cin, Cout, rps)
#define CW(T_, O_, I_)                                               \
    do {                                                             \
        if (SEG == 64) CWK(T_, O_, I_, 64, false);                   \
        else if (T_ == 9 && W % 32) CWK(T_, O_, I_, 32, T_ == 9);    \
        else CWK(T_, O_, I_, 32, false);                             \
    } while (0)
#define CW_I(T_, O_) do { if (CBI == 64) CW(T_, O_, 64); else CW(T_, O_, 32); } while (0)
#define CW_O(T_) do { if (CBO == 64) CW_I(T_, 64); else CW_I(T_, 32); } while (0)
    if (taps == 9) CW_O(9);
    else CW_O(1);
#undef CWK
#undef CW
#undef CW_I
#undef CW_O
    queue_sum(J, part, (int)g.y, np, per, dW, db);
    *used += g.y * np;
    return hipGetLastError() == hipSuccess ? 0 : XBG_E_HIP;
}

void queue_flip(FlipJobs& J, size_t w, int taps, int cout, int cin) {
    J.j[J.count++] = FlipJob{w, taps, cout, cin, J.blocks};
    J.blocks += (int)nblk((size_t)taps * cout * cin);
}

// deterministic initialisation: He-normal weights from a counter-based hash
// (Box-Muller on two 24-bit uniforms), zero biases
unsigned long long mix64(unsigned long long x) {
    x += 0x9E3779B97F4A7C15ull;
    x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
    x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
    return x ^ (x >> 31);
}
double gauss(unsigned seed, size_t i) {
    unsigned long long h = mix64(((unsigned long long)seed << 40) ^ (unsigned long long)i);
    double u1 = ((h >> 40) + 0.5) / 16777216.0, u2 = (((h >> 16) & 0xFFFFFF) + 0.5) / 16777216.0;
    return std::sqrt(-2.0 * std::log(u1)) * std::cos(6.283185307179586 * u2);
}

}  // namespace

extern "C" {

const char* xbg_sur_last_error(const xbg_sur* s) { return s ? s->err.c_str() : g_sur_error.c_str(); }

int xbg_sur_destroy(xbg_sur* s) {
    if (!s) return XBG_OK;
    if (s->st) hipStreamSynchronize(s->st);
    for (void* p : s->allocs) hipFree(p);
    if (s->hloss) hipHostFree(s->hloss);
    if (s->loss_done) hipEventDestroy(s->loss_done);
    if (s->st) hipStreamDestroy(s->st);
    delete s;
    return XBG_OK;
}

int xbg_sur_create(int nmax, int H, int W, unsigned seed, xbg_sur** out) {
    if (!out || nmax < 1 || H < 16 || H % 16 || !((W / 8 == 32 && W % 8 == 0) || (W % 512 == 0)))
        return sfail(nullptr, XBG_E_ARG, "xbg_sur_create: need H a multiple of 16 and W = 256 or a multiple of 512");
    *out = nullptr;
    xbg_sur* s = new xbg_sur();
    s->nmax = nmax;
    s->H = H;
    s->W = W;
    auto bail = [&](int rc) {
        xbg_sur_destroy(s);
        return rc;
    };
    const int spec[17][4] = {{32, 32, 9, 1},   {32, 32, 9, 1},   {32, 64, 9, 1},   {64, 64, 9, 1},
                             {64, 128, 9, 1},  {128, 128, 9, 1}, {128, 256, 9, 1}, {256, 256, 9, 1},
                             {256, 128, 1, 0}, {256, 128, 9, 1}, {128, 128, 9, 1}, {128, 64, 1, 0},
                             {128, 64, 9, 1},  {64, 64, 9, 1},   {64, 32, 1, 0},   {64, 32, 9, 1},
                             {32, 32, 9, 1}};
    size_t off = 0;
    for (auto& q : spec) {
        ConvL c{q[0], q[1], q[2], q[3], off, 0};
        off += (size_t)c.taps * c.cout * c.cin;
        c.b = off;
        off += c.cout;
        s->L.push_back(c);
    }
    ConvL head{32, 5, 1, 0, off, 0};
    off += 5 * 32;
    head.b = off;
    off += 5;
    s->L.push_back(head);
    s->nparam = off;
    if (hipStreamCreateWithFlags(&s->st, hipStreamNonBlocking) != hipSuccess)
        return bail(sfail(nullptr, XBG_E_HIP, "xbg_sur_create: stream"));
    auto A = [&](void** p, size_t bytes) -> bool {
        if (hipMalloc(p, bytes ? bytes : 16) != hipSuccess) return false;
        s->allocs.push_back(*p);  // freed by xbg_sur_destroy on any failure below
        return hipMemset(*p, 0, bytes) == hipSuccess;
    };
    const size_t P0 = (size_t)nmax * H * W, P1 = P0 / 4, P2 = P0 / 16, P3 = P0 / 64;
    bool ok = A((void**)&s->P, off * 4) && A((void**)&s->G, off * 4) && A((void**)&s->M, off * 4) &&
              A((void**)&s->V, off * 4) && A((void**)&s->P16, off * 2) && A((void**)&s->Wd, off * 2);
    s->npart = (size_t)32 << 20;
    ok = ok && A((void**)&s->part, s->npart * 4) && A((void**)&s->lossp, (MSE_PARTS + 1) * 8) &&
         hipHostMalloc((void**)&s->hloss, sizeof(double), hipHostMallocDefault) == hipSuccess &&
         hipEventCreateWithFlags(&s->loss_done, hipEventDisableTiming) == hipSuccess;
    struct B {
        bf16** p;
        size_t n;
    } acts[] = {{&s->x8, P0 * 8}, {&s->e0a, P0 * 32}, {&s->e0, P0 * 32},  {&s->p1, P1 * 32},
                {&s->e1a, P1 * 64}, {&s->e1, P1 * 64},  {&s->p2, P2 * 64},  {&s->e2a, P2 * 128},
                {&s->e2, P2 * 128}, {&s->p3, P3 * 128}, {&s->b3a, P3 * 256}, {&s->b3, P3 * 256},
                {&s->u2, P3 * 128}, {&s->d2a, P2 * 128}, {&s->d2, P2 * 128},
                {&s->u1, P2 * 64},  {&s->d1a, P1 * 64}, {&s->d1, P1 * 64},
                {&s->u0, P1 * 32},  {&s->d0a, P0 * 32}, {&s->d0, P0 * 32},
                {&s->g_e0a, P0 * 32}, {&s->g_e0, P0 * 32}, {&s->g_e1a, P1 * 64},
                {&s->g_e1, P1 * 64}, {&s->g_e2a, P2 * 128}, {&s->g_e2, P2 * 128},
                {&s->g_b3a, P3 * 256}, {&s->g_b3, P3 * 256}, {&s->g_u2, P3 * 128},
                {&s->g_d2a, P2 * 128}, {&s->g_d2, P2 * 128}, {&s->g_u1, P2 * 64},
                {&s->g_d1a, P1 * 64}, {&s->g_d1, P1 * 64}, {&s->g_u0, P1 * 32},
                {&s->g_d0a, P0 * 32}, {&s->g_d0, P0 * 32}};
    for (auto& b : acts) ok = ok && A((void**)b.p, b.n * 2);
    ok = ok && A((void**)&s->y, P0 * 5 * 4) && A((void**)&s->gy, P0 * 5 * 4);
    if (!ok) return bail(sfail(nullptr, XBG_E_HIP, "xbg_sur_create: out of device memory"));
    // He-normal initialisation
    std::vector<float> h(off, 0.0f);
    for (auto& c : s->L) {
        double sd = std::sqrt(2.0 / (c.taps * c.cin));
        if (!c.relu) sd = std::sqrt(1.0 / (c.taps * c.cin));
        for (size_t i = 0; i < (size_t)c.taps * c.cout * c.cin; i++) h[c.w + i] = (float)(sd * gauss(seed, c.w + i));
    }
    if (hipMemcpy(s->P, h.data(), off * 4, hipMemcpyHostToDevice) != hipSuccess)
        return bail(sfail(nullptr, XBG_E_HIP, "xbg_sur_create: upload"));
    k_f32_to_bf16<<<nblk(off), 256, 0, s->st>>>(s->P, s->P16, off);
    if (hipStreamSynchronize(s->st) != hipSuccess) return bail(sfail(nullptr, XBG_E_HIP, "xbg_sur_create: init"));
    *out = s;
    return XBG_OK;
}

size_t xbg_sur_nparams(const xbg_sur* s) { return s ? s->nparam : 0; }

int xbg_sur_get_params(xbg_sur* s, float* host) {
    if (!s || !host) return XBG_E_ARG;
    SHIP(s, hipStreamSynchronize(s->st));
    SHIP(s, hipMemcpy(host, s->P, s->nparam * 4, hipMemcpyDeviceToHost));
    return XBG_OK;
}

int xbg_sur_set_params(xbg_sur* s, const float* host) {
    if (!s || !host) return XBG_E_ARG;
    SHIP(s, hipStreamSynchronize(s->st));
    SHIP(s, hipMemcpy(s->P, host, s->nparam * 4, hipMemcpyHostToDevice));
    k_f32_to_bf16<<<nblk(s->nparam), 256, 0, s->st>>>(s->P, s->P16, s->nparam);
    SHIP(s, hipMemsetAsync(s->M, 0, s->nparam * 4, s->st));
    SHIP(s, hipMemsetAsync(s->V, 0, s->nparam * 4, s->st));
    s->adam_t = 0;
    SHIP(s, hipStreamSynchronize(s->st));
    return XBG_OK;
}

int xbg_sur_get_grads(xbg_sur* s, float* host) {
    if (!s || !host) return XBG_E_ARG;
    SHIP(s, hipStreamSynchronize(s->st));
    SHIP(s, hipMemcpy(host, s->G, s->nparam * 4, hipMemcpyDeviceToHost));
    return XBG_OK;
}

}  // extern "C"

namespace {

// the network's outputs into y (FP32 [n][H][W][5])
int sur_forward(xbg_sur* s, const bf16* x8, int n, float* y) {
    hipStream_t st = s->st;
    const int H = s->H, W = s->W;
    const ConvL& hd = s->L[17];
    auto Wt = [&](int l) { return s->P16 + s->L[l].w; };
    auto Bs = [&](int l) { return s->P + s->L[l].b; };
    int rc = 0;
    // convolution l of X on h x w pixels, through the epilogue E
#define CONV(l, EPI, RELU, X, h, w, ...)                                                                       \
    if ((rc = conv<EPI, RELU>(st, X, Wt(l), Bs(l), CEpi{__VA_ARGS__}, n, h, w, s->L[l].cin, \
                              s->L[l].cout, s->L[l].taps)))                                                    \
        return sfail(s, rc, "conv " #l);
    CONV(0, E_STORE, true, plain(x8, 8), H, W, s->e0a);
    CONV(1, E_POOL, true, plain(s->e0a, 32), H, W, s->e0, s->p1);
    CONV(2, E_STORE, true, plain(s->p1, 32), H / 2, W / 2, s->e1a);
    CONV(3, E_POOL, true, plain(s->e1a, 64), H / 2, W / 2, s->e1, s->p2);
    CONV(4, E_STORE, true, plain(s->p2, 64), H / 4, W / 4, s->e2a);
    CONV(5, E_POOL, true, plain(s->e2a, 128), H / 4, W / 4, s->e2, s->p3);
    CONV(6, E_STORE, true, plain(s->p3, 128), H / 8, W / 8, s->b3a);
    CONV(7, E_STORE, true, plain(s->b3a, 256), H / 8, W / 8, s->b3);
    CONV(8, E_STORE, false, plain(s->b3, 256), H / 8, W / 8, s->u2);
    CONV(9, E_STORE, true, concat(s->u2, s->e2, 128), H / 4, W / 4, s->d2a);
    CONV(10, E_STORE, true, plain(s->d2a, 128), H / 4, W / 4, s->d2);
    CONV(11, E_STORE, false, plain(s->d2, 128), H / 4, W / 4, s->u1);
    CONV(12, E_STORE, true, concat(s->u1, s->e1, 64), H / 2, W / 2, s->d1a);
    CONV(13, E_STORE, true, plain(s->d1a, 64), H / 2, W / 2, s->d1);
    CONV(14, E_STORE, false, plain(s->d1, 64), H / 2, W / 2, s->u0);
    CONV(15, E_STORE, true, concat(s->u0, s->e0, 32), H, W, s->d0a);
    CONV(16, E_HEAD, true, plain(s->d0a, 32), H, W, s->d0, nullptr, nullptr, nullptr, 0, s->P + hd.w, s->P + hd.b, y);
#undef CONV
    SHIP(s, hipGetLastError());
    return 0;
}

// one convolution's backward: from g, the gradient of its pre-activation
// output, dW, db and, unless EPI is -1, the data gradient through EPI
template <int EPI>
int conv_bwd(xbg_sur* s, int l, CSrc X, const bf16* g, const CEpi& E, int n, int H, int W) {
    hipStream_t st = s->st;
    const ConvL& c = s->L[l];
    int rc;
    if ((rc = conv_wgrad(st, X, g, s->G + c.w, s->G + c.b, s->part, s->npart, &s->upart, s->sums, n, H, W, c.cin, c.cout,
                         c.taps)))
        return sfail(s, rc, "wgrad " + std::to_string(l));
    if constexpr (EPI >= 0)
        if ((rc = conv<EPI, false>(st, plain(g, c.cout), s->Wd + c.w, nullptr, E, n, H, W, c.cout, c.cin, c.taps)))
            return sfail(s, rc, "dgrad " + std::to_string(l));
    return 0;
}

// the loss of s->y on its way to s->hloss and, with grad, its gradient into s->gy
int sur_loss_grad(xbg_sur* s, const bf16* t5, int n, int grad) {
    hipStream_t st = s->st;
    const size_t ne = (size_t)n * s->H * s->W * 5;
    const size_t want = (ne + 1023) / 1024;
    const int nb = want < MSE_PARTS ? (int)want : MSE_PARTS;
    k_mse<<<nb, 256, 0, st>>>(s->y, t5, ne, grad ? s->gy : nullptr, s->lossp);
    k_mean<<<1, 256, 0, st>>>(s->lossp, nb, (double)ne, s->lossp + MSE_PARTS);
    SHIP(s, hipMemcpyAsync(s->hloss, s->lossp + MSE_PARTS, sizeof(double), hipMemcpyDeviceToHost, st));
    SHIP(s, hipEventRecord(s->loss_done, st));
    return 0;
}

// waits for the loss (not for what was queued behind it)
int sur_loss_wait(xbg_sur* s, double* loss) {
    SHIP(s, hipEventSynchronize(s->loss_done));
    if (loss) *loss = *s->hloss;
    return 0;
}

int sur_backward(xbg_sur* s, const bf16* x8, int n) {
    hipStream_t st = s->st;
    const int H = s->H, W = s->W;
    const size_t P0 = (size_t)n * H * W;
    int rc;
    const ConvL& hd = s->L[17];
    {
        int nb = 1024;
        int ppb = (int)((P0 + nb - 1) / nb);
        nb = (int)((P0 + ppb - 1) / ppb);
        k_head_bwd<<<nb, 256, 0, st>>>(s->gy, s->P + hd.w, s->d0, s->g_d0, P0, ppb, s->part);
        s->sums.count = s->sums.blocks = 0;
        queue_sum(s->sums, s->part, nb, HK * HC + HK, HK * HC, s->G + hd.w, s->G + hd.b);
        s->upart = (size_t)nb * (HK * HC + HK);
        FlipJobs F{};
        for (int l = 1; l < 17; l++) queue_flip(F, s->L[l].w, s->L[l].taps, s->L[l].cout, s->L[l].cin);
        k_flip_weights<<<F.blocks, 256, 0, st>>>(s->P16, s->Wd, F);
    }
    // layer l: its input, the gradient of its output before the activation,
    // and where the gradient of its input goes (masked by the activation
    // that made the input, so that it is the next layer's g)
#define BWD(l, EPI, X, g, h, w, ...) \
    if ((rc = conv_bwd<EPI>(s, l, X, g, CEpi{__VA_ARGS__}, n, h, w))) return rc;
    BWD(16, E_STORE, plain(s->d0a, 32), s->g_d0, H, W, s->g_d0a, nullptr, s->d0a);
    // a concatenation's gradient: the coarse part's, and the skip's, to which
    // the pooled path adds below
    BWD(15, E_UPSUM, concat(s->u0, s->e0, 32), s->g_d0a, H, W, s->g_u0, s->g_e0, nullptr, nullptr, 32);
    BWD(14, E_STORE, plain(s->d1, 64), s->g_u0, H / 2, W / 2, s->g_d1, nullptr, s->d1);
    BWD(13, E_STORE, plain(s->d1a, 64), s->g_d1, H / 2, W / 2, s->g_d1a, nullptr, s->d1a);
    BWD(12, E_UPSUM, concat(s->u1, s->e1, 64), s->g_d1a, H / 2, W / 2, s->g_u1, s->g_e1, nullptr, nullptr, 64);
    BWD(11, E_STORE, plain(s->d2, 128), s->g_u1, H / 4, W / 4, s->g_d2, nullptr, s->d2);
    BWD(10, E_STORE, plain(s->d2a, 128), s->g_d2, H / 4, W / 4, s->g_d2a, nullptr, s->d2a);
    BWD(9, E_UPSUM, concat(s->u2, s->e2, 128), s->g_d2a, H / 4, W / 4, s->g_u2, s->g_e2, nullptr, nullptr, 128);
    BWD(8, E_STORE, plain(s->b3, 256), s->g_u2, H / 8, W / 8, s->g_b3, nullptr, s->b3);
    BWD(7, E_STORE, plain(s->b3a, 256), s->g_b3, H / 8, W / 8, s->g_b3a, nullptr, s->b3a);
    BWD(6, E_UNPOOL, plain(s->p3, 128), s->g_b3a, H / 8, W / 8, s->g_e2, nullptr, s->e2, s->g_e2);
    BWD(5, E_STORE, plain(s->e2a, 128), s->g_e2, H / 4, W / 4, s->g_e2a, nullptr, s->e2a);
    BWD(4, E_UNPOOL, plain(s->p2, 64), s->g_e2a, H / 4, W / 4, s->g_e1, nullptr, s->e1, s->g_e1);
    BWD(3, E_STORE, plain(s->e1a, 64), s->g_e1, H / 2, W / 2, s->g_e1a, nullptr, s->e1a);
    BWD(2, E_UNPOOL, plain(s->p1, 32), s->g_e1a, H / 2, W / 2, s->g_e0, nullptr, s->e0, s->g_e0);
    BWD(1, E_STORE, plain(s->e0a, 32), s->g_e0, H, W, s->g_e0a, nullptr, s->e0a);
    BWD(0, -1, plain(x8, 8), s->g_e0a, H, W, nullptr);
#undef BWD
    run_sums(st, s->sums);
    SHIP(s, hipGetLastError());
    return 0;
}

}  // namespace

extern "C" {

int xbg_sur_forward(xbg_sur* s, const void* x8, int n, float* y) {
    if (!s || !x8 || n < 1 || n > s->nmax) return sfail(s, XBG_E_ARG, "xbg_sur_forward: bad argument");
    int rc = sur_forward(s, (const bf16*)x8, n, y ? y : s->y);
    if (rc) return rc;
    SHIP(s, hipStreamSynchronize(s->st));
    return XBG_OK;
}

int xbg_sur_loss(xbg_sur* s, const void* x8, const void* t5, int n, double* loss) {
    if (!s || !x8 || !t5 || n < 1 || n > s->nmax) return sfail(s, XBG_E_ARG, "xbg_sur_loss: bad argument");
    int rc = sur_forward(s, (const bf16*)x8, n, s->y);
    if (!rc) rc = sur_loss_grad(s, (const bf16*)t5, n, 0);
    if (!rc) rc = sur_loss_wait(s, loss);
    return rc;
}

}  // extern "C"

namespace {
// Forward, loss and every parameter gradient, queued.  The caller may refill
// or free its batch once the loss is there, with the backward still running,
// whose last kernel (layer 0's weight gradient) reads the inputs: that takes
// a copy, made ahead of the loss.
int sur_gradients(xbg_sur* s, const void* x8, const void* t5, int n) {
    if (!s || !x8 || !t5 || n < 1 || n > s->nmax) return sfail(s, XBG_E_ARG, "xbg_sur_backward: bad argument");
    SHIP(s, hipMemcpyAsync(s->x8, x8, (size_t)n * s->H * s->W * 8 * sizeof(bf16), hipMemcpyDeviceToDevice, s->st));
    int rc = sur_forward(s, s->x8, n, s->y);
    if (!rc) rc = sur_loss_grad(s, (const bf16*)t5, n, 1);
    if (!rc) rc = sur_backward(s, s->x8, n);
    if (rc) hipStreamSynchronize(s->st);  // nothing queued reads the batch after an error either
    return rc;
}
}  // namespace

extern "C" {

int xbg_sur_backward(xbg_sur* s, const void* x8, const void* t5, int n, double* loss) {
    int rc = sur_gradients(s, x8, t5, n);
    if (!rc) SHIP(s, hipStreamSynchronize(s->st));
    if (!rc) rc = sur_loss_wait(s, loss);
    return rc;
}

// The update is queued before the loss is waited for: the device runs on
// while the host takes the loss.
int xbg_sur_train_step(xbg_sur* s, const void* x8, const void* t5, int n, double lr, double* loss) {
    int rc = sur_gradients(s, x8, t5, n);
    if (rc) return rc;
    s->adam_t++;
    const float b1 = 0.9f, b2 = 0.999f;
    const float bc1 = 1.0f - std::pow(b1, (float)s->adam_t), bc2 = 1.0f - std::pow(b2, (float)s->adam_t);
    k_adam<<<nblk(s->nparam), 256, 0, s->st>>>(s->P, s->P16, s->G, s->M, s->V, s->nparam, (float)lr, b1, b2, 1e-8f,
                                               bc1, bc2);
    SHIP(s, hipGetLastError());
    return sur_loss_wait(s, loss);
}

int xbg_sur_sync(xbg_sur* s) {
    if (!s) return XBG_E_ARG;
    SHIP(s, hipStreamSynchronize(s->st));
    return XBG_OK;
}

// Layer-level entry points on caller device buffers (tests, benchmarks).
int xbg_sur_conv_fwd(const void* X, const void* Wt, const float* bias, void* Y, int n, int H, int W, int Cin,
                     int Cout, int taps, int relu) {
    const CSrc src = plain((const bf16*)X, Cin);
    const CEpi out{(bf16*)Y};
    int rc = relu ? conv<E_STORE, true>(nullptr, src, (const bf16*)Wt, bias, out, n, H, W, Cin, Cout, taps)
                  : conv<E_STORE, false>(nullptr, src, (const bf16*)Wt, bias, out, n, H, W, Cin, Cout, taps);
    if (rc) return sfail(nullptr, rc, "xbg_sur_conv_fwd: unsupported shape");
    if (hipDeviceSynchronize() != hipSuccess) return sfail(nullptr, XBG_E_HIP, "xbg_sur_conv_fwd: run");
    return XBG_OK;
}

int xbg_sur_conv_dgrad(const void* dZ, const void* Wt, void* dX, int n, int H, int W, int Cin, int Cout, int taps) {
    bf16* Wd = nullptr;
    if (hipMalloc((void**)&Wd, (size_t)taps * Cin * Cout * 2) != hipSuccess) return XBG_E_HIP;
    FlipJobs F{};
    queue_flip(F, 0, taps, Cout, Cin);
    k_flip_weights<<<F.blocks, 256>>>((const bf16*)Wt, Wd, F);
    int rc = conv<E_STORE, false>(nullptr, plain((const bf16*)dZ, Cout), Wd, nullptr, CEpi{(bf16*)dX}, n, H, W, Cout, Cin, taps);
    hipError_t e = hipDeviceSynchronize();
    hipFree(Wd);
    if (rc) return sfail(nullptr, rc, "xbg_sur_conv_dgrad: unsupported shape");
    return e == hipSuccess ? XBG_OK : XBG_E_HIP;
}

int xbg_sur_conv_wgrad(const void* X, const void* dZ, float* dW, float* db, int n, int H, int W, int Cin, int Cout,
                       int taps) {
    // weights of up to 16 M values, with their bias sums
    const size_t np = ((size_t)16 << 20) + (Cout > 0 ? Cout : 0);
    float* part = nullptr;
    if (hipMalloc((void**)&part, np * 4) != hipSuccess) return XBG_E_HIP;
    SumJobs J{};
    size_t used = 0;
    int rc = conv_wgrad(nullptr, plain((const bf16*)X, Cin), (const bf16*)dZ, dW, db, part, np, &used, J, n, H, W, Cin, Cout, taps);
    run_sums(nullptr, J);
    hipError_t e = hipDeviceSynchronize();
    hipFree(part);
    if (rc) return sfail(nullptr, rc, "xbg_sur_conv_wgrad: unsupported shape");
    return e == hipSuccess ? XBG_OK : XBG_E_HIP;
}

}  // extern "C"

namespace {

struct InNorm {
    float mean[7], std[7];  // zb, zs, uu, vv, Hm0, Tp, dir
};

// Surrogate inputs of one domain: x8[i] = the normalised zb, zs, uu, vv of
// cell i and the offshore Hm0, Tp, mean direction, then a zero.
__global__ __launch_bounds__(256) void k_pack_inputs(const float* __restrict__ zb, const float* __restrict__ zs,
                                                     const float* __restrict__ uu, const float* __restrict__ vv,
                                                     size_t n, float Hm0, float Tp, float dir, InNorm nm,
                                                     bf16* __restrict__ x8) {
    size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const float v[7] = {zb[i], zs[i], uu[i], vv[i], Hm0, Tp, dir};
    bf16x8 o;
#pragma unroll
    for (int k = 0; k < 7; k++) o[k] = to_bf16((v[k] - nm.mean[k]) / nm.std[k]);
    o[7] = to_bf16(0.0f);
    *(bf16x8*)(x8 + i * 8) = o;
}

}  // namespace

extern "C" int xbg_sur_pack_inputs(const float* zb, const float* zs, const float* uu, const float* vv, size_t n,
                                   double Hm0, double Tp, double dir, const float* norm14, void* x8, void* stream) {
    if (!zb || !zs || !uu || !vv || !norm14 || !x8) return sfail(nullptr, XBG_E_ARG, "xbg_sur_pack_inputs: NULL");
    InNorm nm;
    for (int k = 0; k < 7; k++) {
        nm.mean[k] = norm14[k];
        nm.std[k] = norm14[7 + k];
    }
    // on the stream that produced the fields (a domain's stream is
    // non-blocking: the null stream would not wait for its window means)
    hipStream_t st = (hipStream_t)stream;
    k_pack_inputs<<<nblk(n), 256, 0, st>>>(zb, zs, uu, vv, n, (float)Hm0, (float)Tp, (float)dir, nm, (bf16*)x8);
    if (hipGetLastError() != hipSuccess || hipStreamSynchronize(st) != hipSuccess)
        return sfail(nullptr, XBG_E_HIP, "xbg_sur_pack_inputs: run");
    return XBG_OK;
}
