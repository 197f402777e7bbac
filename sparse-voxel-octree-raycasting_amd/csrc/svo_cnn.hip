// svo_cnn.hip -- learned hole filler: a 4-layer 3x3 CNN with hand-written
// BF16 MFMA forward / backward kernels (FP32 accumulate) and Adam, trained on
// (warped frame, full raycast) pairs the pipeline produces itself.  No
// counterpart in the reference (it only has the fixed filter of
// kernel.cl:404-470); the plain warp path is unchanged by this file.
//
// Network: conv3x3 5->32, ReLU, 32->32, ReLU, 32->32, ReLU, 32->3 (linear),
// zero "same" padding at crop borders.  Channels are padded to multiples of
// 16 (input 5 -> 16, output 3 -> 16); padded weights stay zero.
// Input features per pixel of the pre-filter warped frame: RGB of the
// colorized screen word (0 at holes), depth z/(z+64) (0 at holes), hole mask.
//
// Tensors are NHWC bf16 over a batch of crops.  One wave computes an 8x8
// output tile: 4 M-tiles of 16 pixels x (COUT/16) N-tiles with
// v_mfma_f32_16x16x16_bf16 (A = 16 pixels x 16 input channels from LDS,
// B = 16 input x 16 output channels from the weights, K = 9 taps x CIN).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "svo_ctx.h"
#include "svo_internal.h"

namespace {

typedef short s4v __attribute__((ext_vector_type(4)));
typedef float f4v __attribute__((ext_vector_type(4)));
typedef uint16_t bf16;

__device__ __forceinline__ bf16 f2bf(float f)
{
    uint32_t u = __float_as_uint(f);
    u += 0x7fffu + ((u >> 16) & 1u);  // round to nearest even
    return (bf16)(u >> 16);
}
__device__ __forceinline__ float bf2f(bf16 h) { return __uint_as_float((uint32_t)h << 16); }
constexpr uint32_t HOLE_WORD = 0xffffff00u;
// The four layers' channels, and the flat parameter vector: per layer W
// [9][cout][cin] then b [cout].  kWofs counts weights only (the bf16 copies).
constexpr int kCin[4] = {16, 32, 32, 32}, kCout[4] = {32, 32, 32, 16};
constexpr int kWofs[5] = {0, 4608, 13824, 23040, 27648};
constexpr int kPofs[5] = {0, 4640, 13888, 23136, 27760};
constexpr int kParams = kPofs[4];
// the layer that holds index i of one of these tables
__device__ __forceinline__ int layer_of(const int (&ofs)[5], int i)
{
    return (i >= ofs[1]) + (i >= ofs[2]) + (i >= ofs[3]);
}
constexpr int TILE = 8;          // output tile edge per wave
constexpr int HALO = TILE + 2;   // input tile edge

// MODE 0: + bias, ReLU, bf16 out.  MODE 1: + bias, fp32 out (last layer).
// MODE 2: no bias, multiplied by (mask_src > 0), bf16 out (backward data).
// At training sizes a SIMD has one wave, so latency bounds it: the halo's
// loads go out together, the masks of the backward before the products, and
// the taps are unrolled so that the weights are read ahead.  16 crops of
// 64x64, 32 -> 32 channels: forward 10.8 -> 7.8 us, backward 16.5 -> 8.8.
// Work items (crop, 8x8 tile) are taken grid-stride; the crop count is B, or
// min(*bcount, B) when bcount is given (batches sized on the device).
template <int CIN, int COUT, int MODE>
__global__ __launch_bounds__(64) void k_conv(const bf16* __restrict__ X, const bf16* __restrict__ Wt,
                                             const float* __restrict__ bias, const bf16* __restrict__ mask_src,
                                             void* Yout, int H, int W, int B, const uint32_t* bcount)
{
    constexpr int CS = CIN + 4;  // LDS pixel stride (bank spread)
    __shared__ __align__(16) bf16 xs[HALO * HALO * CS];
    const int lane = threadIdx.x;
    const int tiles_x = W / TILE, tiles_y = H / TILE;
    const int nb = bcount ? min((int)*bcount, B) : B;
    for (int item = blockIdx.x; item < nb * tiles_x * tiles_y; item += gridDim.x) {
    const int b = item / (tiles_x * tiles_y);
    const int t = item % (tiles_x * tiles_y);
    const int y0 = (t / tiles_x) * TILE, x0 = (t % tiles_x) * TILE;
    __syncthreads();  // previous item's LDS reads are done
    // stage the (TILE+2)^2 x CIN input halo, zero outside the crop
    constexpr int UNITS = HALO * HALO * (CIN / 4), LOADS = (UNITS + 63) / 64;
    uint2 v[LOADS];
#pragma unroll
    for (int k = 0; k < LOADS; k++) {
        const int i = lane + 64 * k, pix = i / (CIN / 4), c4 = (i % (CIN / 4)) * 4;
        const int yy = y0 + pix / HALO - 1, xx = x0 + pix % HALO - 1;
        v[k] = make_uint2(0u, 0u);
        if (i < UNITS && yy >= 0 && yy < H && xx >= 0 && xx < W)
            v[k] = *(const uint2*)(X + (((size_t)b * H + yy) * W + xx) * CIN + c4);
    }
#pragma unroll
    for (int k = 0; k < LOADS; k++) {
        const int i = lane + 64 * k;
        if (i < UNITS) *(uint2*)(xs + i / (CIN / 4) * CS + (i % (CIN / 4)) * 4) = v[k];
    }
    constexpr int NT = COUT / 16;
    const int row = lane & 15, kq = (lane >> 4) * 4;
    // backward: the ReLU masks are read ahead of the products
    bf16 keep[4][NT][4];
    if (MODE == 2)
        for (int m = 0; m < 4; m++)
            for (int n = 0; n < NT; n++)
                for (int i = 0; i < 4; i++) {
                    const int p = m * 16 + kq + i, py = p / TILE, px = p % TILE;
                    keep[m][n][i] = mask_src[(((size_t)b * H + y0 + py) * W + x0 + px) * COUT + n * 16 + row];
                }
    __syncthreads();

    f4v acc[4][NT];
    for (int m = 0; m < 4; m++)
        for (int n = 0; n < NT; n++) acc[m][n] = f4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int tap = 0; tap < 9; tap++) {
        const int dy = tap / 3, dx = tap % 3;
        for (int kc = 0; kc < CIN / 16; kc++) {
            s4v bfr[NT];
            for (int n = 0; n < NT; n++)
                bfr[n] = *(const s4v*)(Wt + ((size_t)tap * COUT + n * 16 + row) * CIN + kc * 16 + kq);
            for (int m = 0; m < 4; m++) {
                const int p = m * 16 + row, py = p / TILE, px = p % TILE;
                const s4v afr = *(const s4v*)(xs + ((py + dy) * HALO + px + dx) * CS + kc * 16 + kq);
                for (int n = 0; n < NT; n++)
                    acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(afr, bfr[n], acc[m][n], 0, 0, 0);
            }
        }
    }
    // D layout: lane holds pixels 4*(lane/16)+i of the M-tile, channel lane%16
    for (int m = 0; m < 4; m++)
        for (int n = 0; n < NT; n++) {
            const int co = n * 16 + row;
            for (int i = 0; i < 4; i++) {
                const int p = m * 16 + kq + i, py = p / TILE, px = p % TILE;
                const size_t o = (((size_t)b * H + y0 + py) * W + x0 + px) * COUT + co;
                float v = acc[m][n][i];
                if (MODE == 0) {
                    v += bias[co];
                    v = v > 0.f ? v : 0.f;
                    ((bf16*)Yout)[o] = f2bf(v);
                } else if (MODE == 1) {
                    ((float*)Yout)[o] = v + bias[co];
                } else {
                    // ReLU derivative: the forward output (>= 0) is positive
                    ((bf16*)Yout)[o] = keep[m][n][i] != 0 ? f2bf(v) : (bf16)0;
                }
            }
        }
    }
}

// The gradients of layers lo .. lo + gridDim.z - 1 in one launch (dz of every
// layer is kept): a layer by itself has 9 workgroups per crop, which leaves
// most CUs idle at the usual 16 to 32 crops.
struct GradArgs {
    const bf16* x[4];   // a layer's input
    const bf16* dz[4];  // the gradient of its output before the ReLU
    float* part_w;      // per layer [B][9][cout][cin], from layer lo on
    float* part_b;      // per layer [db blocks][32]
    float* grads;       // flat, as the parameters
    int B, H, W, lo, db_blocks;
};

// dW partials of crop b: sum over the crop's pixels p of dZ[p][co] X[p + tap
// - 1][ci].  grid = (crops, 3 tap rows, layers), DW_SLICES waves per
// workgroup: wave s loops over pixel slice s (a multiple of 16 pixels), K = 16
// pixels per MFMA (A = dZ^T: co x pixels, B = shifted X: pixels x ci); the
// waves' sums are added in slice order through LDS and written to
// part[b][tap][co][ci]; k_sum_grads adds the crops' partials in crop order, so
// the gradient does not depend on scheduling.
// Both operands are read transposed, two bytes at a time, so the loads and
// their addresses bound it.  A row's three taps share them: 8 for dZ and, as
// the taps' four pixels overlap, 12 for X instead of 48 (all 32 channels).
// 16 crops of 64x64, all layers: 98 us with a launch per layer and a tap per
// workgroup, 70 so in one launch, 20 with the three taps.
constexpr int DW_SLICES = 16;
template <int CIN, int COUT>
__device__ __forceinline__ void conv_dw(const bf16* __restrict__ X, const bf16* __restrict__ dZ,
                                        float* __restrict__ part, int H, int W, float* s_acc)
{
    const int b = blockIdx.x, dy = (int)blockIdx.y - 1, sl = threadIdx.x >> 6;
    const int lane = threadIdx.x & 63, row = lane & 15, kq = (lane >> 4) * 4;
    constexpr int MT = COUT / 16, NT = CIN / 16;
    f4v acc[3][MT][NT];
    for (int t = 0; t < 3; t++)
        for (int m = 0; m < MT; m++)
            for (int n = 0; n < NT; n++) acc[t][m][n] = f4v{0.f, 0.f, 0.f, 0.f};
    const int npix = H * W;  // a multiple of 16
    const int len = (npix / 16 + DW_SLICES - 1) / DW_SLICES * 16;
    const int kb = min(npix, sl * len), ke = min(npix, kb + len);
    const bf16* dz = dZ + (size_t)b * npix * COUT + row;
    const bf16* xb = X + (size_t)b * npix * CIN + row;
    constexpr int U = 2;  // steps whose loads are issued together
    for (int k0 = kb; k0 < ke; k0 += 16 * U) {
        s4v afr[U][MT], bfr[U][3][NT];
#pragma unroll
        for (int u = 0; u < U; u++) {
            // past the slice: the last step's addresses again, and zeros
            const bool in = k0 + 16 * u < ke;
            const int p = min(k0 + 16 * u, ke - 16) + kq;
            const bf16* za = dz + (size_t)p * COUT;
            for (int m = 0; m < MT; m++) {
                s4v v;
                for (int j = 0; j < 4; j++) v[j] = (short)za[j * COUT + m * 16];
                afr[u][m] = in ? v : s4v{0, 0, 0, 0};
            }
            // p is a multiple of 4 and W of 8: the four pixels share a row,
            // and only the pixel before and the one after can be outside it
            const int y = p / W + dy, x = p % W;
            const bool in_y = in && y >= 0 && y < H, in_l = in_y && x > 0, in_r = in_y && x + 4 < W;
            const bf16* xa = xb + (size_t)(min(max(y, 0), H - 1) * W + x) * CIN;
            const bf16* xl = xa - (x > 0 ? CIN : 0);
            const bf16* xr = xa + (x + 4 < W ? 4 : 3) * CIN;
            for (int n = 0; n < NT; n++) {
                short v[6];
                v[0] = (short)xl[n * 16];
                for (int j = 0; j < 4; j++) v[j + 1] = (short)xa[j * CIN + n * 16];
                v[5] = (short)xr[n * 16];
                v[0] = in_l ? v[0] : (short)0;
                for (int j = 1; j < 5; j++) v[j] = in_y ? v[j] : (short)0;
                v[5] = in_r ? v[5] : (short)0;
                for (int t = 0; t < 3; t++) bfr[u][t][n] = s4v{v[t], v[t + 1], v[t + 2], v[t + 3]};
            }
        }
#pragma unroll
        for (int u = 0; u < U; u++)
            for (int t = 0; t < 3; t++)
                for (int m = 0; m < MT; m++)
                    for (int n = 0; n < NT; n++)
                        acc[t][m][n] =
                            __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(afr[u][m], bfr[u][t][n], acc[t][m][n], 0, 0, 0);
    }
    for (int t = 0; t < 3; t++) {
        if (t) __syncthreads();  // the tap before has been read
        for (int m = 0; m < MT; m++)
            for (int n = 0; n < NT; n++)
                for (int i = 0; i < 4; i++) {
                    const int co = m * 16 + kq + i, ci = n * 16 + row;
                    s_acc[sl * COUT * CIN + co * CIN + ci] = acc[t][m][n][i];
                }
        __syncthreads();
        float* dw = part + ((size_t)b * 9 + blockIdx.y * 3 + t) * COUT * CIN;
        for (int e = threadIdx.x; e < COUT * CIN; e += 64 * DW_SLICES) {
            float v = 0.f;
            for (int k = 0; k < DW_SLICES; k++) v += s_acc[k * COUT * CIN + e];
            dw[e] = v;
        }
    }
}

__global__ __launch_bounds__(64 * DW_SLICES) void k_conv_dw(GradArgs a)
{
    __shared__ float s_acc[DW_SLICES * 32 * 32];
    const int l = a.lo + (int)blockIdx.z;
    float* part = a.part_w + (size_t)a.B * (kWofs[l] - kWofs[a.lo]);
    if (l == 0) conv_dw<16, 32>(a.x[0], a.dz[0], part, a.H, a.W, s_acc);
    else if (l == 3) conv_dw<32, 16>(a.x[3], a.dz[3], part, a.H, a.W, s_acc);
    else conv_dw<32, 32>(a.x[l], a.dz[l], part, a.H, a.W, s_acc);
}

// db partial of block b: part[b][co] = sum over its DB_PIXELS pixels of
// dZ[p][co] (each thread a fixed stride of pixels, then the threads of a
// channel in order)
constexpr int DB_PIXELS = 256;
template <int COUT>
__device__ __forceinline__ void conv_db(const bf16* __restrict__ dZ, float* __restrict__ part, int npix, float* s_sum)
{
    const int co = threadIdx.x % COUT, lane_p = threadIdx.x / COUT;
    const int p0 = blockIdx.x * DB_PIXELS, p1 = min(p0 + DB_PIXELS, npix);
    float s = 0.f;
#pragma unroll 8
    for (int p = p0 + lane_p; p < p1; p += 256 / COUT) s += bf2f(dZ[(size_t)p * COUT + co]);
    s_sum[threadIdx.x] = s;
    __syncthreads();
    if (threadIdx.x < COUT) {
        float t = 0.f;
        for (int j = 0; j < 256 / COUT; j++) t += s_sum[j * COUT + threadIdx.x];
        part[(size_t)blockIdx.x * COUT + threadIdx.x] = t;
    }
}
__global__ __launch_bounds__(256) void k_conv_db(GradArgs a)
{
    __shared__ float s_sum[256];
    const int l = a.lo + (int)blockIdx.y;
    float* part = a.part_b + (size_t)a.db_blocks * 32 * blockIdx.y;
    const int npix = a.B * a.H * a.W;
    if (l == 3) conv_db<16>(a.dz[3], part, npix, s_sum);
    else conv_db<32>(a.dz[l], part, npix, s_sum);
}

// The partials added up, layers lo .. hi - 1.  The first workgroups take 256
// weights each (a layer's are a multiple of 256): one thread per weight adds
// the crops in order.  The others take one bias each: thread t adds partials
// t, t + 256, ... in order, then a fixed pairwise tree over the 256 threads.
__global__ __launch_bounds__(256) void k_sum_grads(GradArgs a, int hi)
{
    const int wblocks = (kWofs[hi] - kWofs[a.lo]) / 256;
    const int t = threadIdx.x;
    if ((int)blockIdx.x < wblocks) {
        const int i = kWofs[a.lo] + (int)blockIdx.x * 256 + t;
        const int l = layer_of(kWofs, i), n = kWofs[l + 1] - kWofs[l], e = i - kWofs[l];
        const float* part = a.part_w + (size_t)a.B * (kWofs[l] - kWofs[a.lo]) + e;
        float s = 0.f;
#pragma unroll 8
        for (int p = 0; p < a.B; p++) s += part[(size_t)p * n];
        a.grads[kPofs[l] + e] = s;
        return;
    }
    __shared__ float s[256];
    const int bi = (int)blockIdx.x - wblocks, l = a.lo + bi / 32, e = bi % 32;  // (layer 3 has 16 biases)
    const int n = kCout[l];
    const float* part = a.part_b + (size_t)a.db_blocks * 32 * (l - a.lo) + e;
    float v = 0.f;
    for (int p = t; p < a.db_blocks; p += 256) v += part[(size_t)p * n];
    s[t] = v;
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
        if (t < h) s[t] += s[t + h];
        __syncthreads();
    }
    if (t == 0) a.grads[kPofs[l + 1] - n + e] = s[0];
}

// *sum += v of every thread of a workgroup of 256, one atomic (16 ns each on
// the same word: one per thread or per wave took 16 us at 65,536 pixels)
__device__ __forceinline__ void add_once(float v, float* sum)
{
    __shared__ float s[4];
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    if (__lane_id() == 0) s[threadIdx.x >> 6] = v;
    __syncthreads();
    v = (s[0] + s[1]) + (s[2] + s[3]);
    if (threadIdx.x == 0 && v != 0.f) atomicAdd(sum, v);
}

// masked MSE on RGB: loss += sum mask*(pred-t)^2 / (3*count); dZ = d loss/d pred
__global__ __launch_bounds__(256) void k_loss(const float* __restrict__ pred, const float* __restrict__ target,
                                              const float* __restrict__ mask, bf16* dZ, float* loss, int npix,
                                              const float* __restrict__ mask_count)
{
    const float inv_count = *mask_count > 0.f ? 1.f / (3.f * *mask_count) : 0.f;
    float l = 0.f;
    for (int p = blockIdx.x * 256 + threadIdx.x; p < npix; p += gridDim.x * 256) {
        uint32_t g[3];
        float lp = 0.f;
        for (int c = 0; c < 3; c++) {
            const float d = pred[(size_t)p * 16 + c] - target[(size_t)p * 3 + c];
            lp += mask[p] * d * d;
            g[c] = f2bf(2.f * mask[p] * d * inv_count);
        }
        l += lp * inv_count;
        uint4* z = (uint4*)(dZ + (size_t)p * 16);
        z[0] = make_uint4(g[0] | (g[1] << 16), g[2], 0u, 0u);
        z[1] = make_uint4(0u, 0u, 0u, 0u);
    }
    add_once(l, loss);
}

// Input features of crop c (origin from `origins`, or tile list -> tile*16-4):
// RGB of the colorized word of the CNN input planes (plane 0 as the gate of a
// learned frame leaves it), camera depth z/(z+64) and the hole mask; zero
// outside the screen and at holes.  With `image`, also the target RGB (full
// raycast) and the loss mask (pixels that are holes in `mask_words`, else in
// the input, inside the screen), counting mask pixels into *mask_count.
__device__ __forceinline__ void rgb_of(uint32_t word, float& r, float& g, float& b)
{
    const int a = (int)word, c = a & 3;
    const float i = (float)(a & (255 - 7));
    float tr = 1.0f, tg = 1.0f, tb = 1.0f;
    if (c == 1) { tg = 0.7f; tb = 0.3f; }
    else if (c == 2) { tr = 1.5f; tg = 0.8f; tb = 0.1f; }
    else if (c == 3) { tr = 0.2f; tg = 0.8f; tb = 0.2f; }
    r = fminf((float)(int)(i * tr), 255.f) * (1.f / 255.f);
    g = fminf((float)(int)(i * tg), 255.f) * (1.f / 255.f);
    b = fminf((float)(int)(i * tb), 255.f) * (1.f / 255.f);
}

struct FeatArgs {
    const uint32_t* words;   // screen words of the CNN input (hole channel)
    const float4* coords;    // coords of the CNN input
    const uint32_t* mask_words;  // training: the loss covers pixels that are holes here (else `words`)
    const uint32_t* image;   // full-raycast image (targets) or null
    int res_x, res_y, crop;
    const int2* origins;     // explicit crop origins, or null
    const uint32_t* tiles;   // tile list (origin = tile*16 - 4), or null
    int tiles_x;
    const uint32_t* count;   // device crop count (tile list), or null
    int max_crops;
    float m0x, m0y, m0z, r20, r21, r22;
    bf16* x;
    float* target;
    float* mask;
    float* mask_count;
};

__global__ __launch_bounds__(256) void k_features(FeatArgs a)
{
    const int nb = a.count ? min((int)*a.count, a.max_crops) : a.max_crops;
    const size_t per = (size_t)a.crop * a.crop;
    float cnt = 0.f;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < (size_t)nb * per; i += (size_t)gridDim.x * 256) {
        const int c = (int)(i / per), q = (int)(i % per);
        int ox, oy;
        if (a.origins) {
            ox = a.origins[c].x;
            oy = a.origins[c].y;
        } else {
            const int t = (int)a.tiles[c];
            ox = (t % a.tiles_x) * 16 - 4;
            oy = (t / a.tiles_x) * 16 - 4;
        }
        const int x = ox + q % a.crop, y = oy + q / a.crop;
        float f[5] = {0.f, 0.f, 0.f, 0.f, 0.f};
        float tr = 0.f, tg = 0.f, tb = 0.f, m = 0.f;
        if (x >= 0 && y >= 0 && x < a.res_x && y < a.res_y) {
            const size_t o = (size_t)y * a.res_x + x;
            const uint32_t w = a.words[o];
            m = (a.mask_words ? a.mask_words[o] : w) == HOLE_WORD ? 1.f : 0.f;
            if (w == HOLE_WORD) {
                f[4] = 1.f;
            } else {
                rgb_of(w, f[0], f[1], f[2]);
                const float4 cc = a.coords[o];
                const float qx = cc.x - a.m0x, qy = cc.y - a.m0y, qz = cc.z - a.m0z;
                const float z = fmaxf((qx * a.r20 + qy * a.r21) + qz * a.r22, 0.f);
                f[3] = z / (z + 64.f);
            }
            if (a.image) {
                const uint32_t px = a.image[o];
                tr = (float)((px >> 16) & 255u) * (1.f / 255.f);
                tg = (float)((px >> 8) & 255u) * (1.f / 255.f);
                tb = (float)(px & 255u) * (1.f / 255.f);
            }
        }
        uint4* xo = (uint4*)(a.x + i * 16);
        xo[0] = make_uint4(f2bf(f[0]) | ((uint32_t)f2bf(f[1]) << 16), f2bf(f[2]) | ((uint32_t)f2bf(f[3]) << 16),
                           f2bf(f[4]), 0u);
        xo[1] = make_uint4(0u, 0u, 0u, 0u);
        if (a.target) {
            a.target[i * 3 + 0] = tr;
            a.target[i * 3 + 1] = tg;
            a.target[i * 3 + 2] = tb;
            a.mask[i] = m;
            cnt += m;
        }
    }
    if (!a.target) return;
    add_once(cnt, a.mask_count);
}

__device__ __forceinline__ uint32_t rgb_word(float r, float g, float b)
{
    const uint32_t R = (uint32_t)fminf(fmaxf(r * 255.f + 0.5f, 0.f), 255.f);
    const uint32_t G = (uint32_t)fminf(fmaxf(g * 255.f + 0.5f, 0.f), 255.f);
    const uint32_t B = (uint32_t)fminf(fmaxf(b * 255.f + 0.5f, 0.f), 255.f);
    return B | (G << 8) | (R << 16);
}

// CNN RGB of the centre 16x16 of each tile crop -> 256 colorized words per tile
__global__ __launch_bounds__(256) void k_stage_fill(const float* __restrict__ out, const uint32_t* __restrict__ count,
                                                    int max_crops, uint32_t* __restrict__ staged)
{
    const int nb = min((int)*count, max_crops);
    for (int i = blockIdx.x * 256 + threadIdx.x; i < nb * 256; i += gridDim.x * 256) {
        const int c = i / 256, q = i % 256;
        const float* v = out + ((size_t)c * 576 + (size_t)((q >> 4) + 4) * 24 + (q & 15) + 4) * 16;
        staged[i] = rgb_word(v[0], v[1], v[2]);
    }
}

// staged CNN colours -> image at the tile pixels that are still holes in
// `words` (plane 2: the frame after its rays, before the filter)
__global__ __launch_bounds__(256) void k_cnn_apply(const uint32_t* __restrict__ staged,
                                                   const uint32_t* __restrict__ tiles,
                                                   const uint32_t* __restrict__ count, int max_crops,
                                                   const uint32_t* __restrict__ words, uint32_t* image, int res_x,
                                                   int res_y, int tiles_x)
{
    const int nb = min((int)*count, max_crops);
    for (int i = blockIdx.x * 256 + threadIdx.x; i < nb * 256; i += gridDim.x * 256) {
        const int c = i / 256, q = i % 256;
        const int t = (int)tiles[c];
        const int x = (t % tiles_x) * 16 + (q & 15), y = (t / tiles_x) * 16 + (q >> 4);
        if (x >= res_x || y >= res_y) continue;
        const size_t o = (size_t)y * res_x + x;
        if (words[o] == HOLE_WORD) image[o] = staged[i];
    }
}

// ---------------------------------------------------------------- fused tile inference
// One workgroup (4 waves) runs the whole network on one 24x24 crop around a
// 16x16 gate tile, activations in LDS.  Each layer is evaluated only where
// the centre 16x16 output needs it: layer 1 on 22x22, layer 2 on 20x20,
// layer 3 on 18x18, layer 4 on 16x16 (the crop border's zero padding never
// reaches the centre, so this equals the full-crop network there).  Layer 1
// uses v_mfma_f32_16x16x16_bf16 over K = 16 channels per tap, layers 2-4
// v_mfma_f32_16x16x32_bf16 over K = 32 (lane: pixel or output channel l%16,
// input channels 8*(l/16)..+7).
//
// Three resources bound a tile: the matrix cores (1,584 MFMAs of 16 cycles
// over 4 SIMDs), the LDS reads of the pixel fragments, and the vector
// instructions around them (addresses, bias, ReLU, bf16).  An M-tile per 16
// consecutive pixels reads nine fragments per pair of output channel groups
// and computes nine swizzled addresses.  Here a wave sweeps a band of rows of
// the leftmost 16 columns: each input row's three fragments (dx = 0..2) feed
// the three output rows they belong to, so a row costs three reads instead of
// nine, from three addresses per layer with the row as the instruction's
// offset.  The remaining columns (6, 4 and 2 of layers 1-3) are M-tiles of 16
// pixels each, a wave's M-tiles of a layer computed together.  Every output
// adds its taps 0..8 in that order.  A wave computes 16 of the hidden layers'
// 32 output channels, so layers 1-3's weights stay in its registers for the
// whole launch (layer 4's come from the L2 behind layer 3), a tile has four
// barriers, and the next tile's crop is on its way from memory during layers
// 3 and 4.  6,250 tiles of a 1920x1024 learned frame, stage time with nothing
// beside it on one device: 276.5 us with nine reads per M-tile and each
// layer's weights staged in LDS, 203 with the sweep and the resident weights,
// 178 with the next row's fragments read behind a row's first MFMAs, 169 with
// layer 4's RGB stored from its registers and the crop fetched ahead.  The
// matrix cores are then busy in 42 % of the cycles (counters); two waves per
// SIMD (LDS and registers both allow no more) leave each other's stalls
// uncovered.
typedef __bf16 bf8v __attribute__((ext_vector_type(8)));

// 32-channel buffers: rows of TILE_PITCH pixels of 64 bytes; the 16-byte
// channel group g of column x sits in slot g ^ ((x >> 1) & 3).  A 128-bit LDS
// read is served 8 lanes at a time from 128 bytes of banks: 8 consecutive
// columns of one group then land on 8 distinct 16-byte slots (column parity x
// slot).  The slot depends on the column alone, so a row further down is a
// constant offset; the odd pitch shifts the next row by half of the banks,
// which spreads M-tiles of several short rows.
constexpr int TILE_PITCH = 25;
__device__ __forceinline__ int at32(int y, int x, int g)
{
    return (y * TILE_PITCH + x) * 32 + ((g ^ ((x >> 1) & 3)) << 3);
}
// the 24x24 input, 16-channel pixels: the 8-byte group k (4 channels) of
// column x sits in slot k ^ ((x >> 2) & 3); a 64-bit read is served 16 lanes
// at a time from 128 bytes, and 16 consecutive columns (32-byte stride) of
// one group then cover 16 distinct 8-byte slots
__device__ __forceinline__ int at16(int y, int x, int k)
{
    return (y * 24 + x) * 16 + ((k ^ ((x >> 2) & 3)) << 2);
}

// One view's CNN tiles in frame mode: features of the crop at tile*16 - 4
// from the view's CNN input planes, 256 colorized words per tile to `staged`;
// the apply step writes them into `image` where plane 2 still holds holes.
struct TileView {
    const uint32_t* words;
    const float4* coords;
    int res_x, res_y, tiles_x;
    const uint32_t* tiles;
    const uint32_t* count;
    int max_tiles;
    float m0x, m0y, m0z, r20, r21, r22;
    uint32_t* staged;
    const uint32_t* plane2;
    uint32_t* image;
};

struct TileArgs {
    // frame mode (x == null): one view, or a device table of n_views views
    // whose tile lists are concatenated (first[i] = the first tile of view i,
    // first[n_views] = all tiles)
    TileView v;
    const TileView* views;
    const uint32_t* first;
    int n_views;
    // explicit mode: x [n][24][24][16] bf16 -> out [n][16][16][3] float
    const bf16* x;
    float* out;
    int n;
    const bf16* w[4];  // [9][32][16], [9][32][32], [9][32][32], [9][16][32]
    const float* b[4];
};

// first tile of each batched view (after their gates), one thread
__global__ void k_tile_first(const TileView* views, int n, uint32_t* first)
{
    uint32_t acc = 0;
    for (int i = 0; i < n; i++) {
        first[i] = acc;
        acc += (uint32_t)min((int)*views[i].count, views[i].max_tiles);
    }
    first[n] = acc;
}

// k_cnn_apply for every view of a batch (grid y = view)
__global__ __launch_bounds__(256) void k_cnn_apply_views(const TileView* views)
{
    const TileView& V = views[blockIdx.y];
    const int nb = min((int)*V.count, V.max_tiles);
    for (int i = blockIdx.x * 256 + threadIdx.x; i < nb * 256; i += gridDim.x * 256) {
        const int c = i / 256, q = i % 256;
        const int t = (int)V.tiles[c];
        const int x = (t % V.tiles_x) * 16 + (q & 15), y = (t / V.tiles_x) * 16 + (q >> 4);
        if (x >= V.res_x || y >= V.res_y) continue;
        const size_t o = (size_t)y * V.res_x + x;
        if (V.plane2[o] == HOLE_WORD) V.image[o] = V.staged[i];
    }
}

// All tile layers compute the transposed product D[channel][pixel] (the
// weights are the MFMA's A operand, the pixels its B operand), so a lane ends
// with four consecutive output channels of one pixel and stores them as one
// 8-byte write.

// relu(acc + bias) of four channels as four bf16 (round to nearest even, as f2bf)
typedef float f2v __attribute__((ext_vector_type(2)));
typedef __bf16 bf2v __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint2 relu_pack(f4v acc, f4v bias)
{
    f4v v = acc + bias;
    for (int i = 0; i < 4; i++) v[i] = fmaxf(v[i], 0.f);
    union {
        bf2v h[2];
        uint2 u;
    } o;
    o.h[0] = __builtin_convertvector(f2v{v[0], v[1]}, bf2v);
    o.h[1] = __builtin_convertvector(f2v{v[2], v[3]}, bf2v);
    return o.u;
}

// one layer's weights and biases of a wave's 16 output channels: fragment
// [tap] = this lane's output channel and input channels; bias of the 4
// channels it ends with
template <typename Frag>
struct TileWeights {
    Frag w[9];
    f4v b;
    // W: [9][cout][cin], the channels from co0 on
    __device__ __forceinline__ void load(const bf16* __restrict__ W, const float* __restrict__ bias, int cout, int cin,
                                         int co0, int row, int kg)
    {
#pragma unroll
        for (int t = 0; t < 9; t++)
            w[t] = *(const Frag*)(W + (t * cout + co0 + row) * cin + kg * (int)(sizeof(Frag) / 2));
        b = *(const f4v*)(bias + co0 + kg * 4);
    }
};

__device__ __forceinline__ f4v tile_mfma(s4v w, s4v x, f4v acc)
{
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(w, x, acc, 0, 0, 0);
}
__device__ __forceinline__ f4v tile_mfma(bf8v w, bf8v x, f4v acc)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, x, acc, 0, 0, 0);
}

// fragment address of input pixel (y, x): 16-channel input or 32-channel buffer
__device__ __forceinline__ int tile_at(s4v, int y, int x, int kg) { return at16(y, x, kg); }
__device__ __forceinline__ int tile_at(bf8v, int y, int x, int kg) { return at32(y, x, kg); }
template <typename Frag>
constexpr int tile_row_step()
{
    return sizeof(Frag) == 8 ? 24 * 16 : TILE_PITCH * 32;
}

// ROWS output rows from y0 on, columns 0..15: acc[r]
template <int ROWS, typename Frag>
__device__ __forceinline__ void tile_sweep(const bf16* in, int y0, const TileWeights<Frag>& W, int row, int kg,
                                           f4v (&acc)[ROWS])
{
    const bf16* base[3];
    for (int dx = 0; dx < 3; dx++) base[dx] = in + tile_at(Frag(), y0, row + dx, kg);
#pragma unroll
    for (int r = 0; r < ROWS; r++) acc[r] = f4v{0.f, 0.f, 0.f, 0.f};
    // the next row's fragments are read behind this row's first three MFMAs
    Frag f[2][3];
#pragma unroll
    for (int dx = 0; dx < 3; dx++) f[0][dx] = *(const Frag*)base[dx];
#pragma unroll
    for (int j = 0; j < ROWS + 2; j++) {
#pragma unroll
        for (int dx = 0; dx < 3; dx++) {
#pragma unroll
            for (int dy = 0; dy < 3; dy++) {
                const int r = j - dy;
                if (r >= 0 && r < ROWS) acc[r] = tile_mfma(W.w[dy * 3 + dx], f[j & 1][dx], acc[r]);
            }
            __builtin_amdgcn_sched_barrier(0);
            if (dx == 0 && j + 1 < ROWS + 2) {
#pragma unroll
                for (int d = 0; d < 3; d++)
                    f[(j + 1) & 1][d] = *(const Frag*)(base[d] + (j + 1) * tile_row_step<Frag>());
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
}

// a hidden layer: EDGE x EDGE output pixels (EDGE - 16 columns beside the
// swept 16) from `in` into the 32-channel buffer `out`; wave w computes
// channels 16 * (w & 1) .. + 15 of half of the rows (w >> 1) and of every
// second M-tile of the other columns
template <int EDGE, typename Frag>
__device__ __forceinline__ void tile_layer(const bf16* in, bf16* out, const TileWeights<Frag>& W, int wave, int lane)
{
    constexpr int ROWS = EDGE / 2;
    asm volatile("" : "+v"(lane));  // the addresses are computed here, not kept in registers across tiles
    const int row = lane & 15, kg = lane >> 4, band = wave >> 1, y0 = band * ROWS;
    const int g = (wave & 1) * 2 + (kg >> 1), gofs = (kg & 1) * 4;  // this lane's 4 output channels
    f4v acc[ROWS];
    tile_sweep<ROWS>(in, y0, W, row, kg, acc);
    bf16* o = out + at32(y0, row, g) + gofs;
#pragma unroll
    for (int r = 0; r < ROWS; r++) *(uint2*)(o + r * TILE_PITCH * 32) = relu_pack(acc[r], W.b);
    // its M-tiles band, band + 2, ... of the other columns together, so their
    // chains of nine dependent MFMAs overlap
    constexpr int RC = EDGE - 16, CNT = EDGE * RC, NM = ((CNT + 15) / 16 + 1) / 2;
    const bf16* base[NM][3];
    f4v c[NM];
#pragma unroll
    for (int m = 0; m < NM; m++) {
        const int i = min((band + 2 * m) * 16 + row, CNT - 1);  // past the end: the last pixel again, not stored
        for (int dx = 0; dx < 3; dx++) base[m][dx] = in + tile_at(Frag(), i / RC, 16 + i % RC + dx, kg);
        c[m] = f4v{0.f, 0.f, 0.f, 0.f};
    }
    Frag f[2][NM];
#pragma unroll
    for (int m = 0; m < NM; m++) f[0][m] = *(const Frag*)base[m][0];
#pragma unroll
    for (int tap = 0; tap < 9; tap++) {
        if (tap < 8)
#pragma unroll
            for (int m = 0; m < NM; m++)
                f[(tap + 1) & 1][m] =
                    *(const Frag*)(base[m][(tap + 1) % 3] + (tap + 1) / 3 * tile_row_step<Frag>());
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int m = 0; m < NM; m++) c[m] = tile_mfma(W.w[tap], f[tap & 1][m], c[m]);
        __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int m = 0; m < NM; m++) {
        const int i = (band + 2 * m) * 16 + row;
        if (i < CNT) *(uint2*)(out + at32(i / RC, 16 + i % RC, g) + gofs) = relu_pack(c[m], W.b);
    }
}

// The crop of tile c, pixels tid, tid + 256, tid + 512 of its 576: read from
// memory into registers (fetch), then features into the LDS input (put).
template <bool kExplicit>
struct TileCrop {  // frame mode: screen word and position
    uint32_t word[3];
    float px[3], py[3], pz[3];
    bool in[3];  // inside the screen
};
template <>
struct TileCrop<true> {
    uint4 lo[3], hi[3];
};

__device__ __forceinline__ const TileView* tile_view_of(const TileArgs& a, int c, int& lc)
{
    lc = c;
    if (!a.views) return &a.v;
    int lo = 0, hi = a.n_views - 1;  // the last view whose first tile is <= c
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if ((int)a.first[mid] <= c) lo = mid;
        else hi = mid - 1;
    }
    lc = c - (int)a.first[lo];
    return &a.views[lo];
}

__device__ __forceinline__ void tile_fetch(const TileArgs& a, int c, int tid, TileCrop<true>& q)
{
    asm volatile("" : "+v"(tid));  // as in tile_layer
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const int p = min(tid + 256 * k, 575);
        const uint4* src = (const uint4*)(a.x + ((size_t)c * 576 + p) * 16);
        q.lo[k] = src[0];
        q.hi[k] = src[1];
    }
}

__device__ __forceinline__ void tile_fetch(const TileArgs& a, int c, int tid, TileCrop<false>& q)
{
    asm volatile("" : "+v"(tid));  // as in tile_layer
    int lc;
    const TileView* V = tile_view_of(a, c, lc);
    const int t = (int)V->tiles[lc];
    const int ox = (t % V->tiles_x) * 16 - 4, oy = (t / V->tiles_x) * 16 - 4;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const int p = tid + 256 * k;
        const int x = ox + p % 24, y = oy + p / 24;
        q.in[k] = p < 576 && x >= 0 && y >= 0 && x < V->res_x && y < V->res_y;
        if (!q.in[k]) continue;
        const size_t o = (size_t)y * V->res_x + x;
        q.word[k] = V->words[o];
        const float4 pos = V->coords[o];
        q.px[k] = pos.x;
        q.py[k] = pos.y;
        q.pz[k] = pos.z;
    }
}

__device__ __forceinline__ void tile_put(const TileArgs&, int, int tid, const TileCrop<true>& q, bf16* P)
{
    asm volatile("" : "+v"(tid));
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const int p = tid + 256 * k, y = p / 24, x = p % 24;
        if (p >= 576) continue;
        *(uint2*)(P + at16(y, x, 0)) = make_uint2(q.lo[k].x, q.lo[k].y);
        *(uint2*)(P + at16(y, x, 1)) = make_uint2(q.lo[k].z, q.lo[k].w);
        *(uint2*)(P + at16(y, x, 2)) = make_uint2(q.hi[k].x, q.hi[k].y);
        *(uint2*)(P + at16(y, x, 3)) = make_uint2(q.hi[k].z, q.hi[k].w);
    }
}

__device__ __forceinline__ void tile_put(const TileArgs& a, int c, int tid, const TileCrop<false>& q, bf16* P)
{
    asm volatile("" : "+v"(tid));
    int lc;
    const TileView* V = tile_view_of(a, c, lc);
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const int p = tid + 256 * k, y = p / 24, x = p % 24;
        if (p >= 576) continue;
        float f[5] = {0.f, 0.f, 0.f, 0.f, 0.f};
        if (q.in[k]) {
            if (q.word[k] == HOLE_WORD) {
                f[4] = 1.f;
            } else {
                rgb_of(q.word[k], f[0], f[1], f[2]);
                const float qx = q.px[k] - V->m0x, qy = q.py[k] - V->m0y, qz = q.pz[k] - V->m0z;
                const float z = fmaxf((qx * V->r20 + qy * V->r21) + qz * V->r22, 0.f);
                f[3] = z / (z + 64.f);
            }
        }
        *(uint2*)(P + at16(y, x, 0)) = make_uint2((uint32_t)f2bf(f[0]) | ((uint32_t)f2bf(f[1]) << 16),
                                                  (uint32_t)f2bf(f[2]) | ((uint32_t)f2bf(f[3]) << 16));
        *(uint2*)(P + at16(y, x, 1)) = make_uint2((uint32_t)f2bf(f[4]), 0u);
        *(uint2*)(P + at16(y, x, 2)) = make_uint2(0u, 0u);
        *(uint2*)(P + at16(y, x, 3)) = make_uint2(0u, 0u);
    }
}

// LDS pixels of the 32-channel buffers (the last row ends at its last column)
constexpr int tile_pixels(int edge) { return (edge - 1) * TILE_PITCH + edge; }

// two waves per SIMD: 256 registers each, the weights need 99 of them
template <bool kExplicit>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_cnn_tiles(TileArgs a)
{
    __shared__ __align__(16) bf16 P[tile_pixels(20) * 32];  // the 24x24 input, then layer 2's output
    __shared__ __align__(16) bf16 Q[tile_pixels(22) * 32];  // layer 1's output, then layer 3's
    static_assert(576 * 16 <= tile_pixels(20) * 32, "the input fits in P");
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, row = lane & 15, kg = lane >> 4;
    const int n = kExplicit ? a.n : a.views ? (int)a.first[a.n_views] : min((int)*a.v.count, a.v.max_tiles);
    int c = blockIdx.x;
    if (c >= n) return;
    const int co0 = (wave & 1) * 16;  // this wave's channels of the hidden layers
    TileWeights<s4v> w1;
    TileWeights<bf8v> w2, w3;
    w1.load(a.w[0], a.b[0], 32, 16, co0, row, kg);
    w2.load(a.w[1], a.b[1], 32, 32, co0, row, kg);
    w3.load(a.w[2], a.b[2], 32, 32, co0, row, kg);
    TileCrop<kExplicit> crop;
    tile_fetch(a, c, tid, crop);
    for (; c < n; c += gridDim.x) {
        tile_put(a, c, tid, crop, P);  // every wave is past layer 3 of the tile before: P is free
        __syncthreads();
        tile_layer<22>(P, Q, w1, wave, lane);
        __syncthreads();
        tile_layer<20>(Q, P, w2, wave, lane);
        __syncthreads();
        if (c + (int)gridDim.x < n) tile_fetch(a, c + gridDim.x, tid, crop);
        // layer 4's weights are read again per tile: 36 more registers would spill
        const bf16* w4p = a.w[3];
        asm volatile("" : "+s"(w4p));
        TileWeights<bf8v> w4;
        w4.load(w4p, a.b[3], 16, 32, 0, row, kg);
        tile_layer<18>(P, Q, w3, wave, lane);
        __syncthreads();
        // layer 4: RGB are the first channels, held by the lanes of kg 0
        f4v acc[4];
        tile_sweep<4>(Q, wave * 4, w4, row, kg, acc);
        if (kg == 0) {
            int lc;
            const TileView* V = tile_view_of(a, c, lc);
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const f4v v = acc[r] + w4.b;
                const int px = (wave * 4 + r) * 16 + row;
                if (kExplicit) {
                    float* o = a.out + ((size_t)c * 256 + px) * 3;
                    o[0] = v[0];
                    o[1] = v[1];
                    o[2] = v[2];
                } else {
                    V->staged[(size_t)lc * 256 + px] = rgb_word(v[0], v[1], v[2]);
                }
            }
        }
    }
}

// All parameters at once: with kStep an Adam step first (FP32 master weights;
// m, v moments, bias-corrected), then the weights' bf16 copies, forward
// [9][cout][cin] and for the backward data W'[t][ci][co] = W[8-t][co][ci].
// (16 launches of 2.5 us each and the gaps between them before.)
template <bool kStep>
__global__ __launch_bounds__(256) void k_params(float* __restrict__ w, const float* __restrict__ g,
                                                float* __restrict__ m, float* __restrict__ v,
                                                bf16* __restrict__ wbf, bf16* __restrict__ wflip, float lr, float b1,
                                                float b2, float c1, float c2, float eps)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= kParams) return;
    float x = w[i];
    if (kStep) {
        const float gi = g[i];
        const float mi = b1 * m[i] + (1.f - b1) * gi;
        const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
        m[i] = mi;
        v[i] = vi;
        x -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
        w[i] = x;
    }
    const int l = layer_of(kPofs, i), e = i - kPofs[l], cin = kCin[l], cout = kCout[l], per = cin * cout;
    if (e >= 9 * per) return;  // a bias
    const int t = e / per, co = e % per / cin, ci = e % cin;
    const bf16 h = f2bf(x);
    wbf[kWofs[l] + e] = h;
    wflip[kWofs[l] + ((8 - t) * cin + ci) * cout + co] = h;
}

}  // namespace

// ====================================================================== host
struct CnnLayer {
    float* w;     // fp32 master [9][cout][cin]
    float* b;     // fp32 [cout]
    bf16* wbf;    // forward weights
    bf16* wflip;  // backward-data weights [9][cin][cout]
};

struct svo_cnn {
    int device = 0;
    int n_cu = 256;        // compute units of the device (tile kernel grid)
    hipStream_t stream = nullptr;
    CnnLayer L[4] = {};  // into params, wbf, wflip
    float *params = nullptr, *grads = nullptr, *m = nullptr, *v = nullptr;  // flat, kParams each
    bf16 *wbf = nullptr, *wflip = nullptr;
    float* h_grads = nullptr;  // pinned: kParams gradients and the loss
    int step = 0;
    // activation workspace for the current batch size, one allocation of 288
    // bytes per pixel (x0 is its start)
    size_t cap_pix = 0;
    bf16* x0 = nullptr;    // [pix][16]
    bf16* y[3] = {};       // [pix][32]
    float* out = nullptr;  // [pix][16]
    // and what gradients need beside it, allocated by the first call that
    // makes them: 240 bytes per pixel (dz[0] is its start)
    size_t cap_grad = 0;
    bf16* dz[4] = {};      // [pix][32], the last layer's [pix][16]
    float* target = nullptr;
    float* mask = nullptr;
    float* loss = nullptr;
    float* mask_count = nullptr;
    int2* origins = nullptr;
    int max_origins = 0;
    bool fused = true;     // per-tile fused inference kernel for the frame fill
    bf16* xt = nullptr;    // explicit-mode tile inputs / outputs
    float* ot = nullptr;
    size_t cap_tiles = 0;
    float* part = nullptr;  // gradient partials: per crop and tap, then per block
    size_t cap_part = 0;
};

#define RCC(x)             \
    do {                   \
        int _r = (x);      \
        if (_r) return _r; \
    } while (0)

#define HIPCHECK(expr)                                                                    \
    do {                                                                                  \
        hipError_t _e = (expr);                                                           \
        if (_e != hipSuccess)                                                             \
            return svo_fail(SVO_ERR_HIP, "%s failed: %s", #expr, hipGetErrorString(_e)); \
    } while (0)

static void free_forward_ws(svo_cnn* n)
{
    (void)hipFree(n->x0);
    n->x0 = nullptr;
    n->cap_pix = 0;
}

static void free_grad_ws(svo_cnn* n)
{
    (void)hipFree(n->dz[0]);
    n->dz[0] = nullptr;
    n->cap_grad = 0;
}

// The workspace of a forward over pix pixels (a multiple of 64), and of its
// gradients.  One allocation each: the first gradients of 16 crops of 64x64 by a
// new network take 0.33 ms, 2.0 with an allocation per array (eleven).
static int ensure_ws(svo_cnn* n, size_t pix, bool grads)
{
    if (pix > n->cap_pix) {
        free_forward_ws(n);
        if (hipMalloc(&n->x0, pix * (16 * 2 + 3 * 32 * 2 + 16 * 4)) != hipSuccess) {
            n->x0 = nullptr;
            return svo_fail(SVO_ERR_NOMEM, "CNN workspace for %zu pixels", pix);
        }
        for (int l = 0; l < 3; l++) n->y[l] = n->x0 + pix * (16 + l * 32);
        n->out = (float*)(n->x0 + pix * (16 + 3 * 32));
        n->cap_pix = pix;
    }
    if (grads && pix > n->cap_grad) {
        free_grad_ws(n);
        if (hipMalloc(&n->dz[0], pix * (3 * 32 * 2 + 16 * 2 + 3 * 4 + 4)) != hipSuccess) {
            n->dz[0] = nullptr;
            return svo_fail(SVO_ERR_NOMEM, "CNN gradient workspace for %zu pixels", pix);
        }
        for (int l = 1; l < 4; l++) n->dz[l] = n->dz[0] + pix * l * 32;
        n->target = (float*)(n->dz[3] + pix * 16);
        n->mask = n->target + pix * 3;
        n->cap_grad = pix;
    }
    return SVO_OK;
}

static unsigned nb(size_t n) { return (unsigned)((n + 255) / 256); }

static int refresh_bf16(svo_cnn* n)
{
    hipLaunchKernelGGL(k_params<false>, dim3(nb(kParams)), dim3(256), 0, n->stream, n->params, (const float*)nullptr,
                       (float*)nullptr, (float*)nullptr, n->wbf, n->wflip, 0.f, 0.f, 0.f, 1.f, 1.f, 0.f);
    HIPCHECK(hipGetLastError());
    return SVO_OK;
}

extern "C" int svo_cnn_destroy(svo_cnn* n)
{
    if (!n) return SVO_OK;
    (void)hipSetDevice(n->device);
    (void)hipStreamSynchronize(n->stream);
    free_forward_ws(n);
    free_grad_ws(n);
    for (float* p : {n->params, n->grads, n->m, n->v}) (void)hipFree(p);
    (void)hipFree(n->wbf);
    (void)hipFree(n->wflip);
    (void)hipHostFree(n->h_grads);
    (void)hipFree(n->loss);
    (void)hipFree(n->mask_count);
    (void)hipFree(n->part);
    (void)hipFree(n->origins);
    (void)hipFree(n->xt);
    (void)hipFree(n->ot);
    if (n->stream) (void)hipStreamDestroy(n->stream);
    delete n;
    return SVO_OK;
}

extern "C" size_t svo_cnn_param_count(void)
{
    return kParams;
}

extern "C" int svo_cnn_create(svo_cnn** out, int device, uint64_t seed)
{
    if (!out) return svo_fail(SVO_ERR_ARG, "null output pointer");
    *out = nullptr;
    HIPCHECK(hipSetDevice(device));
    svo_cnn* n = new svo_cnn();
    n->device = device;
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, device) == hipSuccess && prop.multiProcessorCount > 0)
        n->n_cu = prop.multiProcessorCount;
    if (hipStreamCreateWithFlags(&n->stream, hipStreamNonBlocking) != hipSuccess ||
        hipMalloc(&n->loss, 4) != hipSuccess || hipMalloc(&n->mask_count, 4) != hipSuccess) {
        svo_cnn_destroy(n);
        return svo_fail(SVO_ERR_HIP, "CNN set-up failed");
    }
    // He-normal init of the real channels (Box-Muller over a splitmix stream)
    uint64_t st = seed * 0x9E3779B97F4A7C15ull + 1;
    auto next = [&]() {
        st += 0x9E3779B97F4A7C15ull;
        uint64_t z = st;
        z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
        z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
        return ((z ^ (z >> 31)) >> 11) * (1.0 / 9007199254740992.0);
    };
    const int real_in[4] = {5, 32, 32, 32}, real_out[4] = {32, 32, 32, 3};
    std::vector<float> w(kParams, 0.f);
    for (int li = 0; li < 4; li++) {
        const double sd = sqrt(2.0 / (9.0 * real_in[li])) * (li == 3 ? 0.5 : 1.0);
        for (int t = 0; t < 9; t++)
            for (int co = 0; co < real_out[li]; co++)
                for (int ci = 0; ci < real_in[li]; ci++) {
                    double u1 = std::max(next(), 1e-12), u2 = next();
                    w[kPofs[li] + (t * kCout[li] + co) * kCin[li] + ci] = (float)(sd * sqrt(-2 * log(u1)) * cos(6.283185307179586 * u2));
                }
    }
    bool ok = true;
    for (float** p : {&n->params, &n->grads, &n->m, &n->v}) ok = ok && hipMalloc(p, kParams * 4) == hipSuccess;
    for (bf16** p : {&n->wbf, &n->wflip}) ok = ok && hipMalloc(p, kWofs[4] * 2) == hipSuccess;
    ok = ok && hipHostMalloc((void**)&n->h_grads, (kParams + 1) * 4, hipHostMallocDefault) == hipSuccess;
    if (!ok) {
        svo_cnn_destroy(n);
        return svo_fail(SVO_ERR_NOMEM, "CNN weights");
    }
    (void)hipMemcpy(n->params, w.data(), kParams * 4, hipMemcpyHostToDevice);
    for (float* p : {n->m, n->v}) (void)hipMemset(p, 0, kParams * 4);
    for (int l = 0; l < 4; l++)
        n->L[l] = {n->params + kPofs[l], n->params + kPofs[l + 1] - kCout[l], n->wbf + kWofs[l], n->wflip + kWofs[l]};
    int rc = refresh_bf16(n);
    if (rc) {
        svo_cnn_destroy(n);
        return rc;
    }
    HIPCHECK(hipStreamSynchronize(n->stream));
    *out = n;
    return SVO_OK;
}

// flat parameter vector: per layer W [9][cout][cin] then b [cout]
extern "C" int svo_cnn_get_params(svo_cnn* n, float* dst, size_t count)
{
    if (!n || !dst || count != svo_cnn_param_count()) return svo_fail(SVO_ERR_ARG, "need %zu floats", svo_cnn_param_count());
    HIPCHECK(hipStreamSynchronize(n->stream));
    HIPCHECK(hipMemcpy(dst, n->params, kParams * 4, hipMemcpyDeviceToHost));
    return SVO_OK;
}

extern "C" int svo_cnn_set_params(svo_cnn* n, const float* src, size_t count)
{
    if (!n || !src || count != svo_cnn_param_count()) return svo_fail(SVO_ERR_ARG, "need %zu floats", svo_cnn_param_count());
    HIPCHECK(hipStreamSynchronize(n->stream));
    HIPCHECK(hipMemcpy(n->params, src, kParams * 4, hipMemcpyHostToDevice));
    return refresh_bf16(n);
}

static unsigned conv_grid(int B, int H, int W) { return (unsigned)std::min(B * (H / TILE) * (W / TILE), 16384); }

int cnn_forward_dev(svo_cnn* n, int B, int H, int W, const uint32_t* bcount = nullptr)
{
    const unsigned g = conv_grid(B, H, W);
    hipLaunchKernelGGL((k_conv<16, 32, 0>), dim3(g), dim3(64), 0, n->stream, n->x0, n->L[0].wbf, n->L[0].b,
                       (const bf16*)nullptr, (void*)n->y[0], H, W, B, bcount);
    hipLaunchKernelGGL((k_conv<32, 32, 0>), dim3(g), dim3(64), 0, n->stream, n->y[0], n->L[1].wbf, n->L[1].b,
                       (const bf16*)nullptr, (void*)n->y[1], H, W, B, bcount);
    hipLaunchKernelGGL((k_conv<32, 32, 0>), dim3(g), dim3(64), 0, n->stream, n->y[1], n->L[2].wbf, n->L[2].b,
                       (const bf16*)nullptr, (void*)n->y[2], H, W, B, bcount);
    hipLaunchKernelGGL((k_conv<32, 16, 1>), dim3(g), dim3(64), 0, n->stream, n->y[2], n->L[3].wbf, n->L[3].b,
                       (const bf16*)nullptr, (void*)n->out, H, W, B, bcount);
    HIPCHECK(hipGetLastError());
    return SVO_OK;
}

// Partials of all layers' weights at most: beyond it (more than 2,427 crops)
// the gradients are made layer by layer through one layer's partials.
constexpr size_t kPartBytes = (size_t)1 << 28;

// backward from n->out vs n->target/n->mask; gradients into n->grads
// (per-crop and per-block partials added in a fixed order)
int cnn_backward_dev(svo_cnn* n, int B, int H, int W)
{
    const size_t pix = (size_t)B * H * W;
    const unsigned g = conv_grid(B, H, W);
    const unsigned gdb = (unsigned)((pix + DB_PIXELS - 1) / DB_PIXELS);
    const int together = (size_t)B * kWofs[4] * 4 <= kPartBytes ? 4 : 1;  // layers per launch
    const size_t need_w = (size_t)B * (together == 4 ? kWofs[4] : 9 * 32 * 32);
    const size_t need = need_w + (size_t)gdb * 32 * together;
    if (need > n->cap_part) {
        (void)hipFree(n->part);
        n->part = nullptr;
        n->cap_part = 0;
        if (hipMalloc(&n->part, need * 4) != hipSuccess) return svo_fail(SVO_ERR_NOMEM, "gradient partials");
        n->cap_part = need;
    }
    HIPCHECK(hipMemsetAsync(n->loss, 0, 4, n->stream));
    hipLaunchKernelGGL(k_loss, dim3(std::min(nb(pix / 4), 1024u)), dim3(256), 0, n->stream, n->out, n->target,
                       n->mask, n->dz[3], n->loss, (int)pix, n->mask_count);
    hipLaunchKernelGGL((k_conv<16, 32, 2>), dim3(g), dim3(64), 0, n->stream, n->dz[3], n->L[3].wflip,
                       (const float*)nullptr, n->y[2], (void*)n->dz[2], H, W, B, (const uint32_t*)nullptr);
    hipLaunchKernelGGL((k_conv<32, 32, 2>), dim3(g), dim3(64), 0, n->stream, n->dz[2], n->L[2].wflip,
                       (const float*)nullptr, n->y[1], (void*)n->dz[1], H, W, B, (const uint32_t*)nullptr);
    hipLaunchKernelGGL((k_conv<32, 32, 2>), dim3(g), dim3(64), 0, n->stream, n->dz[1], n->L[1].wflip,
                       (const float*)nullptr, n->y[0], (void*)n->dz[0], H, W, B, (const uint32_t*)nullptr);
    GradArgs a{{n->x0, n->y[0], n->y[1], n->y[2]}, {n->dz[0], n->dz[1], n->dz[2], n->dz[3]},
               n->part, n->part + need_w, n->grads, B, H, W, 0, (int)gdb};
    for (; a.lo < 4; a.lo += together) {
        const int hi = a.lo + together;
        const int biases = 32 * (together - 1) + kCout[hi - 1];
        hipLaunchKernelGGL(k_conv_dw, dim3((unsigned)B, 3, (unsigned)together), dim3(64 * DW_SLICES), 0, n->stream, a);
        hipLaunchKernelGGL(k_conv_db, dim3(gdb, (unsigned)together), dim3(256), 0, n->stream, a);
        hipLaunchKernelGGL(k_sum_grads, dim3((unsigned)((kWofs[hi] - kWofs[a.lo]) / 256 + biases)), dim3(256), 0,
                           n->stream, a, hi);
    }
    HIPCHECK(hipGetLastError());
    return SVO_OK;
}

int cnn_adam_dev(svo_cnn* n, float lr)
{
    n->step++;
    const float b1 = 0.9f, b2 = 0.999f;
    const float c1 = 1.f - powf(b1, (float)n->step), c2 = 1.f - powf(b2, (float)n->step);
    hipLaunchKernelGGL(k_params<true>, dim3(nb(kParams)), dim3(256), 0, n->stream, n->params, (const float*)n->grads,
                       n->m, n->v, n->wbf, n->wflip, lr, b1, b2, c1, c2, 1e-8f);
    HIPCHECK(hipGetLastError());
    return SVO_OK;
}

static int check_shape(int B, int H, int W)
{
    if (B <= 0 || H <= 0 || W <= 0 || H % TILE || W % TILE || (size_t)B * H * W > (1u << 26) || (H * W) % 16)
        return svo_fail(SVO_ERR_ARG, "batch %dx%dx%d: H and W must be positive multiples of 8", B, H, W);
    return SVO_OK;
}

// Raw forward on host data: x = [B][H][W][16] bf16 bits, out = [B][H][W][16] fp32.
extern "C" int svo_cnn_forward(svo_cnn* n, const uint16_t* x, int B, int H, int W, float* out)
{
    if (!n || !x || !out) return svo_fail(SVO_ERR_ARG, "null argument");
    int rc = check_shape(B, H, W);
    if (rc) return rc;
    HIPCHECK(hipSetDevice(n->device));
    const size_t pix = (size_t)B * H * W;
    rc = ensure_ws(n, pix, false);
    if (rc) return rc;
    HIPCHECK(hipMemcpyAsync(n->x0, x, pix * 16 * 2, hipMemcpyHostToDevice, n->stream));
    rc = cnn_forward_dev(n, B, H, W);
    if (rc) return rc;
    HIPCHECK(hipMemcpyAsync(out, n->out, pix * 16 * 4, hipMemcpyDeviceToHost, n->stream));
    HIPCHECK(hipStreamSynchronize(n->stream));
    return SVO_OK;
}

// Raw loss + gradients (no update): target [B][H][W][3], mask [B][H][W];
// grads written as the flat parameter vector layout; returns the loss.
extern "C" int svo_cnn_gradients(svo_cnn* n, const uint16_t* x, const float* target, const float* mask, int B, int H,
                                 int W, float* grads, size_t count, float* loss)
{
    if (!n || !x || !target || !mask || !grads || !loss) return svo_fail(SVO_ERR_ARG, "null argument");
    if (count != svo_cnn_param_count()) return svo_fail(SVO_ERR_ARG, "need %zu floats", svo_cnn_param_count());
    int rc = check_shape(B, H, W);
    if (rc) return rc;
    HIPCHECK(hipSetDevice(n->device));
    const size_t pix = (size_t)B * H * W;
    rc = ensure_ws(n, pix, true);
    if (rc) return rc;
    HIPCHECK(hipMemcpyAsync(n->x0, x, pix * 16 * 2, hipMemcpyHostToDevice, n->stream));
    HIPCHECK(hipMemcpyAsync(n->target, target, pix * 3 * 4, hipMemcpyHostToDevice, n->stream));
    HIPCHECK(hipMemcpyAsync(n->mask, mask, pix * 4, hipMemcpyHostToDevice, n->stream));
    if ((rc = cnn_forward_dev(n, B, H, W))) return rc;
    float cnt = 0.f;  // while the forward runs
    for (size_t i = 0; i < pix; i++) cnt += mask[i];
    HIPCHECK(hipMemcpyAsync(n->mask_count, &cnt, 4, hipMemcpyHostToDevice, n->stream));
    if ((rc = cnn_backward_dev(n, B, H, W))) return rc;
    HIPCHECK(hipMemcpyAsync(n->h_grads, n->grads, kParams * 4, hipMemcpyDeviceToHost, n->stream));
    HIPCHECK(hipMemcpyAsync(n->h_grads + kParams, n->loss, 4, hipMemcpyDeviceToHost, n->stream));
    HIPCHECK(hipStreamSynchronize(n->stream));
    memcpy(grads, n->h_grads, kParams * 4);
    *loss = n->h_grads[kParams];
    return SVO_OK;
}

static FeatArgs feat_args(svo_cnn* n, svo_ctx* c, const svo_frame_params* p, int crop)
{
    FeatArgs a;
    memset(&a, 0, sizeof(a));
    a.words = c->d_cnn_words;
    a.coords = c->d_cnn_coords;
    a.res_x = c->res_x;
    a.res_y = c->res_y;
    a.crop = crop;
    a.tiles_x = c->n_tiles_x;
    a.m0x = p->m0[0]; a.m0y = p->m0[1]; a.m0z = p->m0[2];
    a.r20 = p->row2[0]; a.r21 = p->row2[1]; a.r22 = p->row2[2];
    a.x = n->x0;
    return a;
}

// One Adam step on n_crops crop x crop windows of the current frame pair:
// features from the warp context's last learned-frame CNN input (plane 0 as
// its gate left it), targets from the full context's image, loss on the
// pixels still holes after the warp frame's rays.  Both contexts must have
// rendered the same camera.  The CNN's stream waits for both contexts.
extern "C" int svo_cnn_train_step(svo_cnn* n, svo_ctx* warp, svo_ctx* full, const svo_frame_params* p, int n_crops,
                                  int crop, uint64_t seed, float lr, float* loss_out)
{
    if (!n || !warp || !full || !p) return svo_fail(SVO_ERR_ARG, "null argument");
    if (warp->res_x != full->res_x || warp->res_y != full->res_y || !warp->d_screen)
        return svo_fail(SVO_ERR_STATE, "contexts must share one resolution");
    if (!warp->cnn_input)
        return svo_fail(SVO_ERR_STATE, "the warp context has rendered no learned frame since its last resize");
    if (n_crops <= 0 || n_crops > 256 || crop < 16 || crop % 8 || crop > warp->res_x || crop > warp->res_y)
        return svo_fail(SVO_ERR_ARG, "bad crop batch %d x %d", n_crops, crop);
    HIPCHECK(hipSetDevice(n->device));
    int rc = ensure_ws(n, (size_t)n_crops * crop * crop, true);
    if (rc) return rc;
    if (n->max_origins < n_crops) {
        (void)hipFree(n->origins);
        n->origins = nullptr;
        HIPCHECK(hipMalloc(&n->origins, sizeof(int2) * 256));
        n->max_origins = 256;
    }
    std::vector<int2> org(n_crops);
    uint64_t st = seed * 0x9E3779B97F4A7C15ull + 0x1234567ull;
    for (auto& o : org) {
        st = st * 6364136223846793005ull + 1442695040888963407ull;
        o.x = (int)((st >> 33) % (uint64_t)(warp->res_x - crop + 1));
        st = st * 6364136223846793005ull + 1442695040888963407ull;
        o.y = (int)((st >> 33) % (uint64_t)(warp->res_y - crop + 1));
    }
    // order after both contexts' queued frames
    hipEvent_t e1, e2;
    HIPCHECK(hipEventCreateWithFlags(&e1, hipEventDisableTiming));
    HIPCHECK(hipEventCreateWithFlags(&e2, hipEventDisableTiming));
    (void)hipEventRecord(e1, warp->stream);
    (void)hipEventRecord(e2, full->stream);
    (void)hipStreamWaitEvent(n->stream, e1, 0);
    (void)hipStreamWaitEvent(n->stream, e2, 0);
    HIPCHECK(hipMemcpyAsync(n->origins, org.data(), sizeof(int2) * n_crops, hipMemcpyHostToDevice, n->stream));
    HIPCHECK(hipMemsetAsync(n->mask_count, 0, 4, n->stream));
    FeatArgs a = feat_args(n, warp, p, crop);
    a.mask_words = warp->d_screen + 2 * warp->N;  // holes left after the frame's rays
    a.image = full->d_image;
    a.origins = n->origins;
    a.max_crops = n_crops;
    a.target = n->target;
    a.mask = n->mask;
    a.mask_count = n->mask_count;
    const size_t pix = (size_t)n_crops * crop * crop;
    hipLaunchKernelGGL(k_features, dim3(std::min(nb(pix / 2), 1024u)), dim3(256), 0, n->stream, a);
    HIPCHECK(hipGetLastError());
    if ((rc = cnn_forward_dev(n, n_crops, crop, crop)) || (rc = cnn_backward_dev(n, n_crops, crop, crop)) ||
        (rc = cnn_adam_dev(n, lr)))
        return rc;
    // the next frames of either context wait for this step's reads
    (void)hipEventRecord(e1, n->stream);
    (void)hipStreamWaitEvent(warp->stream, e1, 0);
    (void)hipStreamWaitEvent(full->stream, e1, 0);
    (void)hipEventDestroy(e1);
    (void)hipEventDestroy(e2);
    if (loss_out) {
        HIPCHECK(hipStreamSynchronize(n->stream));
        HIPCHECK(hipMemcpy(loss_out, n->loss, 4, hipMemcpyDeviceToHost));
    }
    return SVO_OK;
}

// Inference on the gate's tile list (24x24 crops around each 16x16 tile of
// the CNN input planes) into the staged colours, queued on `stream`.
static TileArgs tile_args(svo_cnn* n)
{
    TileArgs a;
    memset(&a, 0, sizeof(a));
    for (int i = 0; i < 4; i++) {
        a.w[i] = n->L[i].wbf;
        a.b[i] = n->L[i].b;
    }
    return a;
}

// grid > 0: that many workgroups, at most one per tile (they loop over the
// tile list, so any count covers every tile); 0: two per CU
static int launch_tiles(const TileArgs& a, int max_tiles, int cus, hipStream_t stream, int grid)
{
    const unsigned g = (unsigned)std::max(1, std::min(max_tiles, grid > 0 ? grid : 2 * cus));
    if (a.x)
        hipLaunchKernelGGL(k_cnn_tiles<true>, dim3(g), dim3(256), 0, stream, a);
    else
        hipLaunchKernelGGL(k_cnn_tiles<false>, dim3(g), dim3(256), 0, stream, a);
    HIPCHECK(hipGetLastError());
    return SVO_OK;
}

static TileView tile_view(svo_ctx* c, const svo_frame_params* p, const uint32_t* tile_list,
                          const uint32_t* tile_count, int max_tiles)
{
    TileView v;
    memset(&v, 0, sizeof(v));
    v.words = c->d_cnn_words;
    v.coords = c->d_cnn_coords;
    v.res_x = c->res_x;
    v.res_y = c->res_y;
    v.tiles_x = c->n_tiles_x;
    v.tiles = tile_list;
    v.count = tile_count;
    v.max_tiles = max_tiles;
    v.m0x = p->m0[0]; v.m0y = p->m0[1]; v.m0z = p->m0[2];
    v.r20 = p->row2[0]; v.r21 = p->row2[1]; v.r22 = p->row2[2];
    v.staged = c->d_cnn_out;
    v.plane2 = c->d_screen + 2 * c->N;
    v.image = c->d_image;
    return v;
}

int cnn_fill_tiles(svo_cnn* n, svo_ctx* c, const svo_frame_params* p, const uint32_t* tile_list,
                   const uint32_t* tile_count, int max_tiles, hipStream_t stream, int grid)
{
    if (n->fused) {
        TileArgs a = tile_args(n);
        a.v = tile_view(c, p, tile_list, tile_count, max_tiles);
        return launch_tiles(a, max_tiles, n->n_cu, stream, grid);
    }
    int rc = ensure_ws(n, (size_t)max_tiles * 576, false);
    if (rc) return rc;
    hipStream_t keep = n->stream;
    n->stream = stream;  // run on the frame's stream
    FeatArgs a = feat_args(n, c, p, 24);
    a.tiles = tile_list;
    a.count = tile_count;
    a.max_crops = max_tiles;
    hipLaunchKernelGGL(k_features, dim3(2048), dim3(256), 0, n->stream, a);
    rc = cnn_forward_dev(n, max_tiles, 24, 24, tile_count);
    if (!rc) {
        hipLaunchKernelGGL(k_stage_fill, dim3(2048), dim3(256), 0, n->stream, n->out, tile_count, max_tiles,
                           c->d_cnn_out);
        if (hipGetLastError() != hipSuccess) rc = svo_fail(SVO_ERR_HIP, "CNN fill launch failed");
    }
    n->stream = keep;
    return rc;
}

size_t cnn_tile_view_bytes() { return sizeof(TileView); }

// Every view of a batch in one tile launch: the views' gate tile lists are
// concatenated through a table (host staging h_tab, device copy d_tab, both
// n_views entries; first: n_views + 1 words) written here and copied on
// `stream` ahead of the launch.  The per-layer kernels (fused mode off) run
// view by view.
int cnn_fill_tiles_batch(svo_cnn* n, svo_ctx* const* views, const svo_frame_params* params, int n_views,
                         void* h_tab, void* d_tab, uint32_t* first, hipStream_t stream)
{
    TileView* hv = (TileView*)h_tab;
    int max_all = 0;
    for (int i = 0; i < n_views; i++) {
        svo_ctx* c = views[i];
        const int mt = c->n_tiles_x * c->n_tiles_y;
        hv[i] = tile_view(c, &params[i], c->d_gate_tiles, c->d_gate, mt);
        max_all += mt;
    }
    if (!n->fused) {
        for (int i = 0; i < n_views; i++) {
            svo_ctx* c = views[i];
            RCC(cnn_fill_tiles(n, c, &params[i], c->d_gate_tiles, c->d_gate, c->n_tiles_x * c->n_tiles_y, stream));
        }
        HIPCHECK(hipMemcpyAsync(d_tab, h_tab, sizeof(TileView) * n_views, hipMemcpyHostToDevice, stream));
        return SVO_OK;
    }
    HIPCHECK(hipMemcpyAsync(d_tab, h_tab, sizeof(TileView) * n_views, hipMemcpyHostToDevice, stream));
    hipLaunchKernelGGL(k_tile_first, dim3(1), dim3(1), 0, stream, (const TileView*)d_tab, n_views, first);
    HIPCHECK(hipGetLastError());
    TileArgs a = tile_args(n);
    a.views = (const TileView*)d_tab;
    a.first = first;
    a.n_views = n_views;
    return launch_tiles(a, max_all, n->n_cu, stream, 0);
}

// the staged colours of every view of a batch into their images (the table
// cnn_fill_tiles_batch copied to the device)
int cnn_apply_tiles_batch(const void* d_tab, int n_views, int max_tiles, hipStream_t stream)
{
    const unsigned g = (unsigned)std::max(1, std::min(2048, (max_tiles * 256 + 255) / 256));
    hipLaunchKernelGGL(k_cnn_apply_views, dim3(g, (unsigned)n_views), dim3(256), 0, stream, (const TileView*)d_tab);
    HIPCHECK(hipGetLastError());
    return SVO_OK;
}

int cnn_apply_tiles(svo_ctx* c, const uint32_t* tile_list, const uint32_t* tile_count, int max_tiles,
                    hipStream_t stream)
{
    hipLaunchKernelGGL(k_cnn_apply, dim3(2048), dim3(256), 0, stream, c->d_cnn_out, tile_list, tile_count, max_tiles,
                       c->d_screen + 2 * c->N, c->d_image, c->res_x, c->res_y, c->n_tiles_x);
    HIPCHECK(hipGetLastError());
    return SVO_OK;
}

// The fused tile network on explicit 24x24 crops: x [n][24][24][16] bf16
// features -> out [n][16][16][3] float (the centre 16x16, RGB).
extern "C" int svo_cnn_forward_tiles(svo_cnn* n, const uint16_t* x, int count, float* out)
{
    if (!n || !x || !out || count < 1 || count > (1 << 20)) return svo_fail(SVO_ERR_ARG, "bad tile batch");
    HIPCHECK(hipSetDevice(n->device));
    if ((size_t)count > n->cap_tiles) {
        (void)hipFree(n->xt);
        (void)hipFree(n->ot);
        n->xt = nullptr;
        n->ot = nullptr;
        n->cap_tiles = 0;
        if (hipMalloc(&n->xt, (size_t)count * 576 * 16 * 2) != hipSuccess ||
            hipMalloc(&n->ot, (size_t)count * 256 * 3 * 4) != hipSuccess)
            return svo_fail(SVO_ERR_NOMEM, "tile batch of %d", count);
        n->cap_tiles = (size_t)count;
    }
    HIPCHECK(hipMemcpyAsync(n->xt, x, (size_t)count * 576 * 16 * 2, hipMemcpyHostToDevice, n->stream));
    TileArgs a = tile_args(n);
    a.x = n->xt;
    a.out = n->ot;
    a.n = count;
    RCC(launch_tiles(a, count, n->n_cu, n->stream, 0));
    HIPCHECK(hipMemcpyAsync(out, n->ot, (size_t)count * 256 * 3 * 4, hipMemcpyDeviceToHost, n->stream));
    HIPCHECK(hipStreamSynchronize(n->stream));
    return SVO_OK;
}

extern "C" int svo_cnn_set_fused(svo_cnn* n, int mode)
{
    if (!n) return svo_fail(SVO_ERR_ARG, "null network");
    if (mode < 0 || mode > 2) return svo_fail(SVO_ERR_ARG, "fused mode %d outside 0..2", mode);
    n->fused = mode != 0;
    return SVO_OK;
}
