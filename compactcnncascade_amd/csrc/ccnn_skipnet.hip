// Learned tile skipping: a small proposal network that predicts, from a 1/8-downsampled
// gray frame, which stage-1 tiles of which pyramid levels can hold a window that the
// cascade accepts, so that the others are not computed. No counterpart in the reference:
// the plain cascade is its fallback (tiles the network is not confident about run as
// usual) and the reference its recall is measured against.
//
// Network (SkipNet): input x0 = mean of each 8x8 block of the FP32 gray image / 255 - 0.5
// (H8 x W8 = ceil(H/8) x ceil(W/8)); three 3x3 convolutions with zero padding ("same"),
// 1 -> 8 -> 8 -> SLOTS channels, ReLU after the first two; output channel s = the logit
// that pyramid level with scale index s (InitScales order) has an accepted window whose
// centre lies in the 8x8 frame cell. Levels with scale index >= SLOTS or scale < 0.5 are
// always run.
//
// Kernels (FP32; the inference weights are the trained ones rounded to FP16):
//   k_sn_down8      the network input of every frame of a batch from its gray image
//   k_sn_conv       one 3x3 layer over a set of equally or differently sized frames
//                   (one thread per position, every output channel)
//   k_sn_tile_mask  keep flag of every stage-1 response tile of a batch
//   k_sn_l1_mask    keep flag of every L1 tile: set when a kept response tile reads it
//   k_sn_bce, k_sn_conv_bwd_data, k_sn_conv_bwd_w, k_sn_update, k_sn_loss   training
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdio>
#include <cstring>
#include <type_traits>
#include <vector>

#include "ccnn.h"
#include "ccnn_detector.h"

namespace ccnn {

__device__ __forceinline__ int sn_frame_of(const SnFrame* __restrict__ fr, int nf, int pos)
{
    int lo = 0, hi = nf - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (fr[mid].pos_off <= pos) lo = mid; else hi = mid - 1;
    }
    return lo;
}

// x0 of every frame: levels' LevelDesc of the batch give each frame's gray image; one
// thread per cell. frames[f] = {h8, w8, off, pos_off} with off the frame's cell offset.
__global__ void __launch_bounds__(256) k_sn_down8(const float* __restrict__ gray, const FrameDesc* __restrict__ ft,
                                                  const SnFrame* __restrict__ fr, int nf, int total,
                                                  float* __restrict__ x0)
{
    const int pos = blockIdx.x * 256 + threadIdx.x;
    if (pos >= total) return;
    const int f = sn_frame_of(fr, nf, pos);
    const SnFrame F = fr[f];
    const int c = pos - F.pos_off;
    const int v = c / F.w8, u = c - v * F.w8;
    const FrameDesc& D = ft[f];
    const float* g = gray + D.gray_off;
    const int y0 = 8 * v, x0i = 8 * u;
    const int y1 = min(y0 + 8, D.h), x1 = min(x0i + 8, D.w);
    float s = 0.f;
    for (int y = y0; y < y1; ++y)
        for (int x = x0i; x < x1; ++x) s += g[(size_t)y * D.gp + x];
    const float n = (float)((y1 - y0) * (x1 - x0i));
    x0[F.off + c] = s / n * (1.f / 255.f) - 0.5f;
}

// The 3x3 neighbourhood of (x, y) in a plane of h x w, zeros outside.
__device__ __forceinline__ void sn_window(const float* __restrict__ src, int h, int w, int y, int x, float (&v)[9])
{
#pragma unroll
    for (int k = 0; k < 9; ++k) {
        const int yy = y + k / 3 - 1, xx = x + k % 3 - 1;
        v[k] = (yy >= 0 && yy < h && xx >= 0 && xx < w) ? src[yy * w + xx] : 0.f;
    }
}

// out[f][co][y][x] = relu?(b[co] + sum_{ci,ky,kx} w[co][ci][ky][kx] in[f][ci][y+ky-1][x+kx-1])
// with zero padding. One thread per frame position computes every output channel from the
// 9 * CIN inputs it loads once. fo (optional): the frames' first cells in `in` where they
// lie elsewhere than fr says (a training batch's frames within the whole set).
//
// Bound: the FMA issue (8 -> 24 channels: 1728 per position). The weights are the same for
// every lane, so they come through the scalar cache as SGPR operands, one output channel
// at a time; read as LDS broadcasts the 432 16-byte reads per wave held the LDS four times
// as long as the FMAs take to issue (8 -> 24 channels over 64 frames of 90 x 160 cells: 84
// -> 67 us).
template <int CIN, int COUT>
__global__ void __launch_bounds__(256) k_sn_conv(const float* __restrict__ in, const float* __restrict__ w,
                                                 const float* __restrict__ b, float* __restrict__ out,
                                                 const SnFrame* __restrict__ fr, const long long* __restrict__ fo,
                                                 int nf, int total, int relu)
{
    const int pos = blockIdx.x * 256 + threadIdx.x;
    if (pos >= total) return;
    const int f = sn_frame_of(fr, nf, pos);
    const SnFrame F = fr[f];
    const int c = pos - F.pos_off;
    const int y = c / F.w8, x = c - y * F.w8;
    const int plane = F.h8 * F.w8;
    const float* src = in + (size_t)(fo ? fo[f] : F.off) * CIN;
    float v[CIN][9];
#pragma unroll
    for (int ci = 0; ci < CIN; ++ci) sn_window(src + (size_t)ci * plane, F.h8, F.w8, y, x, v[ci]);
    float* dst = out + (size_t)F.off * COUT + c;
#pragma unroll 1
    for (int co = 0; co < COUT; ++co) {
        float acc = b[co];
        const float* k = w + co * CIN * 9;
#pragma unroll
        for (int ci = 0; ci < CIN; ++ci)
#pragma unroll
            for (int t = 0; t < 9; ++t) acc = __builtin_fmaf(k[ci * 9 + t], v[ci][t], acc);
        if (relu) acc = fmaxf(acc, 0.f);
        dst[(size_t)co * plane] = acc;
    }
}

// Weighted binary cross-entropy with logits, averaged over n outputs: w_i * softplus(-z)
// for a positive label, softplus(z) for a negative one, w_i = pos_weight for positives and
// 1 otherwise; dz = w_i (sigmoid(z) - y) / n, written over z. Each workgroup's share of the
// loss goes to part_loss[blockIdx.x], which k_sn_loss adds up (as adds of a float to one
// address the 86,400 shares of 64 frames of 90 x 160 cells took 1.1 ms). The labels of
// output i of a frame lie at its first cell (fo, or fr's) times the slots.
__global__ void __launch_bounds__(256) k_sn_bce(float* __restrict__ z, const unsigned char* __restrict__ labels,
                                                const long long* __restrict__ fo, int frame_outs, int slots,
                                                float* __restrict__ part_loss, int n, float pos_weight)
{
    __shared__ float s_l[4];
    const int i = blockIdx.x * 256 + threadIdx.x;
    float l = 0.f;
    if (i < n) {
        const int f = i / frame_outs;
        const float zi = z[i];
        const bool pos = labels[fo ? (size_t)fo[f] * slots + (i - f * frame_outs) : (size_t)i] != 0;
        const float wi = pos ? pos_weight : 1.f;
        const float sp = fmaxf(zi, 0.f) + log1pf(expf(-fabsf(zi)));      // softplus(z)
        l = wi * (pos ? sp - zi : sp);
        const float sg = 1.f / (1.f + expf(-zi));
        z[i] = wi * (sg - (pos ? 1.f : 0.f)) / (float)n;
    }
    for (int off = 32; off > 0; off >>= 1) l += __shfl_xor(l, off, 64);
    if ((threadIdx.x & 63) == 0) s_l[threadIdx.x >> 6] = l;
    __syncthreads();
    if (threadIdx.x == 0) part_loss[blockIdx.x] = (s_l[0] + s_l[1] + s_l[2] + s_l[3]) / (float)n;
}

// The losses of several training steps, one workgroup each: the step's n shares added one
// after the other in single precision. The loss has always been such a sum (of adds to one
// address, in the order in which they came), whose rounding is 1e-6 of the loss with 5,000
// shares and 7e-5 with 86,400. A sum without that rounding (6e-8) lies that far from the
// losses which earlier versions report for the same training, so this kernel keeps the
// running sum and gives it a fixed order. Gradients do not depend on it. Bound by the chain
// of dependent adds, 2.5 ns each; the shares come through LDS, SN_LOSS at a time.
constexpr int SN_LOSS = 8192;
__global__ void __launch_bounds__(256) k_sn_loss(const float* __restrict__ part_loss, size_t n,
                                                 float* __restrict__ loss)
{
    __shared__ __align__(16) float s[SN_LOSS];
    const float* src = part_loss + (size_t)blockIdx.x * n;
    float a = 0.f;
    for (size_t i0 = 0; i0 < n; i0 += SN_LOSS) {
        const int m = (int)min((size_t)SN_LOSS, n - i0);
        __syncthreads();
        for (int i = threadIdx.x; i < SN_LOSS; i += 256) s[i] = i < m ? src[i0 + i] : 0.f;
        __syncthreads();
        if (threadIdx.x < 64) {
            // (the zeros past the last share leave the sum, which is not negative, as it is)
            const float4* q = reinterpret_cast<const float4*>(s);
#pragma unroll 16
            for (int i = 0; i < (m + 3) / 4; ++i) {
                const float4 v = q[i];
                a = a + v.x;
                a = a + v.y;
                a = a + v.z;
                a = a + v.w;
            }
        }
    }
    if (threadIdx.x == 0) loss[blockIdx.x] = a;
}

// Gradient of the loss with respect to the layer input: gin[f][ci][y][x] =
// sum_{co,ky,kx} gpre[f][co][y-ky+1][x-kx+1] w[co][ci][ky][kx], times the ReLU mask of the
// input (act_in > 0). One thread per position computes all CIN inputs: each gradient value
// of its neighbourhood is loaded once for all of them (a thread per position and input
// channel loaded it CIN times and was bound by those loads), with the next channel's
// nine loads in flight while the FMAs of this one run; the weights are SGPR operands. The
// two layers of 64 frames of 90 x 160 cells: 1,247 -> 119 us.
template <int CIN, int COUT>
__global__ void __launch_bounds__(256) k_sn_conv_bwd_data(const float* __restrict__ gpre, const float* __restrict__ w,
                                                          const float* __restrict__ act_in, float* __restrict__ gin,
                                                          const SnFrame* __restrict__ fr, int nf, int total)
{
    const int pos = blockIdx.x * 256 + threadIdx.x;
    if (pos >= total) return;
    const int f = sn_frame_of(fr, nf, pos);
    const SnFrame F = fr[f];
    const int c = pos - F.pos_off;
    const int y = c / F.w8, x = c - y * F.w8;
    const int plane = F.h8 * F.w8;
    const float* g = gpre + (size_t)F.off * COUT;
    float acc[CIN], v[9];
#pragma unroll
    for (int ci = 0; ci < CIN; ++ci) acc[ci] = 0.f;
    sn_window(g, F.h8, F.w8, y, x, v);
#pragma unroll 1
    for (int co = 0; co < COUT; ++co) {
        float nv[9];
        sn_window(g + (size_t)min(co + 1, COUT - 1) * plane, F.h8, F.w8, y, x, nv);
        const float* k = w + co * CIN * 9;
        // tap (ky, kx) reads (y - ky + 1, x - kx + 1): the neighbourhood backwards
#pragma unroll
        for (int ci = 0; ci < CIN; ++ci)
#pragma unroll
            for (int t = 0; t < 9; ++t) acc[ci] = __builtin_fmaf(k[ci * 9 + t], v[8 - t], acc[ci]);
#pragma unroll
        for (int t = 0; t < 9; ++t) v[t] = nv[t];
    }
    const size_t o = (size_t)F.off * CIN + c;
#pragma unroll
    for (int ci = 0; ci < CIN; ++ci) gin[o + (size_t)ci * plane] = act_in[o + (size_t)ci * plane] > 0.f ? acc[ci] : 0.f;
}

// Weight and bias gradients of one layer, dw[co][ci][k] = sum over positions of gpre[co]
// times in[ci] at the tap's offset, db[co] = sum of gpre[co]: the product of the COUT x
// positions matrix of gradients and the positions x (9 CIN + 1) matrix of inputs (the last
// column ones, for the biases), on v_mfma_f32_16x16x4_f32 (FP32 products and sums). A
// workgroup takes tiles of SN_TR rows x SN_TC columns of a frame in turn: both operands
// are staged in LDS (gradients zero outside the frame, inputs with a border of one), and
// each wave multiplies one row, four positions per MFMA, one operand value per lane. The
// waves' sums meet in LDS and go to part[blockIdx.x][co][9 CIN + 1]; k_sn_update adds the
// workgroups' sums in a fixed order. (One thread per position and (co, ci) pair read the
// inputs COUT times and the gradients CIN times: the three layers of 64 frames of 90 x 160
// cells 1,568 -> 181 us.) Four workgroups fit a CU's LDS, so 1024 fill the chip: 97 us for
// 8 -> 24 channels against 146 with 512.
constexpr int SN_TR = 4, SN_TC = 64;
constexpr int SN_WGS = 1024;           // workgroups at most (rows of the partial sums)
typedef float sn_f4 __attribute__((ext_vector_type(4)));

template <int CIN, int COUT>
__global__ void __launch_bounds__(256) k_sn_conv_bwd_w(const float* __restrict__ gpre, const float* __restrict__ in,
                                                       const SnFrame* __restrict__ fr,
                                                       const long long* __restrict__ fo, int h8, int w8, int tiles_x,
                                                       int tiles_y, int ntiles, float* __restrict__ part)
{
    constexpr int NC = CIN * 9 + 1, MT = (COUT + 15) / 16, NT = (NC + 15) / 16;
    constexpr int IR = SN_TR + 2, IC = SN_TC + 2;
    constexpr int IS = IR * IC + 1, GS = SN_TR * SN_TC + 1;      // odd channel strides
    constexpr int NE = COUT * NC;
    constexpr int SZ = CIN * IS + COUT * GS > 4 * NE ? CIN * IS + COUT * GS : 4 * NE;
    __shared__ float s[SZ];
    float* const s_in = s;
    float* const s_g = s + CIN * IS;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int q = lane & 15, kk = lane >> 4;
    const int plane = h8 * w8;
    // this lane's operand positions: gradient row (channel) and input column (tap)
    int ga[MT], ia[NT];
    bool gok[MT], iok[NT];
    float ib[NT];
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        const int co = 16 * m + q;
        gok[m] = co < COUT;
        ga[m] = min(co, COUT - 1) * GS + wave * SN_TC + kk;
    }
#pragma unroll
    for (int n = 0; n < NT; ++n) {
        const int col = 16 * n + q, cc = min(col, NC - 2), ci = cc / 9, t = cc - ci * 9;
        iok[n] = col < NC - 1;
        ib[n] = col == NC - 1 ? 1.f : 0.f;
        ia[n] = ci * IS + (wave + t / 3) * IC + t % 3 + kk;
    }
    sn_f4 acc[MT][NT];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int n = 0; n < NT; ++n) acc[m][n] = sn_f4{0.f, 0.f, 0.f, 0.f};
    for (int tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        const int f = tile / (tiles_x * tiles_y), tt = tile - f * tiles_x * tiles_y;
        const int y0 = (tt / tiles_x) * SN_TR, x0 = (tt % tiles_x) * SN_TC;
        const float* gs = gpre + (size_t)fr[f].off * COUT;
        const float* is = in + (size_t)(fo ? fo[f] : fr[f].off) * CIN;
        __syncthreads();
        for (int i = tid; i < COUT * SN_TR * SN_TC; i += 256) {
            const int co = i / (SN_TR * SN_TC), p = i - co * (SN_TR * SN_TC);
            const int y = y0 + p / SN_TC, x = x0 + p % SN_TC;
            s_g[co * GS + p] = (y < h8 && x < w8) ? gs[(size_t)co * plane + y * w8 + x] : 0.f;
        }
        for (int i = tid; i < CIN * IR * IC; i += 256) {
            const int ci = i / (IR * IC), p = i - ci * (IR * IC);
            const int y = y0 + p / IC - 1, x = x0 + p % IC - 1;
            s_in[ci * IS + p] = (y >= 0 && y < h8 && x >= 0 && x < w8) ? is[(size_t)ci * plane + y * w8 + x] : 0.f;
        }
        __syncthreads();
#pragma unroll 4
        for (int p = 0; p < SN_TC; p += 4) {
            float a[MT], b[NT];
#pragma unroll
            for (int m = 0; m < MT; ++m) a[m] = gok[m] ? s_g[ga[m] + p] : 0.f;
#pragma unroll
            for (int n = 0; n < NT; ++n) b[n] = iok[n] ? s_in[ia[n] + p] : ib[n];
#pragma unroll
            for (int m = 0; m < MT; ++m)
#pragma unroll
                for (int n = 0; n < NT; ++n)
                    acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[m], b[n], acc[m][n], 0, 0, 0);
        }
    }
    // lane (q, kk) holds rows 4 kk + r, column q of each product
    __syncthreads();
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int co = 16 * m + 4 * kk + r, col = 16 * n + q;
                if (co < COUT && col < NC) s[wave * NE + co * NC + col] = acc[m][n][r];
            }
    __syncthreads();
    for (int i = tid; i < NE; i += 256)
        part[(size_t)blockIdx.x * NE + i] = (s[i] + s[NE + i]) + (s[2 * NE + i] + s[3 * NE + i]);
}

// The end of a training step: every gradient from the workgroups' partial sums of the
// three layers (part: [rows][cout * (9 cin + 1)] per layer, rows = wgs), in a fixed order;
// then, with m, one Adam step (Kingma & Ba, 2015, with bias correction). 64 parameters per
// workgroup, 16 threads each.
struct SnLayerGrad {
    const float* part;
    int cin, cout, o_w, o_b;      // parameter offsets of the layer's weights and biases
};
struct SnGrads {
    SnLayerGrad l[3];
};

__global__ void __launch_bounds__(1024) k_sn_update(SnGrads G, int wgs, float* __restrict__ grad,
                                                    float* __restrict__ p, float* __restrict__ m,
                                                    float* __restrict__ v, float lr, float b1, float b2, float eps,
                                                    int t)
{
    __shared__ float s[16][64];
    const int lane = threadIdx.x & 63, row = threadIdx.x >> 6;
    // element i of the layers' partial sums back to back
    const int i = blockIdx.x * 64 + lane;
    int k = 0, e = i, ne = 0, nc = 1;
    for (; k < 3; ++k) {
        nc = 9 * G.l[k].cin + 1;
        ne = G.l[k].cout * nc;
        if (e < ne) break;
        e -= ne;
    }
    float a = 0.f;
    if (k < 3) {
        const float* src = G.l[k].part + e;
#pragma unroll 8
        for (int r = row; r < wgs; r += 16) a += src[(size_t)r * ne];
    }
    s[row][lane] = a;
    __syncthreads();
    if (row != 0 || k >= 3) return;
    float g = 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) g += s[r][lane];
    const int co = e / nc, col = e - co * nc;
    const int o = col < nc - 1 ? G.l[k].o_w + co * (nc - 1) + col : G.l[k].o_b + co;
    grad[o] = g;
    if (!m) return;
    const float mi = b1 * m[o] + (1.f - b1) * g;
    const float vi = b2 * v[o] + (1.f - b2) * g * g;
    m[o] = mi;
    v[o] = vi;
    const float mh = mi / (1.f - powf(b1, (float)t)), vh = vi / (1.f - powf(b2, (float)t));
    p[o] -= lr * mh / (sqrtf(vh) + eps);
}

// Keep flag of every response tile of a batch: the largest logit of the slots within
// `srad` of L.scl over the frame cells that hold the centres of the tile's windows (level
// position 4 * x + 11.5, 4 * y + 13.5, divided by the scale), widened by `margin` cells,
// against the logit threshold of slot L.scl. Levels whose scale index has no slot are kept. One wave
// per tile: the lanes share the tile's (slot, cell) pairs and reduce their maxima.
__global__ void __launch_bounds__(256) k_sn_tile_mask(const LevelDesc* __restrict__ levels, int nlevels, int ntiles,
                                                      int TX, int TY, const float* __restrict__ logits,
                                                      const SnFrame* __restrict__ fr, SkipThresholds th, int srad,
                                                      int margin,
                                                      unsigned char* __restrict__ keep)
{
    const int t = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (t >= ntiles) return;
    int lo = 0, hi = nlevels - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (levels[mid].tile_off <= t) lo = mid; else hi = mid - 1;
    }
    const LevelDesc& L = levels[lo];
    int k = 1;
    // levels of scale < 0.5 are cheap (their pixel count falls with the square of the
    // scale) and their tiles span many cells: they always run
    if (L.scl < CCNN_SKIP_SLOTS && L.scale >= 0.5f) {
        const int tt = t - L.tile_off;
        const int tx = tt % L.tiles_x, ty = tt / L.tiles_x;
        const SnFrame F = fr[L.frame];
        // responses of the tile: x in [x0, x1), y in [y0, y1)
        const int x0 = tx * TX, x1 = min(x0 + TX, L.rw), y0 = ty * TY, y1 = min(y0 + TY, L.rh);
        const float inv = 1.f / (8.f * L.scale);
        const int u0 = max(0, (int)floorf((4.f * x0 + 11.5f) * inv) - margin);
        const int u1 = min(F.w8 - 1, (int)floorf((4.f * (x1 - 1) + 11.5f) * inv) + margin);
        const int v0 = max(0, (int)floorf((4.f * y0 + 13.5f) * inv) - margin);
        const int v1 = min(F.h8 - 1, (int)floorf((4.f * (y1 - 1) + 13.5f) * inv) + margin);
        const int s0 = max(0, L.scl - srad), s1 = min(CCNN_SKIP_SLOTS - 1, L.scl + srad);
        const size_t plane = (size_t)F.h8 * F.w8;
        const float* z = logits + (size_t)F.off * CCNN_SKIP_SLOTS + (size_t)s0 * plane;
        const int nu = u1 - u0 + 1, nv = v1 - v0 + 1;
        // a tile whose window centres fall outside the cell grid has no logit: it runs
        if (nu > 0 && nv > 0) {
            const int n = nu * nv, ns = s1 - s0 + 1;
            float mz = -INFINITY;
            for (int i = lane; i < n * ns; i += 64) {
                const int sl = i / n, c = i - sl * n;
                const int v = v0 + c / nu, u = u0 + c % nu;
                mz = fmaxf(mz, z[sl * plane + (size_t)v * F.w8 + u]);
            }
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) mz = fmaxf(mz, __shfl_xor(mz, off, 64));
            k = mz >= th.zt[L.scl];
        }
    }
    if (lane == 0) keep[t] = (unsigned char)k;
}

// Keep flag of every L1 tile: set when a kept response tile of its level reads it (the
// response tile (tx, ty) of TX x TY responses reads pooled L1 columns [2 TX tx, 2 TX tx +
// 2 TX + 8) and rows [2 TY ty, 2 TY ty + 2 TY + 10)).
__global__ void __launch_bounds__(256) k_sn_l1_mask(const LevelDesc* __restrict__ levels, int nlevels, int nl1tiles,
                                                    int ax, int ay, int tx_, int ty_,
                                                    const unsigned char* __restrict__ keep,
                                                    unsigned char* __restrict__ l1_keep)
{
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t >= nl1tiles) return;
    int lo = 0, hi = nlevels - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (levels[mid].l1_tile_off <= t) lo = mid; else hi = mid - 1;
    }
    const LevelDesc& L = levels[lo];
    const int tt = t - L.l1_tile_off;
    const int X0 = (tt % L.l1_tiles_x) * ax, Y0 = (tt / L.l1_tiles_x) * ay;
    // response tiles whose L1 window meets [X0, X0 + ax) x [Y0, Y0 + ay)
    const int rx0 = max(0, (X0 - (2 * tx_ + 8) + 1 + 2 * tx_ - 1) / (2 * tx_));
    const int rx1 = min(L.tiles_x - 1, (X0 + ax - 1) / (2 * tx_));
    const int ry0 = max(0, (Y0 - (2 * ty_ + 10) + 1 + 2 * ty_ - 1) / (2 * ty_));
    const int ry1 = min(L.tiles_y - 1, (Y0 + ay - 1) / (2 * ty_));
    int k = 0;
    for (int ry = ry0; ry <= ry1 && !k; ++ry)
        for (int rx = rx0; rx <= rx1 && !k; ++rx) k = keep[L.tile_off + ry * L.tiles_x + rx];
    l1_keep[t] = (unsigned char)k;
}

namespace {

constexpr int S = CCNN_SKIP_SLOTS;
// parameter layout: w1 [8][1][9], b1 [8], w2 [8][8][9], b2 [8], w3 [S][8][9], b3 [S]
constexpr int oW1 = 0, oB1 = oW1 + 8 * 9, oW2 = oB1 + 8, oB2 = oW2 + 8 * 8 * 9, oW3 = oB2 + 8, oB3 = oW3 + S * 8 * 9;
constexpr int NPAR = oB3 + S;
static_assert(NPAR == CCNN_SKIP_PARAMS, "parameter count");

template <class T>
struct DBuf {
    T* p = nullptr;
    ~DBuf() { if (p) (void)hipFree(p); }
    bool alloc(size_t n) { return hipMalloc((void**)&p, sizeof(T) * (n > 0 ? n : 1)) == hipSuccess; }
};

#define SN_OK(expr)                                                                          \
    do {                                                                                     \
        hipError_t e_ = (expr);                                                              \
        if (e_ != hipSuccess) {                                                              \
            note_error(e_);                                                                  \
            std::fprintf(stderr, "[ccnn] HIP error %s at %s:%d\n", hipGetErrorString(e_),     \
                         __FILE__, __LINE__);                                                \
            return -1;                                                                       \
        }                                                                                    \
    } while (0)

// Device state of one training or gradient run over frames of one size h8 x w8: one
// allocation, carved into the buffers.
struct SnRun {
    static constexpr int KEEP = 64;       // steps whose loss shares are kept at most
    int n = 0, h8 = 0, w8 = 0, total = 0, tiles_x = 0, tiles_y = 0, wgs = 0, keep = 0;
    size_t nloss = 0;                     // loss shares of a step
    DBuf<char> arena;
    SnFrame* fr = nullptr;
    float *a1 = nullptr, *a2 = nullptr, *dz = nullptr, *g2 = nullptr, *g1 = nullptr, *par = nullptr, *grad = nullptr,
          *m = nullptr, *v = nullptr, *loss = nullptr, *part = nullptr, *part_loss = nullptr;

    // steps: the run's steps
    int init(int n_, int h8_, int w8_, long long steps)
    {
        n = n_; h8 = h8_; w8 = w8_;
        total = n * h8 * w8;
        tiles_x = (w8 + SN_TC - 1) / SN_TC;
        tiles_y = (h8 + SN_TR - 1) / SN_TR;
        wgs = (int)std::min<long long>(SN_WGS, (long long)n * tiles_x * tiles_y);
        nloss = ((size_t)total * S + 255) / 256;
        keep = (int)std::min<long long>(KEEP, std::max<long long>(steps, 1));
        std::vector<SnFrame> f(n);
        for (int i = 0; i < n; ++i) f[i] = SnFrame{h8, w8, i * h8 * w8, i * h8 * w8};
        const size_t P = (size_t)total;
        size_t bytes = 0;
        auto carve = [&](auto*& p, size_t count) {
            if (arena.p) p = reinterpret_cast<std::remove_reference_t<decltype(p)>>(arena.p + bytes);
            bytes += (sizeof(*p) * count + 255) / 256 * 256;
        };
        for (int pass = 0; pass < 2; ++pass) {
            bytes = 0;
            carve(fr, n);
            carve(a1, 8 * P); carve(a2, 8 * P); carve(dz, S * P); carve(g2, 8 * P); carve(g1, 8 * P);
            carve(par, NPAR); carve(grad, NPAR); carve(m, NPAR); carve(v, NPAR); carve(loss, keep);
            carve(part, (size_t)wgs * NPAR); carve(part_loss, nloss * keep);
            if (pass == 0 && !arena.alloc(bytes)) return -1;
        }
        SN_OK(hipMemcpy(fr, f.data(), sizeof(SnFrame) * n, hipMemcpyHostToDevice));
        return 0;
    }
    // forward and backward over n frames of x / y (fo: their first cells there, or null when
    // they are the first n): the gradients, the loss shares of step k of the kept ones, and
    // with t > 0 the t-th Adam update of the parameters
    int step(const float* x, const unsigned char* y, const long long* fo, float pos_weight, int k, float lr, int t)
    {
        const int T = total;
        const unsigned blocks = (unsigned)((T + 255) / 256);
        k_sn_conv<1, 8><<<blocks, 256>>>(x, par + oW1, par + oB1, a1, fr, fo, n, T, 1);
        k_sn_conv<8, 8><<<blocks, 256>>>(a1, par + oW2, par + oB2, a2, fr, nullptr, n, T, 1);
        k_sn_conv<8, S><<<blocks, 256>>>(a2, par + oW3, par + oB3, dz, fr, nullptr, n, T, 0);
        k_sn_bce<<<(unsigned)nloss, 256>>>(dz, y, fo, h8 * w8 * S, S, part_loss + nloss * k, T * S, pos_weight);
        SnGrads G;
        float* p = part;
        const int nt = n * tiles_x * tiles_y;
        G.l[0] = SnLayerGrad{p, 8, S, oW3, oB3};
        k_sn_conv_bwd_w<8, S><<<wgs, 256>>>(dz, a2, fr, nullptr, h8, w8, tiles_x, tiles_y, nt, p);
        p += (size_t)wgs * S * 73;
        k_sn_conv_bwd_data<8, S><<<blocks, 256>>>(dz, par + oW3, a2, g2, fr, n, T);
        G.l[1] = SnLayerGrad{p, 8, 8, oW2, oB2};
        k_sn_conv_bwd_w<8, 8><<<wgs, 256>>>(g2, a1, fr, nullptr, h8, w8, tiles_x, tiles_y, nt, p);
        p += (size_t)wgs * 8 * 73;
        k_sn_conv_bwd_data<8, 8><<<blocks, 256>>>(g2, par + oW2, a1, g1, fr, n, T);
        G.l[2] = SnLayerGrad{p, 1, 8, oW1, oB1};
        k_sn_conv_bwd_w<1, 8><<<wgs, 256>>>(g1, x, fr, fo, h8, w8, tiles_x, tiles_y, nt, p);
        k_sn_update<<<(NPAR + 63) / 64, 1024>>>(G, wgs, grad, par, t > 0 ? m : nullptr, v, lr, 0.9f, 0.999f, 1e-8f, t);
        SN_OK(hipGetLastError());
        return 0;
    }
    // the losses of the first `steps` kept steps, on the host
    int losses(int steps, float* out)
    {
        k_sn_loss<<<steps, 256>>>(part_loss, nloss, loss);
        SN_OK(hipGetLastError());
        SN_OK(hipMemcpy(out, loss, sizeof(float) * steps, hipMemcpyDeviceToHost));
        return 0;
    }
};

}  // namespace

hipError_t launch_skipnet(const float* gray, const FrameDesc* ft, const SnFrame* fr, int nf, int cells,
                          const float* par, float* x0, float* a1, float* a2, float* z, const LevelDesc* levels, int nl,
                          int ntiles, int nl1tiles, int shape, const float* threshold, int srad, int margin,
                          unsigned char* keep, unsigned char* l1_keep, hipStream_t st)
{
    if (cells <= 0 || ntiles <= 0) return hipSuccess;
    const TileShape t = tile_shape(shape);
    SkipThresholds th;
    for (int k = 0; k < CCNN_SKIP_SLOTS; ++k) th.zt[k] = std::log(threshold[k] / (1.f - threshold[k]));
    auto blocks = [](long long k) { return (unsigned)((k + 255) / 256); };
    k_sn_down8<<<blocks(cells), 256, 0, st>>>(gray, ft, fr, nf, cells, x0);
    k_sn_conv<1, 8><<<blocks(cells), 256, 0, st>>>(x0, par + oW1, par + oB1, a1, fr, nullptr, nf, cells, 1);
    k_sn_conv<8, 8><<<blocks(cells), 256, 0, st>>>(a1, par + oW2, par + oB2, a2, fr, nullptr, nf, cells, 1);
    k_sn_conv<8, S><<<blocks(cells), 256, 0, st>>>(a2, par + oW3, par + oB3, z, fr, nullptr, nf, cells, 0);
    k_sn_tile_mask<<<(unsigned)((ntiles + 3) / 4), 256, 0, st>>>(levels, nl, ntiles, t.tx, t.ty, z, fr, th, srad, margin, keep);
    k_sn_l1_mask<<<blocks(nl1tiles), 256, 0, st>>>(levels, nl, nl1tiles, t.ax, t.ay, t.tx, t.ty, keep, l1_keep);
    return hipGetLastError();
}

}  // namespace ccnn

using namespace ccnn;

extern "C" int ccnn_skipnet_grad(const float* params, const float* x0, const unsigned char* labels, int n, int h8,
                                 int w8, float pos_weight, float* grad, float* loss)
{
    if (!params || !x0 || !labels || !grad || n <= 0 || h8 <= 0 || w8 <= 0) return -1;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0) return -1;
    SnRun r;
    if (r.init(n, h8, w8, 1) < 0) return -1;
    const size_t P = (size_t)n * h8 * w8;
    DBuf<float> x;
    DBuf<unsigned char> y;
    if (!x.alloc(P) || !y.alloc(S * P)) return -1;
    SN_OK(hipMemcpy(r.par, params, sizeof(float) * NPAR, hipMemcpyHostToDevice));
    SN_OK(hipMemcpy(x.p, x0, sizeof(float) * P, hipMemcpyHostToDevice));
    SN_OK(hipMemcpy(y.p, labels, S * P, hipMemcpyHostToDevice));
    if (r.step(x.p, y.p, nullptr, pos_weight, 0, 0.f, 0) < 0) return -1;
    SN_OK(hipDeviceSynchronize());
    SN_OK(hipMemcpy(grad, r.grad, sizeof(float) * NPAR, hipMemcpyDeviceToHost));
    return loss ? r.losses(1, loss) : 0;
}

extern "C" int ccnn_skipnet_forward(const float* params, const float* x0, int n, int h8, int w8, float* logits)
{
    if (!params || !x0 || !logits || n <= 0 || h8 <= 0 || w8 <= 0) return -1;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0) return -1;
    SnRun r;
    if (r.init(n, h8, w8, 1) < 0) return -1;
    const size_t P = (size_t)n * h8 * w8;
    DBuf<float> x;
    if (!x.alloc(P)) return -1;
    SN_OK(hipMemcpy(r.par, params, sizeof(float) * NPAR, hipMemcpyHostToDevice));
    SN_OK(hipMemcpy(x.p, x0, sizeof(float) * P, hipMemcpyHostToDevice));
    const int T = r.total;
    // (the logits go where a training step keeps their gradients)
    k_sn_conv<1, 8><<<(T + 255) / 256, 256>>>(x.p, r.par + oW1, r.par + oB1, r.a1, r.fr, nullptr, n, T, 1);
    k_sn_conv<8, 8><<<(T + 255) / 256, 256>>>(r.a1, r.par + oW2, r.par + oB2, r.a2, r.fr, nullptr, n, T, 1);
    k_sn_conv<8, S><<<(T + 255) / 256, 256>>>(r.a2, r.par + oW3, r.par + oB3, r.dz, r.fr, nullptr, n, T, 0);
    SN_OK(hipGetLastError());
    SN_OK(hipDeviceSynchronize());
    SN_OK(hipMemcpy(logits, r.dz, sizeof(float) * S * P, hipMemcpyDeviceToHost));
    return 0;
}

extern "C" int ccnn_skipnet_train(float* params, const float* x0, const unsigned char* labels, int n, int h8, int w8,
                                  int epochs, int batch, float lr, float pos_weight, unsigned seed,
                                  float* epoch_loss)
{
    if (!params || !x0 || !labels || n <= 0 || h8 <= 0 || w8 <= 0 || epochs <= 0 || batch <= 0) return -1;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0) return -1;
    batch = std::min(batch, n);
    const int nb = n / batch;                   // steps per epoch
    SnRun r;
    if (r.init(batch, h8, w8, epoch_loss ? (long long)epochs * nb : 1) < 0) return -1;
    const size_t F = (size_t)h8 * w8;
    // the whole set on the device, with the frames' order of an epoch: the kernels read a
    // step's frames where they lie in the set
    DBuf<float> all_x;
    DBuf<unsigned char> all_y;
    DBuf<long long> fo;
    if (!all_x.alloc(F * n) || !all_y.alloc(S * F * n) || !fo.alloc(n)) return -1;
    SN_OK(hipMemcpy(all_x.p, x0, sizeof(float) * F * n, hipMemcpyHostToDevice));
    SN_OK(hipMemcpy(all_y.p, labels, S * F * n, hipMemcpyHostToDevice));
    SN_OK(hipMemcpy(r.par, params, sizeof(float) * NPAR, hipMemcpyHostToDevice));
    SN_OK(hipMemset(r.m, 0, sizeof(float) * NPAR));
    SN_OK(hipMemset(r.v, 0, sizeof(float) * NPAR));
    std::vector<int> order(n);
    for (int i = 0; i < n; ++i) order[i] = i;
    std::vector<long long> off(n);
    // the losses of the last `kept` steps are still on the device; the epochs whose steps
    // have all been read are written as the run goes on
    int kept = 0, read = 0, done = 0;
    double lsum = 0.0;
    auto read_losses = [&]() {
        float l[SnRun::KEEP];
        if (r.losses(kept, l) < 0) return -1;
        for (int k = 0; k < kept; ++k) {
            lsum += l[k];
            if (++read < nb) continue;
            epoch_loss[done++] = (float)(lsum / nb);
            read = 0;
            lsum = 0.0;
        }
        kept = 0;
        return 0;
    };
    unsigned long long st = seed * 6364136223846793005ull + 1442695040888963407ull;
    auto rnd = [&]() {
        st = st * 6364136223846793005ull + 1442695040888963407ull;
        return (unsigned)(st >> 33);
    };
    int t = 0;
    for (int e = 0; e < epochs; ++e) {
        for (int i = n - 1; i > 0; --i) std::swap(order[i], order[rnd() % (unsigned)(i + 1)]);
        for (int i = 0; i < n; ++i) off[i] = (long long)F * order[i];
        SN_OK(hipMemcpy(fo.p, off.data(), sizeof(long long) * n, hipMemcpyHostToDevice));
        for (int b = 0; b < nb; ++b) {
            ++t;
            if (r.step(all_x.p, all_y.p, fo.p + (size_t)b * batch, pos_weight, kept, lr, t) < 0) return -1;
            if (epoch_loss && ++kept == r.keep && read_losses() < 0) return -1;
        }
    }
    if (kept > 0 && read_losses() < 0) return -1;
    SN_OK(hipDeviceSynchronize());
    SN_OK(hipMemcpy(params, r.par, sizeof(float) * NPAR, hipMemcpyDeviceToHost));
    return 0;
}
