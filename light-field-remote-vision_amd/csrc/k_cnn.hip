// Kernels of the warm-start CNN: 3x3 convolutions on the bf16 MFMA units of
// CDNA4 with FP32 accumulation, their backward passes, and the elementwise
// pieces of a U-Net (2x2 average pooling, nearest 2x upsampling, ReLU, the
// squared-error loss, Adam).  No counterpart in the reference (its CNN
// training, sources/CNN/, is a separate TensorFlow tool outside this path).
//
// Layouts.  Activations are NHWC bf16: [B][H][W][C], channels contiguous.
// Weights are [Cout][9][Cin] bf16 (tap t = 3 (dy + 1) + (dx + 1)), so one
// output channel's weights are contiguous along K = 9 Cin.  Gradients of
// activations and weights are FP32.  Input channel counts are multiples of
// 32 (the first layer's are zero-padded), so a K chunk of 32 never straddles
// a tap.
//
// The convolution is an implicit GEMM: C[cout][pixel] = sum_k W[cout][k]
// A[k][pixel] with A[(t, ci)][p] = X[p + offset(t)][ci] (0 outside the image),
// by chunk of 32 input channels over a 2-D pixel tile whose halo serves all 9
// taps (v_mfma_f32_16x16x32_bf16).  Skips, ReLU, pooling, upsampling and the
// prediction ride on its loads and its epilogue.  The backward pass with
// respect to the input is the same kernel on the output gradient with the
// weights flipped in space and transposed in channels; the weight gradient is
// another MFMA kernel whose K runs over pixels.
#include "lfrv_internal.hpp"
#include "tile_common.hpp"

#include <algorithm>
#include <climits>

namespace lfrv {

typedef short s4v __attribute__((ext_vector_type(4)));
typedef float f4v __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint16_t f2bf(float f)
{
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return 0x7fc0;  // NaN stays NaN
    u += 0x7fffu + ((u >> 16) & 1u);                      // round to nearest even
    return (uint16_t)(u >> 16);
}

__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

constexpr int kCvBK = 32, kCvPitch = 40;  // LDS rows of 40 bf16 (80 B, 16-byte aligned)

typedef __bf16 bf8v __attribute__((ext_vector_type(8)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

typedef unsigned short u16x4 __attribute__((ext_vector_type(4)));

// What a convolution does with its sums (CnnConv, lfrv_internal.hpp).  The
// fused forms leave no elementwise pass of the network outside the
// convolutions: what each replaced read and wrote the activations (or their
// FP32 gradients) once more.
template <int EPI>
__device__ __forceinline__ void conv_epilogue(const CnnConv &a, f4v (&v)[4], int img, int y, int x, int co)
{
    // v[i]: channels co .. co + 3 of pixel (y + i, x); y is a multiple of 4, x of this lane: lane & 1
    const bool xin = x < a.W && co < a.Cout;
    if constexpr (EPI == CNN_F32) {
        float *Y = (float *)a.Y;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            if (!xin || y + i >= a.H) continue;
            const size_t o = ((size_t)(img * a.H + y + i) * a.W + x) * a.Cout + co;
            if (a.vec) *(f4v *)(Y + o) = v[i];
            else
                for (int r = 0; r < 4; r++)
                    if (co + r < a.Cout) Y[o + r] = v[i][r];
        }
    } else if constexpr (EPI == CNN_HEAD) {
        const size_t HW = (size_t)a.H * a.W;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            if (!xin || y + i >= a.H || co != 0) continue;
#pragma unroll
            for (int r = 0; r < 3; r++) {
                const size_t o = ((size_t)img * 3 + r) * HW + (size_t)(y + i) * a.W + x;
                ((float *)a.Y)[o] = a.base[o] + v[i][r];
            }
        }
    } else if constexpr (EPI == CNN_FWD) {
        u16x4 h[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const bool in = xin && y + i < a.H;
            const size_t o = in ? ((size_t)(img * a.H + y + i) * a.W + x) * a.Cout + co : 0;
            if (a.aux) {
                const u16x4 sk = *(const u16x4 *)(a.aux + o);
#pragma unroll
                for (int r = 0; r < 4; r++) v[i][r] += bf2f(sk[r]);
            }
#pragma unroll
            for (int r = 0; r < 4; r++) h[i][r] = f2bf(a.relu ? fmaxf(v[i][r], 0.0f) : v[i][r]);
            if (in) *(u16x4 *)((uint16_t *)a.Y + o) = h[i];
        }
        if (a.pool) {  // (H and W even: a pair of rows and of lanes is whole)
#pragma unroll
            for (int i = 0; i < 4; i += 2) {
                u16x4 q;
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const float t0 = bf2f(h[i][r]), t1 = bf2f(h[i + 1][r]);
                    q[r] = f2bf(0.25f * ((t0 + __shfl_xor(t0, 1)) + (t1 + __shfl_xor(t1, 1))));
                }
                if (xin && y + i < a.H && !(x & 1))
                    *(u16x4 *)(a.pool + ((size_t)(img * (a.H / 2) + (y + i) / 2) * (a.W / 2) + x / 2) * a.Cout + co) = q;
            }
        }
    } else if constexpr (EPI == CNN_MASK) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            if (!xin || y + i >= a.H) continue;
            const size_t o = ((size_t)(img * a.H + y + i) * a.W + x) * a.Cout + co;
            const u16x4 act = *(const u16x4 *)(a.aux + o);
            u16x4 h;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                if (!(bf2f(act[r]) > 0.0f)) v[i][r] = 0.0f;
                h[r] = f2bf(v[i][r]);
            }
            if (a.dskip) *(f4v *)(a.dskip + o) = v[i];
            *(u16x4 *)((uint16_t *)a.Y + o) = h;
        }
    } else if constexpr (EPI == CNN_MASK_UP) {
#pragma unroll
        for (int i = 0; i < 4; i += 2) {
            float t[4];
#pragma unroll
            for (int r = 0; r < 4; r++)
                t[r] = (v[i][r] + __shfl_xor(v[i][r], 1)) + (v[i + 1][r] + __shfl_xor(v[i + 1][r], 1));
            if (!xin || y + i >= a.H || (x & 1)) continue;
            const size_t o = ((size_t)(img * (a.H / 2) + (y + i) / 2) * (a.W / 2) + x / 2) * a.Cout + co;
            const u16x4 act = *(const u16x4 *)(a.aux + o);
            u16x4 h;
#pragma unroll
            for (int r = 0; r < 4; r++) h[r] = f2bf(bf2f(act[r]) > 0.0f ? t[r] : 0.0f);
            *(u16x4 *)((uint16_t *)a.Y + o) = h;
        }
    } else {  // CNN_MASK_POOL
#pragma unroll
        for (int i = 0; i < 4; i++) {
            if (!xin || y + i >= a.H) continue;
            const size_t o0 = ((size_t)(img * 2 * a.H + 2 * (y + i)) * 2 * a.W + 2 * x) * a.Cout + co;
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const size_t o = o0 + ((size_t)(k >> 1) * 2 * a.W + (k & 1)) * a.Cout;
                const u16x4 act = *(const u16x4 *)(a.aux + o);
                const f4v ds = *(const f4v *)(a.dskip + o);
                u16x4 h;
#pragma unroll
                for (int r = 0; r < 4; r++) h[r] = f2bf(bf2f(act[r]) > 0.0f ? ds[r] + 0.25f * v[i][r] : 0.0f);
                *(u16x4 *)((uint16_t *)a.Y + o) = h;
            }
        }
    }
}

// v[p][co] = sum_{t,ci} W[co][t][ci] X[p + off(t)][ci] + bias[co], then the epilogue EPI.
// A block owns 16 x 16 pixels (a wave 4 rows of 16) and BN = 16 NJ output
// channels.  Per chunk of 32 input channels the tile's 18 x 18 halo and the
// weights of all 9 taps go to LDS once.  The sums run by chunk, in a chunk by
// tap in row order, and take the bias last, whatever NJ: in bf16 the network
// amplifies a sum's last bit, so the order is part of the result.  A wave
// holds the four halo rows that a row of taps meets, three operands each, and
// a row of taps on replaces one of them: 18 + 9 NJ LDS reads for 36 NJ MFMAs
// (reading per tap would be 36 + 9 NJ), so that NJ = 4 is bound by the matrix
// units and not by LDS.  The weights are the MFMA's first operand, so a lane
// ends with 4 consecutive channels of one pixel and stores them at once.  The
// next chunk's (or tile's) loads are in flight while this one is multiplied; a
// block runs through its tiles, and with 32 input channels keeps the weights.
// With up, X is half the image's size and read as its 2x nearest upsampling.
// One image of 1024 x 1024: the forward of 15 layers, with what rides on them,
// 0.79 ms; 1.41 with pooling, upsampling and prediction as passes of their own;
// 8 of 256 x 256 forwards and backwards: the step 1.71 ms against 5.66, of
// which the weight gradient took 2.7.
template <int EPI, int NJ>
__global__ void __launch_bounds__(256, NJ == 4 ? 2 : NJ == 2 ? 3 : 4) k_conv3x3(CnnConv a)
{
    constexpr int FM = 4, TH = 16, TW = 16, HX = TW + 2, HP = HX * (TH + 2), BN = 16 * NJ;
    constexpr int NA = (HP * 4 + 255) / 256, NB = (36 * BN + 255) / 256;
    __shared__ __align__(16) uint16_t As[HP * kCvPitch];
    __shared__ __align__(16) uint16_t Bs[9 * BN * kCvPitch];
    __shared__ __align__(16) float bias[BN];
    const int H = a.H, W = a.W, Cin = a.Cin, Cout = a.Cout;
    const int ntx = (W + TW - 1) / TW, nty = (H + TH - 1) / TH, ntiles = a.B * ntx * nty;
    const int co0 = blockIdx.y * BN;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int ncc = Cin / kCvBK;
    const int Hs = H >> a.up, Ws = W >> a.up;  // X's own size
    // loads always read a valid address; what lies outside is zeroed on its way to LDS
    u32x4 ar[NA], br[NB];
    unsigned amask = 0;
    // (a value that the compiler does not see through: the staging's addresses are formed per chunk and not
    // kept, or spilled, over the whole loop)
    auto own_tid = [&]() {
        int t = tid;
        asm volatile("" : "+v"(t));
        return t;
    };
    auto load = [&](int tile, int cc) {
        const int img = tile / (ntx * nty), trem = tile - img * ntx * nty, ty = trem / ntx, tx = trem - ty * ntx;
        const int tid = own_tid();
        amask = 0;
#pragma unroll
        for (int j = 0; j < NA; j++) {
            const int idx = tid + 256 * j, hp = idx >> 2, hy = hp / HX, hx = hp - hy * HX;
            const int y = ty * TH - 1 + hy, x = tx * TW - 1 + hx;
            const bool in = hp < HP && y >= 0 && y < H && x >= 0 && x < W;
            ar[j] = *(const u32x4 *)(a.X + (in ? ((size_t)(img * Hs + (y >> a.up)) * Ws + (x >> a.up)) * Cin : 0) +
                                     cc * kCvBK + 8 * (idx & 3));
            amask |= (in ? 1u : 0u) << j;
        }
    };
    auto load_weights = [&](int cc) {
        const int tid = own_tid();
#pragma unroll
        for (int j = 0; j < NB; j++) {
            const int idx = tid + 256 * j, t = idx / (4 * BN), r = (idx >> 2) - t * BN;
            const bool in = idx < 36 * BN && co0 + r < Cout;
            const unsigned o = (in ? (unsigned)((co0 + r) * 9 + t) * Cin : 0u) + 8 * (idx & 3);  // (a layer's weights: far under 2^31)
            br[j] = *(const u32x4 *)(a.Wt + cc * kCvBK + o);
        }
    };
    const u32x4 z = {0u, 0u, 0u, 0u};
    auto store = [&](bool weights) {
        const int tid = own_tid();
#pragma unroll
        for (int j = 0; j < NA; j++) {
            const int idx = tid + 256 * j;
            if ((idx >> 2) < HP) *(u32x4 *)(&As[(idx >> 2) * kCvPitch + 8 * (idx & 3)]) = (amask >> j & 1) ? ar[j] : z;
        }
        if (weights)
#pragma unroll
            for (int j = 0; j < NB; j++) {
                const int idx = tid + 256 * j, row = idx >> 2;  // t BN + r
                if (idx < 36 * BN)
                    *(u32x4 *)(&Bs[row * kCvPitch + 8 * (idx & 3)]) = co0 + row % BN < Cout ? br[j] : z;
            }
    };
    const uint16_t *al = As + (wv * FM * HX + (lane & 15)) * kCvPitch + 8 * (lane >> 4);
    const uint16_t *bl = Bs + (lane & 15) * kCvPitch + 8 * (lane >> 4);
    if (tid < BN) bias[tid] = a.bias && co0 + tid < Cout ? a.bias[co0 + tid] : 0.0f;
    bool weights = true;
    load(blockIdx.x, 0);
    load_weights(0);
    for (int tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        f4v acc[NJ][FM];
#pragma unroll
        for (int j = 0; j < NJ; j++)
#pragma unroll
            for (int i = 0; i < FM; i++) acc[j][i] = f4v{0.f, 0.f, 0.f, 0.f};
        for (int cc = 0; cc < ncc; cc++) {
            __syncthreads();  // the former chunk is multiplied out
            store(weights);
            __syncthreads();
            const int nc = cc + 1 < ncc ? cc + 1 : 0, nt = nc ? tile : tile + (int)gridDim.x;
            weights = ncc > 1;
            if (nt < ntiles) {
                load(nt, nc);
                if (weights) load_weights(nc);
            }
            bf8v px[FM][3], w[2][NJ];  // halo row r at px[r % FM]; tap t's weights at w[t % 2]
            auto load_tap = [&](int t) __attribute__((always_inline)) {
#pragma unroll
                for (int j = 0; j < NJ; j++) w[t % 2][j] = *(const bf8v *)(bl + (t * BN + 16 * j) * kCvPitch);
            };
            auto load_row = [&](int r) __attribute__((always_inline)) {
#pragma unroll
                for (int dx = 0; dx < 3; dx++) px[r % FM][dx] = *(const bf8v *)(al + (r * HX + dx) * kCvPitch);
            };
            load_tap(0);
#pragma unroll
            for (int r = 0; r < FM; r++) load_row(r);
#pragma unroll
            for (int t = 0; t < 9; t++) {
                const int dy = t / 3, dx = t % 3;
                if (t < 8) load_tap(t + 1);
                __builtin_amdgcn_sched_barrier(0);  // the next tap's weights in registers, none beyond
#pragma unroll
                for (int i = 0; i < FM; i++)
#pragma unroll
                    for (int j = 0; j < NJ; j++)
                        acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[t % 2][j], px[(i + dy) % FM][dx], acc[j][i], 0, 0, 0);
                if (dx == 2 && dy < 2) load_row(dy + FM);
            }
        }
        const int img = tile / (ntx * nty), trem = tile - img * ntx * nty, ty = trem / ntx, tx = trem - ty * ntx;
#pragma unroll
        for (int j = 0; j < NJ; j++) {
            const f4v b = *(const f4v *)(bias + 16 * j + 4 * (lane >> 4));
#pragma unroll
            for (int i = 0; i < FM; i++) acc[j][i] += b;
            conv_epilogue<EPI>(a, acc[j], img, ty * TH + wv * FM, tx * TW + (lane & 15), co0 + 16 * j + 4 * (lane >> 4));
        }
    }
}

// Weight and bias gradient, split over pixels:
//   dW[co][t][ci] += sum_p dU[p][co] X[p + off(t)][ci],  db[co] += sum_p dU[p][co].
// GEMM with M = co, N = (tap, ci), K = pixels.  A block owns BCO x BCI output
// and input channels and all 9 taps, so one staging of dU and of X with its
// halo serves 9 BCO BCI products per pixel.  The pixels go in 8 x 8 cells; a
// stage is four cells, one for each 16-lane group of an MFMA operand (its 8 K
// values are 8 pixels of a row), so images of any width fill the K of 32.
// Both operands lie in LDS as they lie in memory, channels contiguous, and are
// transposed by ds_read_b64_tr_b16 on the way to the registers.  A row of X
// is read once per column offset and multiplied with the three rows of dU it
// meets (3 NCO MFMAs per operand), which keeps the MFMAs ahead of the LDS
// reads.  The bias gradient is one more product, with ones.
// LDS: the pixel pitch is an odd multiple of 32 bytes and the cells are half
// the banks apart, so the 4 x 16 channel blocks of two lane groups never meet
// in a bank.  The next stage's loads are in flight while this one is
// multiplied.
// Splitting K over at most kWgBlocks blocks in all (two per CU; 512 against
// the 36 k blocks of one tap, 64 x 32 channels and 512 pixels each that this
// replaced) keeps the partial sums few.  With ws they go there, [split][co][9]
// [ci] and then [split][co], for k_wgrad_reduce; without, they are added to
// dW by atomics.
// 8 scenes of 256 x 256: the 15 layers together 536 us and 114 us for the sums
// of the splits, against 2400 us and 960 us for the bias sums in a kernel of
// their own (36,864 atomic partial sums of 64 x 32 per layer at most).
constexpr int kWgBlocks = 512;
constexpr int kWgCell = 8, kWgHalo = kWgCell + 2, kWgMaxBCI = 64;

template <int NCO, int WCO, int WCI>
struct WgDims {
    static constexpr int BCO = 16 * NCO * WCO, BCI = 16 * WCI;
    static constexpr int pitch(int c) { return (2 * c / 32) % 2 ? 2 * c : 2 * c + 32; }  // bytes per pixel
    // bytes per cell, half the banks (128 of 256 bytes) past a multiple of all of them
    static constexpr int cell(int px, int c) { return px * pitch(c) + (384 - px * pitch(c) % 256) % 256; }
    static constexpr int PD = pitch(BCO), PX = pitch(BCI);
    static constexpr int SD = cell(kWgCell * kWgCell, BCO), SX = cell(kWgHalo * kWgHalo, BCI);
    static constexpr int GD = BCO / 8, GX = BCI / 8;  // 16-byte groups per pixel
    static constexpr int ND = (4 * kWgCell * kWgCell * GD + 255) / 256, NX = (4 * kWgHalo * kWgHalo * GX + 255) / 256;
};

__device__ __forceinline__ bf8v lds_transpose8(const char *p, int pitch)
{
    typedef __attribute__((address_space(3))) s4v *lds_ptr;
    const s4v lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)p);
    const s4v hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(p + 4 * pitch));
    typedef short s8v __attribute__((ext_vector_type(8)));
    return __builtin_bit_cast(bf8v, (s8v)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}

// grid (splits, co blocks, ci blocks); split k takes stages k, k + splits, ...
template <int NCO, int WCO, int WCI>
__global__ void __launch_bounds__(256, WCI == 4 ? 1 : 2)  // (its LDS fits twice in a CU but with 64 input channels)
k_conv3x3_wgrad(const uint16_t *__restrict__ dU, const uint16_t *__restrict__ X, float *__restrict__ dW,
                float *__restrict__ db, float *__restrict__ ws, int B, int H, int W, int Cin, int Cout, int up)
{
    using D = WgDims<NCO, WCO, WCI>;
    static_assert(WCO * WCI == 4, "four waves");
    constexpr int R = kWgCell, HX = kWgHalo;
    __shared__ __align__(16) char ds[4 * D::SD];
    __shared__ __align__(16) char xs[4 * D::SX];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, wco = wv / WCI, wci = wv % WCI;
    const int co0 = blockIdx.y * D::BCO, ci0 = blockIdx.z * D::BCI;
    const int ncx = (W + R - 1) / R, ncy = (H + R - 1) / R, ncells = B * ncx * ncy;
    const int nstages = (ncells + 3) / 4;
    const int Hs = H >> up, Ws = W >> up;  // X's own size (with up: half, read as its 2x nearest upsampling)
    u32x4 dr[D::ND], xr[D::NX];
    unsigned dmask = 0, xmask = 0;
    const u32x4 z = {0u, 0u, 0u, 0u};
    // (every load reads a valid address; what lies outside is zeroed on its way to LDS)
    auto load = [&](int st) {
        dmask = xmask = 0;
#pragma unroll
        for (int j = 0; j < D::ND; j++) {
            const int idx = tid + 256 * j, q = idx % D::GD, px = idx / D::GD, c = px / (R * R);
            const int cell = 4 * st + c, b = cell / (ncx * ncy), rem = cell - b * ncx * ncy;
            const int cy = rem / ncx, cx = rem - cy * ncx;
            const int y = cy * R + px / R % R, x = cx * R + px % R;
            const bool in = c < 4 && cell < ncells && y < H && x < W && co0 + 8 * q < Cout;
            dr[j] = *(const u32x4 *)(dU + (in ? ((size_t)(b * H + y) * W + x) * Cout + co0 + 8 * q : 0));
            dmask |= (in ? 1u : 0u) << j;
        }
#pragma unroll
        for (int j = 0; j < D::NX; j++) {
            const int idx = tid + 256 * j, q = idx % D::GX, px = idx / D::GX, c = px / (HX * HX);
            const int cell = 4 * st + c, b = cell / (ncx * ncy), rem = cell - b * ncx * ncy;
            const int cy = rem / ncx, cx = rem - cy * ncx, hp = px - c * HX * HX;
            const int y = cy * R - 1 + hp / HX, x = cx * R - 1 + hp % HX;
            const bool in = c < 4 && cell < ncells && y >= 0 && y < H && x >= 0 && x < W && ci0 + 8 * q < Cin;
            xr[j] = *(const u32x4 *)(X + (in ? ((size_t)(b * Hs + (y >> up)) * Ws + (x >> up)) * Cin + ci0 + 8 * q : 0));
            xmask |= (in ? 1u : 0u) << j;
        }
    };
    auto store = [&]() {
#pragma unroll
        for (int j = 0; j < D::ND; j++) {
            const int idx = tid + 256 * j, q = idx % D::GD, px = idx / D::GD, c = px / (R * R);
            if (c < 4) *(u32x4 *)(ds + c * D::SD + (px - c * R * R) * D::PD + 16 * q) = (dmask >> j & 1) ? dr[j] : z;
        }
#pragma unroll
        for (int j = 0; j < D::NX; j++) {
            const int idx = tid + 256 * j, q = idx % D::GX, px = idx / D::GX, c = px / (HX * HX);
            if (c < 4) *(u32x4 *)(xs + c * D::SX + (px - c * HX * HX) * D::PX + 16 * q) = (xmask >> j & 1) ? xr[j] : z;
        }
    };
    f4v acc[9][NCO], accb[NCO];
#pragma unroll
    for (int i = 0; i < NCO; i++) {
        accb[i] = f4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int t = 0; t < 9; t++) acc[t][i] = f4v{0.f, 0.f, 0.f, 0.f};
    }
    bf8v ones;
#pragma unroll
    for (int k = 0; k < 8; k++) ones[k] = (__bf16)1.0f;
    const bool bias = db && blockIdx.z == 0 && wci == 0;
    // this lane's share of an operand block: 4 channels of pixel (lane % 16) / 4 of its group's cell
    const int grp = lane >> 4, lp = (lane & 15) >> 2, lc = 4 * (lane & 3);
    const char *dsl = ds + grp * D::SD + lp * D::PD + 2 * (wco * 16 * NCO + lc);
    const char *xsl = xs + grp * D::SX + lp * D::PX + 2 * (wci * 16 + lc);
    load(blockIdx.x);
    for (int st = blockIdx.x; st < nstages; st += gridDim.x) {
        __syncthreads();  // the former stage is multiplied out
        store();
        __syncthreads();
        if (st + (int)gridDim.x < nstages) load(st + gridDim.x);
        bf8v a[3][NCO];
#pragma unroll
        for (int hr = 0; hr < HX; hr++) {
            if (hr < R)
#pragma unroll
                for (int i = 0; i < NCO; i++) {
                    a[hr % 3][i] = lds_transpose8(dsl + hr * R * D::PD + 32 * i, D::PD);
                    if (bias) accb[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[hr % 3][i], ones, accb[i], 0, 0, 0);
                }
#pragma unroll
            for (int dx = 0; dx < 3; dx++) {
                const bf8v b = lds_transpose8(xsl + (hr * HX + dx) * D::PX, D::PX);
#pragma unroll
                for (int dy = 0; dy < 3; dy++) {
                    const int r = hr - dy;  // the row of dU that tap (dy, dx) pairs with this row of X
                    if (r < 0 || r >= R) continue;
#pragma unroll
                    for (int i = 0; i < NCO; i++)
                        acc[3 * dy + dx][i] =
                            __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[r % 3][i], b, acc[3 * dy + dx][i], 0, 0, 0);
                }
            }
        }
    }
    const size_t nw = (size_t)Cout * 9 * Cin;
    float *wsp = ws ? ws + (size_t)blockIdx.x * (nw + Cout) : nullptr;
    const int ci = ci0 + wci * 16 + (lane & 15);
#pragma unroll
    for (int i = 0; i < NCO; i++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int co = co0 + (wco * NCO + i) * 16 + 4 * (lane >> 4) + r;
            if (co >= Cout) continue;
            if (ci < Cin)
#pragma unroll
                for (int t = 0; t < 9; t++) {
                    const size_t o = ((size_t)co * 9 + t) * Cin + ci;
                    if (wsp) wsp[o] = acc[t][i][r];
                    else atomicAdd(dW + o, acc[t][i][r]);
                }
            if (bias && (lane & 15) == 0) {
                if (wsp) wsp[nw + co] = accb[i][r];
                else atomicAdd(db + co, accb[i][r]);
            }
        }
}

// g[i] = sum over the splits of ws[split][i], in split order by four
// interleaved chains; the weights and biases of a layer are contiguous in g.
__global__ void __launch_bounds__(256)
k_wgrad_reduce(const float *__restrict__ ws, float *__restrict__ g, size_t n, int splits)
{
    __shared__ float part[4][64];
    const int x = threadIdx.x & 63, y = threadIdx.x >> 6;
    const size_t i = (size_t)blockIdx.x * 64 + x;
    float s = 0.0f;
    if (i < n) {
        const float *p = ws + i;
#pragma unroll 8
        for (int k = y; k < splits; k += 4) s += p[(size_t)k * n];
    }
    part[y][x] = s;
    __syncthreads();
    if (y == 0 && i < n) g[i] = (part[0][x] + part[1][x]) + (part[2][x] + part[3][x]);
}

__global__ void k_fill_f32(float *__restrict__ a, size_t n, float v)
{
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) a[i] = v;
}

__global__ void k_f32_to_bf16(const float *__restrict__ a, uint16_t *__restrict__ b, size_t n)
{
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        b[i] = f2bf(a[i]);
}

// Wf[ci][t][co] = W[co][8 - t][ci]: the weights of the input-gradient
// convolutions, every layer of the list in one launch (grid.y).
__global__ void k_flip_weights(const uint16_t *__restrict__ wb, uint16_t *__restrict__ wf, CnnLayers l)
{
    const int Cin = l.cin[blockIdx.y], Cout = l.cout[blockIdx.y];
    const uint16_t *Wt = wb + l.woff[blockIdx.y];
    uint16_t *Wf = wf + l.woff[blockIdx.y];
    const size_t n = (size_t)Cout * 9 * Cin;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        const int co = (int)(i % Cout);
        const size_t q = i / Cout;
        const int t = (int)(q % 9);
        const int ci = (int)(q / 9);
        Wf[i] = Wt[((size_t)co * 9 + (8 - t)) * Cin + ci];
    }
}

// Loss of the prediction against the target (planar FP32 [B][3][H][W]):
// per-block partial sums of the squared error (FP64) and the gradient
// d loss / d out = 2 (pred - target) / count as the bf16 the head's backward
// pass reads, NHWC with co channels (0 on the padding channels; co a multiple
// of 8).
__global__ void __launch_bounds__(256)
k_sq_loss(const float *__restrict__ pred, const float *__restrict__ target, uint16_t *__restrict__ dU,
          double *__restrict__ partials, int B, int HW, int co, float scale)
{
    double s = 0.0;
    const size_t n = (size_t)B * HW;
    for (size_t p = (size_t)blockIdx.x * blockDim.x + threadIdx.x; p < n; p += (size_t)gridDim.x * blockDim.x) {
        const size_t b = p / HW, o = p - b * HW;
        uint32_t h[3];
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const size_t q = (b * 3 + c) * HW + o;
            const float d = pred[q] - target[q];
            s += (double)d * d;
            h[c] = f2bf(scale * d);
        }
        u32x4 v = {h[0] | h[1] << 16, h[2], 0u, 0u};
        for (int c = 0; c < co; c += 8) {
            *(u32x4 *)(dU + p * co + c) = v;
            v = u32x4{0u, 0u, 0u, 0u};
        }
    }
    __shared__ double red[16];
    double v[1] = {s};
    block_partials<1>(v, partials, red);
}

// Adam on FP32 master weights (Kingma & Ba, bias-corrected), then the bf16
// copy the convolutions read.  mask (nullable) zeroes the update of padding
// weights.
__global__ void k_adam(float *__restrict__ w, float *__restrict__ m, float *__restrict__ v, const float *__restrict__ g,
                       uint16_t *__restrict__ wb, size_t n, float lr, float b1, float b2, float eps, float c1, float c2)
{
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        const float gi = g[i];
        const float mi = b1 * m[i] + (1.0f - b1) * gi;
        const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
        m[i] = mi;
        v[i] = vi;
        const float wi = w[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
        w[i] = wi;
        if (wb) wb[i] = f2bf(wi);
    }
}

// The warped stack (the network's input): per view, the view's colours
// splatted into the target with the solver's footprint weights and
// normalised by the splatted weight, and min(1, weight); 0 where no footprint
// reached the pixel; channels 4 v .. 4 v + 3 of a bf16 NHWC [N][cpad] tensor,
// the channels beyond 4 V zero.
//
// A footprint splat is a 2 x 2 splat of the entry onto box starts (anchors)
// followed by a D x D box sum (D = dsf, box_weights): per source pixel 4
// anchor taps instead of (D + 1)^2, which is what the atomics cost.  Views go
// in groups of kStackGroup: their anchors (r, g, b, weight sums on a
// (W + D + 1) x (H + D + 1) grid, anchor x0 at column x0 + D) by float
// atomics, then one pass per target tile that box-sums them from LDS and
// writes the group's 4 kStackGroup channels of each pixel in two 16-byte
// stores.
constexpr int kStackGroup = 4;
constexpr int kStackTW = 32, kStackTH = 8;

template <int KS>
__global__ void k_stack_anchor(int w, int h, int W, int H, int WA, int HA, const float *__restrict__ tx,
                               const float *__restrict__ ty, const float *__restrict__ views, int v0, int nv,
                               float *__restrict__ anchors)
{
    constexpr int D = KS - 1;
    const size_t n = (size_t)w * h, NA = (size_t)WA * HA;
    const size_t m = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int g = blockIdx.y;
    if (m >= n || g >= nv) return;
    const size_t k = (size_t)(v0 + g) * n + m;
    const float t0 = tx[k], t1 = ty[k];
    if (!cell_valid(t0, t1, W, H)) return;
    int x0, y0;
    float ax[2], ay[2];
    if (!box_weights<KS>(t0, t1, W, H, x0, y0, ax, ay)) return;
    const float *vp = views + (size_t)(v0 + g) * 3 * n + m;
    const float val[4] = {vp[0], vp[n], vp[2 * n], 1.0f};
    float *A = anchors + (size_t)g * 4 * NA;
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const size_t o = (size_t)(y0 + i + D) * WA + (x0 + j + D);
            const float a = ay[i] * ax[j];
#pragma unroll
            for (int q = 0; q < 4; q++) atomicAdd(A + q * NA + o, a * val[q]);
        }
}

template <int D>
__global__ void __launch_bounds__(kStackTW * kStackTH)
k_stack_box_pack(int W, int H, int WA, int HA, const float *__restrict__ anchors, int nv, uint16_t *__restrict__ out,
                 int cpad, int chan0, int zero_from)
{
    constexpr int LW = kStackTW + D - 1, LH = kStackTH + D - 1, LP = LW * LH, NPL = 4 * kStackGroup;
    __shared__ float win[NPL * LP];
    const size_t NA = (size_t)WA * HA;
    const int x0 = blockIdx.x * kStackTW, y0 = blockIdx.y * kStackTH;
    // pixel (x, y) sums the anchors of box starts x - D + 1 .. x, i.e. anchor
    // columns x + 1 .. x + D; the window starts at column x0 + 1, row y0 + 1
    for (int i = threadIdx.x; i < NPL * LP; i += blockDim.x) {
        const int pl = i / LP, r = i - pl * LP, ly = r / LW, lx = r - ly * LW;
        const int ax = x0 + 1 + lx, ay = y0 + 1 + ly;
        win[i] = (pl < 4 * nv && ax < WA && ay < HA) ? anchors[(size_t)pl * NA + (size_t)ay * WA + ax] : 0.0f;
    }
    __syncthreads();
    const int lx = threadIdx.x % kStackTW, ly = threadIdx.x / kStackTW;
    const int x = x0 + lx, y = y0 + ly;
    if (x >= W || y >= H) return;
    uint16_t ch[NPL];
#pragma unroll
    for (int g = 0; g < kStackGroup; g++) {
        float sum[4];
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const float *pw = win + (4 * g + q) * LP;
            float acc = 0.0f;
#pragma unroll
            for (int i = 0; i < D; i++)
#pragma unroll
                for (int j = 0; j < D; j++) acc += pw[(ly + i) * LW + lx + j];
            sum[q] = acc;
        }
        const float iw = sum[3] > 0.0f ? 1.0f / sum[3] : 0.0f;
        const bool live = g < nv;
        ch[4 * g + 0] = live ? f2bf(sum[0] * iw) : 0;
        ch[4 * g + 1] = live ? f2bf(sum[1] * iw) : 0;
        ch[4 * g + 2] = live ? f2bf(sum[2] * iw) : 0;
        ch[4 * g + 3] = live ? f2bf(fminf(sum[3], 1.0f)) : 0;
    }
    uint16_t *q = out + ((size_t)y * W + x) * cpad + chan0;
    u32x4 lo, hi;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        lo[k] = (uint32_t)ch[2 * k] | ((uint32_t)ch[2 * k + 1] << 16);
        hi[k] = (uint32_t)ch[8 + 2 * k] | ((uint32_t)ch[8 + 2 * k + 1] << 16);
    }
    *(u32x4 *)q = lo;
    *(u32x4 *)(q + 8) = hi;
    // after the last group: the channels beyond the views, zero
    if (zero_from >= 0)
        for (int c = zero_from; c < cpad; c += 8) *(u32x4 *)(out + ((size_t)y * W + x) * cpad + c) = u32x4{0, 0, 0, 0};
}

// ---- launchers --------------------------------------------------------------

inline unsigned int ew_blocks(size_t n) { return (unsigned int)std::min<size_t>((n + 255) / 256, 16384); }

// The output channels per block (64, 32 or 16): the widest that the layer's
// channels fill and that leaves a block for each of the 256 CUs; narrower
// blocks stage the halo more often.
hipError_t cnn_conv(int epi, CnnConv a, hipStream_t s)
{
    if (a.Cin % kCvBK != 0 || (epi != CNN_F32 && a.Cout % 4 != 0)) return hipErrorInvalidValue;
    const long tiles = (long)a.B * ((a.W + 15) / 16) * ((a.H + 15) / 16);
    if (tiles > INT_MAX) return hipErrorInvalidValue;
    const int couts = epi == CNN_HEAD ? 3 : a.Cout;
    a.vec = a.Cout % 4 == 0 && (uintptr_t)a.Y % 16 == 0;
    auto groups = [&](int nj) { return (couts + 16 * nj - 1) / (16 * nj); };
    const int nj = couts > 32 && tiles * groups(4) >= 256 ? 4 : couts > 16 && (tiles * groups(2) >= 256 || couts <= 32) ? 2 : 1;
    // resident blocks per CU: 2 of 64 channels, 3 of 32, 4 of 16; every block the same number of tiles
    const long cap = std::max(1L, (nj == 4 ? 512L : nj == 2 ? 768L : 1024L) / groups(nj));
    const long rounds = (tiles + cap - 1) / cap;
    const dim3 grid((unsigned int)((tiles + rounds - 1) / rounds), (unsigned int)groups(nj));
#define CV(E)                                                          \
    case E:                                                            \
        if (nj == 4) k_conv3x3<E, 4><<<grid, 256, 0, s>>>(a);          \
        else if (nj == 2) k_conv3x3<E, 2><<<grid, 256, 0, s>>>(a);     \
        else k_conv3x3<E, 1><<<grid, 256, 0, s>>>(a);                  \
        break
    switch (epi) {
        CV(CNN_F32);
        CV(CNN_FWD);
        CV(CNN_MASK);
        CV(CNN_MASK_UP);
        CV(CNN_MASK_POOL);
    case CNN_HEAD: k_conv3x3<CNN_HEAD, 1><<<grid, 256, 0, s>>>(a); break;
    default: return hipErrorInvalidValue;
    }
#undef CV
    return hipGetLastError();
}

// The splits of a layer's weight gradient: as many as fill kWgBlocks blocks with
// its channel blocks (see k_conv3x3_wgrad), at most one per stage.
static void wgrad_plan(int B, int H, int W, int Cin, int Cout, bool &tall, bool &wide, dim3 &grid)
{
    tall = Cout > 32;                      // 64 x 32 channels per block
    wide = !tall && Cin % kWgMaxBCI == 0;  // 32 x 64; else 32 x 32
    const int nco = (Cout + (tall ? 63 : 31)) / (tall ? 64 : 32), nci = Cin / (wide ? 64 : 32);
    const int stages = (B * ((H + kWgCell - 1) / kWgCell) * ((W + kWgCell - 1) / kWgCell) + 3) / 4;
    grid = dim3((unsigned int)std::max(1, std::min(stages, kWgBlocks / (nco * nci))), (unsigned int)nco,
                (unsigned int)nci);
}

size_t cnn_wgrad_ws_floats(int B, int H, int W, int Cin, int Cout)
{
    bool tall, wide;
    dim3 grid;
    wgrad_plan(B, H, W, Cin, Cout, tall, wide, grid);
    return grid.x * ((size_t)Cout * 9 * Cin + Cout);
}

// dW (Cout x 9 x Cin) and, when it is not null, db; with ws (of cnn_wgrad_ws_floats)
// they are set (db must follow dW), without ws they are added to.
hipError_t cnn_conv_wgrad(const uint16_t *dU, const uint16_t *X, float *dW, float *db, float *ws, int B, int H, int W,
                          int Cin, int Cout, int up, hipStream_t s)
{
    const size_t nw = (size_t)Cout * 9 * Cin;
    if (Cin % 32 != 0 || Cout % 8 != 0 || (ws && db != dW + nw)) return hipErrorInvalidValue;
    bool tall, wide;
    dim3 grid;
    wgrad_plan(B, H, W, Cin, Cout, tall, wide, grid);
    if (tall) k_conv3x3_wgrad<2, 2, 2><<<grid, 256, 0, s>>>(dU, X, dW, db, ws, B, H, W, Cin, Cout, up);
    else if (wide) k_conv3x3_wgrad<2, 1, 4><<<grid, 256, 0, s>>>(dU, X, dW, db, ws, B, H, W, Cin, Cout, up);
    else k_conv3x3_wgrad<1, 2, 2><<<grid, 256, 0, s>>>(dU, X, dW, db, ws, B, H, W, Cin, Cout, up);
    if (ws) k_wgrad_reduce<<<(unsigned int)((nw + Cout + 63) / 64), 256, 0, s>>>(ws, dW, nw + Cout, (int)grid.x);
    return hipGetLastError();
}

hipError_t cnn_fill(float *a, size_t n, float v, hipStream_t s)
{
    k_fill_f32<<<ew_blocks(n), 256, 0, s>>>(a, n, v);
    return hipGetLastError();
}

hipError_t cnn_to_bf16(const float *a, uint16_t *b, size_t n, hipStream_t s)
{
    k_f32_to_bf16<<<ew_blocks(n), 256, 0, s>>>(a, b, n);
    return hipGetLastError();
}

hipError_t cnn_flip_weights(const uint16_t *wb, uint16_t *wf, const CnnLayers &l, hipStream_t s)
{
    size_t n = 0;
    for (int i = 0; i < l.n; i++) n = std::max(n, (size_t)l.cout[i] * 9 * l.cin[i]);
    if (l.n > 0) k_flip_weights<<<dim3(std::min(ew_blocks(n), 512u), l.n), 256, 0, s>>>(wb, wf, l);
    return hipGetLastError();
}

hipError_t cnn_sq_loss(const float *pred, const float *target, uint16_t *dU, double *partials, int nblocks, int B,
                       int HW, int co, float scale, hipStream_t s)
{
    k_sq_loss<<<nblocks, 256, 0, s>>>(pred, target, dU, partials, B, HW, co, scale);
    return hipGetLastError();
}

int cnn_stack_group() { return kStackGroup; }

size_t cnn_stack_anchor_floats(int W, int H, int dsf) { return (size_t)kStackGroup * 4 * (W + dsf + 1) * (H + dsf + 1); }

// One group of views of the warped stack: anchors (cleared here) then the box
// pass writing channels 4 v0 .. 4 v0 + 4 kStackGroup - 1 (zero for the views
// beyond nv); zero_from >= 0 also clears channels zero_from .. cpad - 1.
hipError_t cnn_stack_group_pass(int dsf, int w, int h, int W, int H, const float *tx, const float *ty,
                                const float *views, int v0, int nv, float *anchors, uint16_t *out, int cpad,
                                int zero_from, hipStream_t s)
{
    const int WA = W + dsf + 1, HA = H + dsf + 1;
    if (nv < 1 || nv > kStackGroup || (4 * v0) % 16 || cpad % 8) return hipErrorInvalidValue;
    hipError_t e = hipMemsetAsync(anchors, 0, cnn_stack_anchor_floats(W, H, dsf) * sizeof(float), s);
    if (e != hipSuccess) return e;
    const size_t n = (size_t)w * h;
    const dim3 ga((unsigned int)((n + 255) / 256), (unsigned int)nv);
    const dim3 gb((W + kStackTW - 1) / kStackTW, (H + kStackTH - 1) / kStackTH);
    switch (dsf) {
#define ST(D)                                                                                                   \
    case D:                                                                                                     \
        k_stack_anchor<D + 1><<<ga, 256, 0, s>>>(w, h, W, H, WA, HA, tx, ty, views, v0, nv, anchors);          \
        k_stack_box_pack<D><<<gb, kStackTW * kStackTH, 0, s>>>(W, H, WA, HA, anchors, nv, out, cpad, 4 * v0,    \
                                                                zero_from);                                     \
        break;
        ST(1) ST(2) ST(3) ST(4)
#undef ST
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t cnn_adam(float *w, float *m, float *v, const float *g, uint16_t *wb, size_t n, float lr, float b1,
                    float b2, float eps, int step, hipStream_t s)
{
    const float c1 = 1.0f - powf(b1, (float)step), c2 = 1.0f - powf(b2, (float)step);
    k_adam<<<ew_blocks(n), 256, 0, s>>>(w, m, v, g, wb, n, lr, b1, b2, eps, c1, c2);
    return hipGetLastError();
}

}  // namespace lfrv
