// Stencil kernels: hole filling (Poisson diffusion, push-pull), the Gaussian
// smoothing of the TV weight.
#include "tile_common.hpp"

#include <hip/hip_ext.h>

#include <cmath>

namespace lfrv {

namespace {

// ---- Poisson diffusion in the holes (gradientIBR.cu:87-152) ---------------

__global__ void k_hole_list(size_t N, const float *__restrict__ vis, int *__restrict__ list,
                            unsigned int *__restrict__ count)
{
    const size_t o = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (o >= N || vis[o] != 0.0f) return;
    const unsigned int k = atomicAdd(count, 1u);
    list[k] = (int)o;
}

// The diffusion runs up to kHoleSweeps Jacobi sweeps per launch: a block takes a
// tile of kHoleTile^2 pixels that holds holes into LDS with a halo as wide as
// the sweeps, and the halo's validity shrinks by a pixel per sweep.
// The stopping rule is still the one after every sweep: a launch leaves the
// energy of each of its sweeps, the next one evaluates the rule on them, and if
// it fired before the last of them runs that many sweeps again from the same
// start.  100 x 75 holes of a 403 x 301 view, 500 sweeps: 0.79 ms; one sweep per
// launch, 2.05 ms (4.1 us each, the launch of a dependent tiny kernel).
// Every block adds up the energies of all of them, so there are at most
// kHoleBlocks, two per CU, which run through the tiles: 1000 tiles of a 700 x
// 700 view, 500 sweeps: 2.3 ms (1024 blocks 2.8, a block per tile 2.5); 8200
// tiles of a 1535 x 1531 view: 10.6 ms (11.3 and 29; one sweep per launch 22.5).
constexpr int kHoleTile = 16, kHoleSweeps = 8, kHoleRegion = kHoleTile + 2 * kHoleSweeps, kHoleBlocks = 512;

// eh[j] holds the energy of sweep j (eh[0] = 0, the energy the first sweep is
// compared with); *stopped the number of sweeps run once the rule has fired.
struct HoleLoop {
    int maxit;
    double eps;
    double *eh;         // maxit + 1
    int *stopped;
    const int *tiles;   // the tiles with holes, in order; *count of them
    const int *count;
};

__global__ void k_hole_init(HoleLoop hl, int ntiles, int *flags)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < ntiles) flags[k] = 0;
    if (k == 0) {
        hl.eh[0] = 0.0;
        *hl.stopped = 0;
    }
}

__global__ void k_hole_flag(int W, int ntx, int nholes, const int *__restrict__ list, int *__restrict__ flags)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= nholes) return;
    const int o = list[k], y = o / W, x = o - y * W;
    flags[y / kHoleTile * ntx + x / kHoleTile] = 1;  // (every writer writes 1)
}

// tiles <- the flagged ones in order (one block of 1024)
__global__ void __launch_bounds__(1024) k_hole_tiles(int ntiles, const int *__restrict__ flags, int *__restrict__ tiles,
                                                     int *__restrict__ count)
{
    __shared__ int wsum[16];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    int base = 0;
    for (int t0 = 0; t0 < ntiles; t0 += 1024) {
        const int t = t0 + threadIdx.x;
        const bool f = t < ntiles && flags[t];
        const unsigned long long m = __ballot(f);
        if (lane == 0) wsum[wv] = __popcll(m);
        __syncthreads();
        int off = base, all = 0;
        for (int w = 0; w < 16; w++) {
            if (w < wv) off += wsum[w];
            all += wsum[w];
        }
        if (f) tiles[off + __popcll(m & ((1ull << lane) - 1))] = t;
        base += all;
        __syncthreads();
    }
    if (threadIdx.x == 0) *count = base;
}

// Sweeps k0 + 1 .. k0 + K (K <= kHoleSweeps; 0 to evaluate the rule alone) of
// the Poisson diffusion, uin to uout: u <- mean of the 4-neighbours (the
// reference's laplacian then add_to) on the hole pixels, all three channels,
// with the energy sum(lap * u_new) of the last channel per sweep.  First the
// stopping rule of gradientIBR.cu:139-143 on the Kprev sweeps of the launch
// before, |E_{j-1} - E_j| < eps or j >= maxit, evaluated by every block alike
// (pin: their block sums; the launch before read uout and wrote uin).
__global__ void __launch_bounds__(512) k_hole_sweeps(int W, int H, int ntx, const float *__restrict__ vis, float *uin,
                                                     float *uout, HoleLoop hl, int k0, int K, int Kprev,
                                                     const double *__restrict__ pin, double *__restrict__ pout)
{
    constexpr int R = kHoleRegion, NP = R * R, NT = 512, PT = NP / NT;
    __shared__ float us[2][3][NP];
    __shared__ double es[kHoleSweeps + 1], ws[NT / 64][kHoleSweeps];
    __shared__ int stop;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int ntiles = *hl.count, n = min(ntiles, (int)gridDim.x);  // n: the blocks with tiles
    if ((int)blockIdx.x >= n) return;
    // (a stop within the launch before is set by this launch, maybe already)
    if (tid == 0) {
        const int st = *hl.stopped;
        stop = st != 0 && st <= k0 - Kprev ? -1 : 0;
        es[0] = hl.eh[k0 - Kprev];
    }
    __syncthreads();
    if (stop < 0) return;
    if (wv < Kprev) {
        double e = 0.0;
        for (int b = lane; b < n; b += 64) e += pin[(size_t)wv * n + b];
        for (int d = 32; d > 0; d >>= 1) e += __shfl_down(e, d);
        if (lane == 0) es[wv + 1] = e;
    }
    __syncthreads();
    if (tid == 0) {
        int j = 1;
        while (j <= Kprev && !(fabs(es[j - 1] - es[j]) < hl.eps || k0 - Kprev + j >= hl.maxit)) j++;
        stop = j <= Kprev ? j : 0;
        if (blockIdx.x == 0) {
            for (int q = 1; q <= (stop ? stop : Kprev); q++) hl.eh[k0 - Kprev + q] = es[q];
            if (stop) *hl.stopped = k0 - Kprev + stop;
        }
    }
    __syncthreads();
    const bool redo = stop != 0;
    if (redo && stop == Kprev) return;  // the launch before ended where the rule fired
    const float *src = redo ? uout : uin;
    float *dst = redo ? uin : uout;
    const int sweeps = redo ? stop : K;
    if (sweeps == 0) return;

    const size_t N = (size_t)W * H;
    double e[kHoleSweeps];
#pragma unroll
    for (int s = 0; s < kHoleSweeps; s++) e[s] = 0.0;
    for (int k = blockIdx.x; k < ntiles; k += n) {
        const int tile = hl.tiles[k], ty = tile / ntx, tx = tile - ty * ntx;
        const int rx = tx * kHoleTile - kHoleSweeps, ry = ty * kHoleTile - kHoleSweeps;
        bool hole[PT], own[PT];
#pragma unroll
        for (int p = 0; p < PT; p++) {
            const int i = tid + p * NT, lx = i % R, ly = i / R, x = rx + lx, y = ry + ly;
            const bool in = x >= 0 && x < W && y >= 0 && y < H;
            const size_t o = in ? (size_t)y * W + x : 0;
            hole[p] = in && vis[o] == 0.0f;
            own[p] = hole[p] && lx >= kHoleSweeps && lx < R - kHoleSweeps && ly >= kHoleSweeps && ly < R - kHoleSweeps;
            // (the region's rim keeps its values: it has no neighbours beyond)
            hole[p] = hole[p] && lx > 0 && lx < R - 1 && ly > 0 && ly < R - 1;
#pragma unroll
            for (int c = 0; c < 3; c++) us[0][c][i] = us[1][c][i] = in ? src[c * N + o] : 0.0f;
        }
        __syncthreads();
#pragma unroll
        for (int s = 0; s < kHoleSweeps; s++) {
            if (s >= sweeps) continue;
#pragma unroll
            for (int p = 0; p < PT; p++) {
                if (!hole[p]) continue;
                const int i = tid + p * NT, x = rx + i % R, y = ry + i / R;
#pragma unroll
                for (int c = 0; c < 3; c++) {
                    const float *u = us[s & 1][c];
                    float mean;
                    if (x > 0 && y > 0 && x < W - 1 && y < H - 1) {  // (a quarter: exact, and no division)
                        mean = 0.25f * (((u[i - 1] + u[i - R]) + u[i + 1]) + u[i + R]);
                    } else {
                        float sm = 0.0f, wsum = 0.0f;
                        if (x > 0) { sm += u[i - 1]; wsum += 1.0f; }
                        if (y > 0) { sm += u[i - R]; wsum += 1.0f; }
                        if (x < W - 1) { sm += u[i + 1]; wsum += 1.0f; }
                        if (y < H - 1) { sm += u[i + R]; wsum += 1.0f; }
                        mean = sm / wsum;
                    }
                    const float lap = mean - u[i];
                    const float un = u[i] + lap;
                    us[(s & 1) ^ 1][c][i] = un;
                    if (c == 2 && own[p]) e[s] += (double)lap * (double)un;
                }
            }
            __syncthreads();
        }
#pragma unroll
        for (int p = 0; p < PT; p++) {
            if (!own[p]) continue;
            const int i = tid + p * NT;
            const size_t o = (size_t)(ry + i / R) * W + rx + i % R;
#pragma unroll
            for (int c = 0; c < 3; c++) dst[c * N + o] = us[sweeps & 1][c][i];
        }
        // (a pixel of us[] that a thread still reads here is its own: it may take the next tile's at once)
    }
    if (redo) return;
#pragma unroll
    for (int s = 0; s < kHoleSweeps; s++) {
        double v = e[s];
        for (int d = 32; d > 0; d >>= 1) v += __shfl_down(v, d);
        if (lane == 0) ws[wv][s] = v;
    }
    __syncthreads();
    if (tid < sweeps) {
        double v = 0.0;
        for (int w = 0; w < NT / 64; w++) v += ws[w][tid];
        pout[(size_t)tid * n + blockIdx.x] = v;
    }
}

// ---- separable Gaussian, clamp to edge (cuda_convolutions.cu:110-237) -------

struct Taps {
    float k[15];
    int r;
};

__global__ void k_conv_rows(int W, int H, Taps t, const float *__restrict__ in, float *__restrict__ out)
{
    const int x = blockIdx.x * blockDim.x + threadIdx.x, y = blockIdx.y;
    if (x >= W) return;
    float s = 0.0f;
    for (int k = -t.r; k <= t.r; k++) {
        const int xx = min(max(x + k, 0), W - 1);
        s += in[(size_t)y * W + xx] * t.k[t.r - k];
    }
    out[(size_t)y * W + x] = s;
}

__global__ void k_conv_cols(int W, int H, Taps t, const float *__restrict__ in, float *__restrict__ out)
{
    const int x = blockIdx.x * blockDim.x + threadIdx.x, y = blockIdx.y;
    if (x >= W) return;
    float s = 0.0f;
    for (int k = -t.r; k <= t.r; k++) {
        const int yy = min(max(y + k, 0), H - 1);
        s += in[(size_t)yy * W + x] * t.k[t.r - k];
    }
    out[(size_t)y * W + x] = s;
}

// ---- push-pull (optimization.cu:210-651), three channels per launch -------
// Images of level s live at img + c*lvl_stride + off[s]; visibility at vis + off[s].
// The centre tap of expand reads row/column i/2 of the coarser level; for an
// odd-sized level that index runs one past the coarser image in the
// reference (optimization.cu:455, 492) and is clamped here.

__device__ __forceinline__ int clampi(int v, int lo, int hi) { return v < lo ? lo : (v > hi ? hi : v); }

// Both passes of a reduction or expansion run in one kernel, which forms the
// few row results that it needs again (the same sums in the same order), and
// the levels of at most kPpTail pixels in one block per channel, in LDS: a
// 256^2 image takes 5 launches where one per level, direction and pass, with
// copies of level 0 around them, took 50 of some 3 us each.
constexpr int kPpTail = 4096;

// Weighted mean of the nonzero values among the five (0 if none).
template <class At>
__device__ __forceinline__ float pp_mean5(At at)
{
    const float a = 0.4f;
    const float k[5] = {0.25f - 0.5f * a, 0.25f, a, 0.25f, 0.25f - 0.5f * a};
    float s = 0.0f, wt = 0.0f;
#pragma unroll
    for (int q = 0; q < 5; q++) {
        const float v = at(q);
        if (v != 0.0f) { s += k[q] * v; wt += k[q]; }
    }
    return (wt == 0.0f) ? 0.0f : s / wt;
}

__device__ __forceinline__ int pp_tap(int i, int q, int n) { return clampi(2 * i - 2 + q, 0, n - 1); }

// Pixel (i, j) of the next coarser level of in (Ws x Hs): rows first.
__device__ __forceinline__ float pp_reduce(const float *in, int Ws, int Hs, int i, int j)
{
    return pp_mean5([&](int q) {
        const float *col = in + pp_tap(j, q, Ws);
        return pp_mean5([&](int r) { return col[(size_t)pp_tap(i, r, Hs) * Ws]; });
    });
}

// Visibility there: OR over the same 5 x 5 support.
template <class V>
__device__ __forceinline__ uint8_t pp_reduce_vis(const V *vis, int Ws, int Hs, int i, int j)
{
    bool v = false;
    for (int r = 0; r < 5; r++)
        for (int q = 0; q < 5; q++) v |= vis[(size_t)pp_tap(i, r, Hs) * Ws + pp_tap(j, q, Ws)] != (V)0;
    return v ? 1 : 0;
}

// Position i of a line of n coarser values, at twice the density.
template <class At>
__device__ __forceinline__ float pp_expand1(int i, int n, At at)
{
    const float a = 0.4f;
    const float k[5] = {0.25f - 0.5f * a, 0.25f, a, 0.25f, 0.25f - 0.5f * a};
    float s = 0.0f;
    if (i % 2 == 0) {
        s += 2.0f * k[0] * at(max((i - 2) / 2, 0));
        s += 2.0f * k[2] * at(min(i / 2, n - 1));
        s += 2.0f * k[4] * at(min((i + 2) / 2, n - 1));
    } else {
        s += 2.0f * k[1] * at(max((i - 1) / 2, 0));
        s += 2.0f * k[3] * at(min((i + 1) / 2, n - 1));
    }
    return s;
}

// Pixel (i, j) of the next finer level of in (ws x hs): rows first.
__device__ __forceinline__ float pp_expand(const float *in, int ws, int hs, int i, int j)
{
    return pp_expand1(j, ws, [&](int x) { return pp_expand1(i, hs, [&](int y) { return in[(size_t)y * ws + x]; }); });
}

// One level down; V: the finer level's visibility is the target's float map (level 0) or bytes.
template <class V>
__global__ void k_pp_reduce(int Ws, int Hs, int ws, int hs, const float *__restrict__ in, size_t in_cstride,
                            const V *__restrict__ vis, float *__restrict__ out, size_t out_cstride,
                            uint8_t *__restrict__ vout)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x, c = blockIdx.y;
    if (k >= ws * hs) return;
    const int i = k / ws, j = k - i * ws;
    out[c * out_cstride + k] = pp_reduce(in + c * in_cstride, Ws, Hs, i, j);
    if (c == 0) vout[k] = pp_reduce_vis(vis, Ws, Hs, i, j);
}

// One level up, where nothing is visible.
__global__ void k_pp_expand(int Ws, int Hs, int ws, int hs, const float *__restrict__ in, float *__restrict__ out,
                            const uint8_t *__restrict__ vis, size_t cstride)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x, c = blockIdx.y;
    if (k >= Ws * Hs || vis[k]) return;
    const int i = k / Ws, j = k - i * Ws;
    out[c * cstride + k] = pp_expand(in + c * cstride, ws, hs, i, j);
}

// The last level up, and U <- filled - U (optimization.cu:629-646); without levels (ws = 0) filled is U.
__global__ void k_pp_finish(int W, int H, int ws, int hs, const float *__restrict__ in, size_t in_cstride,
                            const float *__restrict__ vis, float *__restrict__ U)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x, c = blockIdx.y;
    if (k >= W * H) return;
    const int i = k / W, j = k - i * W;
    const size_t o = (size_t)c * W * H + k;
    const float u = U[o];
    U[o] = (ws == 0 || vis[k] != 0.0f ? u : pp_expand(in + c * in_cstride, ws, hs, i, j)) - u;
}

// Every level below (w, h): down to the coarsest and back up to it, channel
// blockIdx.x, in place.
__global__ void __launch_bounds__(1024) k_pp_tail(int w, int h, int levels, float *__restrict__ img, size_t cstride,
                                                  const uint8_t *__restrict__ vis)
{
    __shared__ float px[kPpTail + kPpTail / 2];  // the levels one behind the other: a quarter of the pixels each
    __shared__ uint8_t vs[kPpTail + kPpTail / 2];
    float *p = img + blockIdx.x * cstride;
    for (int k = threadIdx.x; k < w * h; k += blockDim.x) {
        px[k] = p[k];
        vs[k] = vis[k];
    }
    __syncthreads();
    int o = 0, ws = w, hs = h;
    for (int l = 0; l < levels; l++) {
        const int on = o + ws * hs, wn = ws / 2, hn = hs / 2;
        for (int k = threadIdx.x; k < wn * hn; k += blockDim.x) {
            const int i = k / wn, j = k - i * wn;
            px[on + k] = pp_reduce(px + o, ws, hs, i, j);
            vs[on + k] = pp_reduce_vis(vs + o, ws, hs, i, j);
        }
        __syncthreads();
        o = on;
        ws = wn;
        hs = hn;
    }
    for (int l = levels; l > 0; l--) {
        const int wf = w >> (l - 1), hf = h >> (l - 1), of = o - wf * hf;
        for (int k = threadIdx.x; k < wf * hf; k += blockDim.x) {
            if (vs[of + k]) continue;
            const int i = k / wf, j = k - i * wf;
            px[of + k] = pp_expand(px + o, ws, hs, i, j);
        }
        __syncthreads();
        o = of;
        ws = wf;
        hs = hf;
    }
    for (int k = threadIdx.x; k < w * h; k += blockDim.x) p[k] = px[k];
}

}  // namespace

lfrv_status run_hole_filling(lfrv_ctx *ctx, int iters, double eps, int *ran)
{
    const size_t N = ctx->N;
    unsigned int nh = 0;
    if (ctx->holes_listed) {
        // listed by the visibility pass; its length arrived behind hole_ev
        LFRV_HIP(ctx, hipEventSynchronize(ctx->hole_ev));
        nh = *ctx->hole_count_host;
    } else {
        unsigned int *cnt = ctx->counters + 10;
        LFRV_HIP(ctx, hipMemsetAsync(cnt, 0, sizeof(unsigned int), ctx->stream));
        k_hole_list<<<blocks_for(N), kBlock, 0, ctx->stream>>>(N, ctx->visibility, ctx->hole_list, cnt);
        LFRV_HIP(ctx, hipMemcpyAsync(&nh, cnt, sizeof nh, hipMemcpyDeviceToHost, ctx->stream));
        LFRV_HIP(ctx, hipStreamSynchronize(ctx->stream));
    }
    ctx->n_holes = (int)nh;
    if (ran) *ran = 0;
    if (nh == 0 || iters <= 0) return LFRV_OK;
    float *bufs[2] = {ctx->U, ctx->tmp3N};
    LFRV_HIP(ctx, hipMemcpyAsync(ctx->tmp3N, ctx->U, 3 * N * sizeof(float), hipMemcpyDeviceToDevice, ctx->stream));
    // scratch: the CG's vectors, idle until the solve (per tile of 256 pixels 8 doubles in one, 2 ints in another)
    const int ntx = (ctx->W + kHoleTile - 1) / kHoleTile, ntiles = ntx * ((ctx->H + kHoleTile - 1) / kHoleTile);
    double *psw[2] = {reinterpret_cast<double *>(ctx->cg_q), reinterpret_cast<double *>(ctx->cg_r)};
    int *flags = reinterpret_cast<int *>(ctx->cg_d), *tiles = flags + ntiles;
    int *stopped = reinterpret_cast<int *>(ctx->counters + 12), *count = reinterpret_cast<int *>(ctx->counters + 13);
    const HoleLoop hl{iters, eps, ctx->partials, stopped, tiles, count};
    if ((size_t)iters + 1 > ctx->partials_cap) return fail(ctx, LFRV_E_ARG, "hole filling: too many sweeps");
    k_hole_init<<<blocks_for(ntiles), kBlock, 0, ctx->stream>>>(hl, ntiles, flags);
    k_hole_flag<<<blocks_for(nh), kBlock, 0, ctx->stream>>>(ctx->W, ntx, (int)nh, ctx->hole_list, flags);
    k_hole_tiles<<<1, 1024, 0, ctx->stream>>>(ntiles, flags, tiles, count);
    // (up to the bound at least as many as there are tiles with holes)
    const unsigned int nb = std::min({(unsigned int)ntiles, nh, (unsigned int)kHoleBlocks});
    int launched = 0, chunks = 0, prev = 0, host = 0;
    // the rule is read back after 2 launches, then after every 8 (those enqueued behind a stop return at once)
    while (launched < iters && !host) {
        for (int j = chunks == 0 ? 6 : 0; j < 8 && launched < iters; j++) {
            const int k = std::min(kHoleSweeps, iters - launched);
            k_hole_sweeps<<<nb, 512, 0, ctx->stream>>>(ctx->W, ctx->H, ntx, ctx->visibility, bufs[chunks & 1],
                                                       bufs[(chunks & 1) ^ 1], hl, launched, k, prev,
                                                       psw[(chunks & 1) ^ 1], psw[chunks & 1]);
            launched += k;
            prev = k;
            chunks++;
        }
        // the rule on the last of them (and their redo)
        if (launched == iters)
            k_hole_sweeps<<<nb, 512, 0, ctx->stream>>>(ctx->W, ctx->H, ntx, ctx->visibility, bufs[chunks & 1],
                                                       bufs[(chunks & 1) ^ 1], hl, launched, 0, prev,
                                                       psw[(chunks & 1) ^ 1], psw[chunks & 1]);
        LFRV_LAUNCH(ctx, "hole filling");
        LFRV_HIP(ctx, hipMemcpyAsync(&host, stopped, sizeof host, hipMemcpyDeviceToHost, ctx->stream));
        LFRV_HIP(ctx, hipStreamSynchronize(ctx->stream));
    }
    // (at maxit the rule fires) the result of launch c (1-based) is in bufs[c & 1]
    if (((host + kHoleSweeps - 1) / kHoleSweeps) & 1)
        LFRV_HIP(ctx, hipMemcpyAsync(ctx->U, ctx->tmp3N, 3 * N * sizeof(float), hipMemcpyDeviceToDevice, ctx->stream));
    if (ran) *ran = host;
    return LFRV_OK;
}

lfrv_status run_gauss_smooth(lfrv_ctx *ctx, const float *in, float *out, float *tmp)
{
    // gsl_kernel_gauss_1xn(11, 2.0) (gsl_matrix_convolutions.cpp:42-63)
    Taps t{};
    t.r = 5;
    double s = 0.0, k[11];
    for (int x = -5; x <= 5; x++) {
        k[x + 5] = std::exp(-0.5 * x * x / 4.0);
        s += k[x + 5];
    }
    for (int i = 0; i < 11; i++) t.k[i] = (float)(k[i] / s);
    dim3 bs(256), gs((ctx->W + 255) / 256, ctx->H);
    k_conv_rows<<<gs, bs, 0, ctx->stream>>>(ctx->W, ctx->H, t, in, tmp);
    k_conv_cols<<<gs, bs, 0, ctx->stream>>>(ctx->W, ctx->H, t, tmp, out);
    LFRV_LAUNCH(ctx, "gaussian");
    return LFRV_OK;
}

lfrv_status run_push_pull(lfrv_ctx *ctx, int levels)
{
    const int W = ctx->W, H = ctx->H;
    const size_t N = ctx->N;
    // level offsets inside the pyramid scratch, from level 1 on: level 0 is U itself and the target's map
    std::vector<size_t> off(levels + 1, 0);
    std::vector<int> ws(levels + 1, 0), hs(levels + 1, 0);
    size_t tot = 0;
    int top = 0;
    ws[0] = W;
    hs[0] = H;
    for (int s = 1; s <= levels; s++) {
        const int wsn = W >> s, hsn = H >> s;
        if (wsn <= 0 || hsn <= 0) break;
        ws[s] = wsn;
        hs[s] = hsn;
        off[s] = tot;
        tot += (size_t)wsn * hsn;
        top = s;
    }
    // scratch: pyramid images (3 * tot floats) + vis pyramid (tot bytes)
    const size_t need = 3 * tot + (tot + 3) / 4 + 1;
    if (need > ctx->pp_cap) return fail(ctx, LFRV_E_ARG, "push-pull scratch too small");
    float *img = ctx->pp_scratch;
    uint8_t *vis = reinterpret_cast<uint8_t *>(img + 3 * tot);
    auto grid = [](int w, int h) { return dim3(blocks_for((size_t)w * h), 3); };
    // the levels from `tail` on in one launch
    int tail = 1;
    while (tail < top && (size_t)ws[tail] * hs[tail] > kPpTail) tail++;
    for (int s = 1; s <= tail && s <= top; s++) {
        if (s == 1)
            k_pp_reduce<<<grid(ws[1], hs[1]), kBlock, 0, ctx->stream>>>(W, H, ws[1], hs[1], ctx->U, N, ctx->visibility,
                                                                        img + off[1], tot, vis + off[1]);
        else
            k_pp_reduce<<<grid(ws[s], hs[s]), kBlock, 0, ctx->stream>>>(ws[s - 1], hs[s - 1], ws[s], hs[s],
                                                                        img + off[s - 1], tot, vis + off[s - 1],
                                                                        img + off[s], tot, vis + off[s]);
    }
    if (tail < top)
        k_pp_tail<<<3, 1024, 0, ctx->stream>>>(ws[tail], hs[tail], top - tail, img + off[tail], tot, vis + off[tail]);
    for (int s = std::min(tail, top); s > 1; s--)
        k_pp_expand<<<grid(ws[s - 1], hs[s - 1]), kBlock, 0, ctx->stream>>>(
            ws[s - 1], hs[s - 1], ws[s], hs[s], img + off[s], img + off[s - 1], vis + off[s - 1], tot);
    k_pp_finish<<<grid(W, H), kBlock, 0, ctx->stream>>>(W, H, top ? ws[1] : 0, top ? hs[1] : 0,
                                                        img + (top ? off[1] : 0), tot, ctx->visibility, ctx->U);
    LFRV_LAUNCH(ctx, "push-pull");
    return LFRV_OK;
}

}  // namespace lfrv
