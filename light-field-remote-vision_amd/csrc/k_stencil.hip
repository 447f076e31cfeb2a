// Stencil kernels: hole filling (Poisson diffusion, push-pull), the Gaussian
// smoothing of the TV weight, and the fused primal-dual ROF step.
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

struct HoleState {  // read by the host after each chunk of sweeps
    double e;
    int iters;
    int done;
};

// The diffusion's bookkeeping between sweeps: eh[j] holds the energy of sweep
// j (eh[0] = 0, the energy the first sweep is compared with); *stopped the
// number of sweeps run once the stopping rule has fired.
struct HoleLoop {
    int maxit;
    double eps;
    double *eh;      // maxit + 1
    int *stopped;
    int G;           // blocks of a sweep (its partials per sweep)
};

__global__ void k_hole_init(HoleLoop hl)
{
    if (threadIdx.x == 0) {
        hl.eh[0] = 0.0;
        *hl.stopped = 0;
    }
}

// The stopping rule of gradientIBR.cu:139-143 after sweep j (>= 1), from that
// sweep's block partials: |E_{j-1} - E_j| < eps, or j >= maxit.  Every block
// evaluates it the same way (a deterministic reduction of G partials).
__device__ __forceinline__ bool hole_rule(const HoleLoop &hl, int j, const double *pj, double *red, double &e)
{
    double v[1];
    reduce_partials<1>(pj, hl.G, v, red);
    __shared__ double eb;
    if (threadIdx.x == 0) eb = v[0];  // the sum is valid in thread 0
    __syncthreads();
    e = eb;
    return fabs(hl.eh[j - 1] - e) < hl.eps || j >= hl.maxit;
}

// *hl.stopped read once per block (every thread then takes the same branch)
__device__ __forceinline__ int hole_stopped(const HoleLoop &hl)
{
    __shared__ int sb;
    if (threadIdx.x == 0) sb = *hl.stopped;
    __syncthreads();
    return sb;
}

// Sweep k (1-based) of the Poisson diffusion: first the stopping rule of sweep
// k - 1 (so the rule needs no kernel of its own), then one Jacobi sweep
// u <- mean of the 4-neighbours (the reference's laplacian then add_to) on the
// hole pixels, all three channels, with the energy sum(lap * u_new) of the
// last channel as this sweep's block partials.  pin / pout: the partials of
// sweeps k - 1 and k.
__global__ void __launch_bounds__(256) k_hole_sweep(int W, int H, int nholes, const int *__restrict__ list,
                                                    const float *__restrict__ uin, float *__restrict__ uout,
                                                    HoleLoop hl, int k, const double *pin, double *pout)
{
    __shared__ double red[16];
    if (hole_stopped(hl)) return;
    if (k >= 2) {
        double e;
        const bool done = hole_rule(hl, k - 1, pin, red, e);
        if (blockIdx.x == 0 && threadIdx.x == 0) {
            hl.eh[k - 1] = e;
            if (done) *hl.stopped = k - 1;
        }
        if (done) return;
    }
    const size_t N = (size_t)W * H;
    double v[1] = {0.0};
    for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < nholes; k += gridDim.x * blockDim.x) {
        const int o = list[k];
        const int x = o % W, y = o / W;
        for (int c = 0; c < 3; c++) {
            const float *u = uin + c * N;
            float s = 0.0f, wsum = 0.0f;
            if (x > 0) { s += u[o - 1]; wsum += 1.0f; }
            if (y > 0) { s += u[o - W]; wsum += 1.0f; }
            if (x < W - 1) { s += u[o + 1]; wsum += 1.0f; }
            if (y < H - 1) { s += u[o + W]; wsum += 1.0f; }
            const float lap = s / wsum - u[o];
            const float un = u[o] + lap;
            uout[c * N + o] = un;
            if (c == 2) v[0] += (double)lap * (double)un;
        }
    }
    block_partials<1>(v, pout, red);
}

// The state after the last sweep `last` of a chunk, for the host: the sweeps
// run and whether the rule has fired (one block).
__global__ void __launch_bounds__(kFinalizeThreads) k_hole_state(HoleLoop hl, int last, const double *plast,
                                                                 HoleState *st)
{
    __shared__ double red[16];
    int iters = hole_stopped(hl), done = iters != 0;
    double e = 0.0;
    if (!done) {
        done = hole_rule(hl, last, plast, red, e);
        iters = last;
    }
    if (threadIdx.x == 0) {
        st->iters = iters;
        st->done = done;
        st->e = done && *hl.stopped ? hl.eh[iters] : e;
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
    HoleState *dst = reinterpret_cast<HoleState *>(ctx->scal + 16);
    float *bufs[2] = {ctx->U, ctx->tmp3N};
    LFRV_HIP(ctx, hipMemcpyAsync(ctx->tmp3N, ctx->U, 3 * N * sizeof(float), hipMemcpyDeviceToDevice, ctx->stream));
    unsigned int nb = blocks_for(nh);
    if (nb > 1024) nb = 1024;
    // partials of odd / even sweeps, the energy history and the stop flag
    HoleLoop hl;
    hl.maxit = iters;
    hl.eps = eps;
    hl.G = (int)nb;
    double *psw[2] = {ctx->partials, ctx->partials + 1024};
    hl.eh = ctx->partials + 2048;  // iters + 1 <= partials_cap - 2048, checked below
    hl.stopped = reinterpret_cast<int *>(ctx->counters + 12);
    if ((size_t)iters + 1 > ctx->partials_cap - 2048) return fail(ctx, LFRV_E_ARG, "hole filling: too many sweeps");
    k_hole_init<<<1, 64, 0, ctx->stream>>>(hl);
    int launched = 0;
    HoleState host{};
    while (launched < iters) {
        const int chunk = std::min(16, iters - launched);
        for (int j = 0; j < chunk; j++) {
            const int k = launched + j + 1;  // sweep k reads bufs[(k - 1) & 1]
            k_hole_sweep<<<nb, 256, 0, ctx->stream>>>(ctx->W, ctx->H, (int)nh, ctx->hole_list, bufs[(k - 1) & 1],
                                                      bufs[k & 1], hl, k, psw[(k - 1) & 1], psw[k & 1]);
        }
        launched += chunk;
        k_hole_state<<<1, kFinalizeThreads, 0, ctx->stream>>>(hl, launched, psw[launched & 1], dst);
        LFRV_LAUNCH(ctx, "hole filling");
        LFRV_HIP(ctx, hipMemcpyAsync(&host, dst, sizeof host, hipMemcpyDeviceToHost, ctx->stream));
        LFRV_HIP(ctx, hipStreamSynchronize(ctx->stream));
        if (host.done) break;
    }
    // the result of sweep k (1-based) is in bufs[k & 1]
    if (host.iters & 1)
        LFRV_HIP(ctx, hipMemcpyAsync(ctx->U, ctx->tmp3N, 3 * N * sizeof(float), hipMemcpyDeviceToDevice, ctx->stream));
    if (ran) *ran = host.iters;
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
    // level offsets inside the pyramid scratch: level 0 is a copy of U
    std::vector<size_t> off(levels + 1, 0);
    std::vector<int> ws(levels + 1, 0), hs(levels + 1, 0);
    size_t tot = 0;
    int top = 0;
    ws[0] = W;
    hs[0] = H;
    off[0] = 0;
    tot = N;
    for (int s = 1; s <= levels; s++) {
        const int wsn = W >> s, hsn = H >> s;
        if (wsn <= 0 || hsn <= 0) break;
        ws[s] = wsn;
        hs[s] = hsn;
        off[s] = tot;
        tot += (size_t)wsn * hsn;
        top = s;
    }
    // scratch: pyramid images (3 * tot floats) + vis pyramid (tot bytes); level 0 stays in U and the target's map
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
