// IBR_color (TV super-resolution with warped data terms): the data-term
// gradient and the outer proximal step (dsf = 1: an entry pull; dsf >= 2: the
// assembled anchor-grid operator as a stencil, fused with the first
// primal-dual iteration), the primal energy, and the re-weighting loop with
// its stopping rules on the device.
#include "strip_common.hpp"
#include "tile_common.hpp"

#include <hip/hip_ext.h>

#include <algorithm>
#include <climits>
#include <chrono>
#include <cmath>
#include <vector>

namespace lfrv {

namespace {


// Data-term gradient and the clamped gradient step for one target tile
// (vtv_sr_ista_step_unstructured, optimization.cu:1775-1812):
//   G_int  = sum_i B_i^T (omega (S_i U - v_i)) / cov * sigma^2           (:1835-1966)
//   G_grad = sum_i B_i^T ((dsf^2 S_i lap U - lap v_i) [* omega]) / cov [* sigma^2] * (-step)  (:1969-2116)
//   G = clamp(alpha G_int + beta G_grad, -1, 1);  F = clamp(U + prox_factor G, 0, 1)
// U (tile + halo KS) and lap U (tile + halo KS-1) are staged in LDS; every
// binned entry gathers both, forms the residuals and splats them back.
// Writes F (into G), Uq = U and norm_mask = cov (the reference's buffer ends
// holding the coverage).
template <int KS>
__global__ void __launch_bounds__(kPullMaxThreads) k_sr_dataterm(TileGeom g, TileEntries te, int cap, size_t n, DataTermArgs da,
                                                     const float *__restrict__ U, const float *__restrict__ views,
                                                     const float *__restrict__ vlap, const float *__restrict__ coverage,
                                                     float *__restrict__ Gout, float *__restrict__ Uq,
                                                     float *__restrict__ norm_mask, const int *halt)
{
    if (halt && *halt) return;  // a step enqueued behind a stopping rule that fired
    constexpr int HAL = KS - 1;
    extern __shared__ int smem[];
    const int t = xcd_tile(blockIdx.x, g.ntiles);
    const int tx0 = (t % g.ntx) * g.tw, ty0 = (t / g.ntx) * g.th;
    const int uw = g.tw + 2 * HAL + 2, uh = g.th + 2 * HAL + 2, up = uw * uh;  // U: halo HAL+1
    const int lw = g.tw + 2 * HAL, lh = g.th + 2 * HAL, lpp = lw * lh;         // lap U: halo HAL
    float *ul = reinterpret_cast<float *>(smem);  // 3 * up
    float *ll = ul + 3 * up;                      // 3 * lpp
    int *plds = reinterpret_cast<int *>(ll + 3 * lpp);
    const size_t N = (size_t)g.W * g.H;
    for (int i = threadIdx.x; i < up; i += blockDim.x) {
        const int x = tx0 - HAL - 1 + i % uw, y = ty0 - HAL - 1 + i / uw;
        const bool in = x >= 0 && x < g.W && y >= 0 && y < g.H;
        const size_t o = in ? (size_t)y * g.W + x : 0;
        for (int c = 0; c < 3; c++) ul[c * up + i] = in ? U[c * N + o] : 0.0f;
    }
    __syncthreads();
    const bool need_lap = da.beta > 0.0f;
    if (need_lap) {
        // cuda_laplacian_device (vtv_sr_kernels_unstructured.cu:720-761), no hole gating
        for (int i = threadIdx.x; i < lpp; i += blockDim.x) {
            const int lx = i % lw, ly = i / lw;
            const int x = tx0 - HAL + lx, y = ty0 - HAL + ly;
            const int ui = (ly + 1) * uw + lx + 1;
            for (int c = 0; c < 3; c++) {
                float v = 0.0f;
                if (x >= 0 && x < g.W && y >= 0 && y < g.H) {
                    const float *u = ul + c * up;
                    float s = 0.0f, wsum = 0.0f;
                    if (x > 0) { s += u[ui - 1]; wsum += 1.0f; }
                    if (y > 0) { s += u[ui - uw]; wsum += 1.0f; }
                    if (x < g.W - 1) { s += u[ui + 1]; wsum += 1.0f; }
                    if (y < g.H - 1) { s += u[ui + uw]; wsum += 1.0f; }
                    v = s / wsum - u[ui];
                }
                ll[c * lpp + i] = v;
            }
        }
    }
    // (the pull synchronises before it reads the staged tiles)
    any_pull<KS, 6, 0>(
        g, te, t, plds, cap,
        [&](int e, int x0, int y0, const float(&wx)[KS], const float(&wy)[KS], float om, float(&r)[6]) {
            const int k = te.src[e];
            const unsigned vi = (unsigned)k / (unsigned)n, m = (unsigned)k - vi * (unsigned)n;
            const int bx = x0 - tx0 + HAL, by = y0 - ty0 + HAL;
            float su[3] = {0, 0, 0}, sl[3] = {0, 0, 0};
#pragma unroll
            for (int i = 0; i < KS; i++)
#pragma unroll
                for (int j = 0; j < KS; j++) {
                    const float a = wy[i] * wx[j];
                    const int uidx = (by + i + 1) * uw + bx + j + 1;
                    const int lidx = (by + i) * lw + bx + j;
#pragma unroll
                    for (int c = 0; c < 3; c++) {
                        su[c] += a * ul[c * up + uidx];
                        if (need_lap) sl[c] += a * ll[c * lpp + lidx];
                    }
                }
            const float *vp = views + vi * 3 * n + m;
            const float *lp = vlap + vi * 3 * n + m;
#pragma unroll
            for (int c = 0; c < 3; c++) {
                r[c] = (da.alpha > 0.0f) ? (su[c] - vp[c * n]) * om : 0.0f;
                float rg = 0.0f;
                if (need_lap) {
                    rg = sl[c] * da.dsf2 - lp[c * n];
                    if (da.gw_type != 0) rg *= om;
                }
                r[3 + c] = rg;
            }
        },
        [&](size_t o, int x, int y, const float(&acc)[6]) {
            const float cov = coverage[o];
            const int ui = (y - ty0 + HAL + 1) * uw + (x - tx0) + HAL + 1;
#pragma unroll
            for (int c = 0; c < 3; c++) {
                float G = 0.0f;
                if (da.alpha > 0.0f) {
                    float gi = acc[c];
                    if (cov != 0.0f) gi /= cov;
                    gi *= da.sigma2;
                    G += da.alpha * gi;
                }
                if (need_lap) {
                    float gg = acc[3 + c];
                    if (cov != 0.0f) gg /= cov;
                    if (da.gw_type != 0) gg *= da.sigma2;
                    gg *= -da.grad_step;
                    G += da.beta * gg;
                }
                G = fminf(1.0f, fmaxf(-1.0f, G));
                const float uv = ul[c * up + ui];
                G *= da.prox_factor;
                G += uv;
                G = fminf(1.0f, fmaxf(0.0f, G));
                Gout[c * N + o] = G;
                Uq[c * N + o] = uv;
            }
            if (da.alpha > 0.0f || need_lap) norm_mask[o] = cov;
        });
}

// ---- dsf >= 2: the data term as an assembled operator -------------------------
//
// With t_e the 2 x 2 anchor taps of entry e (box_weights) and BU, BL the box
// sums of U and lap U at the anchors, the data-term sums of one outer step are
// linear in U while omega is fixed:
//   sum_e omega t_e (t_e^T BU - v_e)                 = G9 BU - bI
//   sum_e t_e (dsf^2 t_e^T BL - lap v_e) [* omega]     = dsf^2 G9' BL - bG
// G9 = sum omega t t^T couples each anchor with its 8 neighbours (centre, E,
// S, SE, SW planes; the others are the neighbours' couplings), G9' is the same
// without omega (gw_type 0), bI = sum omega t v, bG = sum t lap v [* omega].
// They are assembled once per set of weights (k_sr_assemble); every outer
// step is then a stencil (k_sr_step_st): box sums, the 9-point
// couplings, and the box sums back onto the pixels.  The step weighs the two
// terms' back-projections by constants of the parameters before adding them
// per pixel (cI = alpha sigma^2, cG = -beta gradient_step [sigma^2]), and the
// back-projection is linear, so with the gradient term the step back-projects
// one residual, cI (G9 BU - bI) + cG (dsf^2 G9' BL - bG), and the assembly
// stores the constant part as one plane set b = cI bI + cG bG.
//
// Anchor grid: point x' in [0, W + dsf) has box start x' + 1 - dsf; it is the
// top-left tap of the cell x' + 1 (cells hold box start cx - dsf).  Pixel x
// lies in the boxes of the points x .. x + dsf - 1.
// (kSrOpsPlanes planes: G9 (5), bI (3) or b (3) with the gradient term, G9' (5))

template <int KS>
__global__ void __launch_bounds__(kPullMaxThreads) k_sr_assemble(TileGeom g, TileEntries te, int cap, int grad,
                                                                 int gw, float ci, float cg, size_t NA,
                                                                 float *__restrict__ ops)
{
    extern __shared__ int smem[];
    constexpr int NC = 44;  // 10 weighted couplings, 12 bI taps, 12 bG taps, 10 unweighted couplings
    const int t = xcd_tile(blockIdx.x, g.ntiles);
    const int tx0 = (t % g.ntx) * g.tw, ty0 = (t / g.ntx) * g.th;
    const int ww = g.tw + 1, wh = g.th + 1, ncw = ww * wh;
    float acc[NC];
    cell_accumulate<KS, NC, false, true, 6, 1>(
        g, te, t, smem, cap, acc,
        [&](int, int, int, const float(&ax)[2], const float(&ay)[2], float om, const float(&pay)[6],
            float(&a)[NC]) {
            const float w[4] = {ay[0] * ax[0], ay[0] * ax[1], ay[1] * ax[0], ay[1] * ax[1]};  // tl tr bl br
            const float pr[10] = {w[0] * w[0], w[1] * w[1], w[2] * w[2], w[3] * w[3], w[0] * w[1],
                                  w[2] * w[3], w[0] * w[2], w[1] * w[3], w[0] * w[3], w[1] * w[2]};
#pragma unroll
            for (int k = 0; k < 10; k++) a[k] += om * pr[k];
#pragma unroll
            for (int k = 0; k < 4; k++)
#pragma unroll
                for (int c = 0; c < 3; c++) a[10 + k * 3 + c] += om * w[k] * pay[c];
            if (grad) {
                const float og = gw ? om : 1.0f;
#pragma unroll
                for (int k = 0; k < 4; k++)
#pragma unroll
                    for (int c = 0; c < 3; c++) a[22 + k * 3 + c] += og * w[k] * pay[3 + c];
#pragma unroll
                for (int k = 0; k < 10; k++) a[34 + k] += pr[k];
            }
        });
    float *part = reinterpret_cast<float *>(smem + 2 * wh + 2);
    const int c = threadIdx.x;
    if (c < ncw) {
#pragma unroll
        for (int k = 0; k < NC; k++) part[k * ncw + c] = acc[k];
    }
    __syncthreads();
    for (int p = threadIdx.x; p < g.tw * g.th; p += blockDim.x) {
        const int lx = p % g.tw, ly = p / g.tw;
        const int x = tx0 + lx, y = ty0 + ly;
        if (x >= g.Wc || y >= g.Hc) continue;
        // own cell (its tl tap), left cell (tr), upper cell (bl), upper-left cell (br)
        const int c00 = (ly + 1) * ww + lx + 1, c10 = c00 - 1, c01 = c00 - ww, c11 = c00 - ww - 1;
        const size_t o = (size_t)y * g.Wc + x;
        auto couple = [&](int base, int plane) {
            ops[(size_t)(plane + 0) * NA + o] = part[(base + 0) * ncw + c00] + part[(base + 1) * ncw + c10] +
                                                part[(base + 2) * ncw + c01] + part[(base + 3) * ncw + c11];
            ops[(size_t)(plane + 1) * NA + o] = part[(base + 4) * ncw + c00] + part[(base + 5) * ncw + c01];
            ops[(size_t)(plane + 2) * NA + o] = part[(base + 6) * ncw + c00] + part[(base + 7) * ncw + c10];
            ops[(size_t)(plane + 3) * NA + o] = part[(base + 8) * ncw + c00];
            ops[(size_t)(plane + 4) * NA + o] = part[(base + 9) * ncw + c10];
        };
        auto tap = [&](int base, int ch) {
            return part[(base + 0 * 3 + ch) * ncw + c00] + part[(base + 1 * 3 + ch) * ncw + c10] +
                   part[(base + 2 * 3 + ch) * ncw + c01] + part[(base + 3 * 3 + ch) * ncw + c11];
        };
        couple(0, 0);
#pragma unroll
        for (int ch = 0; ch < 3; ch++) {
            const float bI = tap(10, ch);
            ops[(size_t)(5 + ch) * NA + o] = grad ? ci * bI + cg * tap(22, ch) : bI;
        }
        if (grad) couple(34, 8);
    }
}

// ---- dsf >= 2: the outer step as a marching stencil -------------------------
//
// A wave owns a strip of the target, 64 columns wide with its halo, and
// marches down its rows; everything between two rows stays in its registers,
// and columns meet by DPP shifts of the wave (folded into the additions), so
// the pass has neither LDS nor barriers.  Per row, from the row of U that
// came last: lap U one row behind; the D-wide row sums of both (D = dsf), and
// their D-high column sums BU, BL kept as D - 1 partial chains; the anchor
// residuals one row behind those, q = G9 BU - bI (with the gradient term the
// weighted sum cI G9 BU + cG dsf^2 G9' BL - b; G9 the 9-point anchor couplings,
// of which five planes are stored and the other four are the neighbours' own,
// shifted over); their row sums and
// column chains back onto the pixels; the clamped gradient step F; the dual
// and primal update.  The output row lags the U row by LAG = D (+ 1 with the
// Laplacian), and LAG columns at each end of the wave are halo: 54 - 60 of the
// 64 lanes have an output.
// Bounds: at large targets the bytes of the step (25 views, 2048^2, dsf 4: 555
// MB in 140 us, 4.0 TB/s; 188 us before), at small ones the latency of the rows
// of one wave (256^2, dsf 2: 6.4 us per step; 7.1 before), in a batch at dsf 2
// with the gradient term the instructions.  The tile form this replaced (32 x
// 16 pixels, nine LDS phases, 2.1 x halo loads) was bound by its LDS and address
// instructions.  Sums run in its order, contractions are written out and the
// projected duals are rounded before they are summed (product), so that the
// results are its own bit for bit: compared at dsf 1 to 4, with and without the
// gradient term, over 50 to 500 steps of several scenes.
// Loads and stores go through buffer descriptors, and a lane or row outside
// its plane takes the offset kOutside, past every buffer: it reads 0 and writes
// nothing, without a compare per value.  Every row issues the same loads and
// stores, outside any branch, so that the waits count exactly the younger ones
// and the next two rows' loads stay in flight.  The rows before the first
// output are peeled off (they need only part of the row's work).
// The arithmetic of a pixel does not depend on the strip it falls in, so
// strips of any height, and batches, give the same bits.

template <int D, bool GRAD>
struct Strip {
    static constexpr int LAG = D + (GRAD ? 1 : 0), OW = 64 - 2 * LAG;  // output columns
};

// The step's buffers (U read, the rest nullable where the caller's form skips it).
struct StepBufs {
    const float *U, *ops, *coverage, *px, *py, *g;
    float *pxout, *pyout, *unew, *uq_relax, *gout, *norm_mask;
};

// Rows y0 .. y1 - 1 of the strip whose first output column is x0.  With PD the
// data term and the first primal-dual iteration (k_pd_steps' update, with
// Uq = U as the step sets it, optimization.cu:1765-1767): the new primal goes
// to unew, with uq_relax the over-relaxed one (vtv_rof.cu:28-45) there, with
// gout F.  Without PD F goes to gout and U to uq_relax.  EXTRA: one of
// uq_relax, gout and norm_mask is given.
template <int D, bool GRAD, bool PD, bool EXTRA, bool WIDE>
__device__ __forceinline__ void sr_strip(int x0, int y0, int y1, int W, int H, int Wc, int Hc, size_t NA,
                                         const DataTermArgs &da, const PdArgs &pa, const StepBufs &sb)
{
    constexpr int LAG = Strip<D, GRAD>::LAG, OW = Strip<D, GRAD>::OW, RING = LAG < kStripGroup ? kStripGroup : 2 * kStripGroup, NB = 3, G = GRAD ? 1 : 0;
    static_assert(LAG < RING && kStripGroup % NB == 0, "the ring holds the rows from the output row to the newest");
    const size_t N = (size_t)W * H;
    const int lane = threadIdx.x & 63, x = x0 - LAG + lane;
    const bool xin = x >= 0 && x < W;
    const int vx = xin ? 4 * x : kOutside, vc = x >= 0 && x < Wc ? 4 * x : kOutside;
    const int vs = lane >= LAG && lane < LAG + OW ? vx : kOutside;  // the lanes with an output
    // cuda_laplacian_device (vtv_sr_kernels_unstructured.cu:720-761), no hole gating: the mean of the neighbours
    // inside the image, on inner and on edge rows
    const float nx = (x > 0 ? 1.0f : 0.0f) + (x < W - 1 ? 1.0f : 0.0f);
    const float n_inner = xin ? nx + 2.0f : 1.0f, n_edge = xin ? nx + (H > 1 ? 1.0f : 0.0f) : 1.0f;
    const float r_inner = 1.0f / n_inner, r_edge = 1.0f / n_edge;
    const float ci = dt_intensity_weight(da), cgd = dt_gradient_weight(da) * da.dsf2;
    const Divisor vden(pa.tau + pa.lam);
    const float vtau = pa.tau * vden.scale, vlam = pa.lam * vden.scale;
    const int has_right = lane_mask(xin && x < W - 1);
    const float gnone = sb.g ? 0.0f : 1.0f;  // the TV weight where there is no map
    const Planes<WIDE> bU(sb.U, 3, N, W), bC(sb.ops, 5, NA, Wc), bB(sb.ops + 5 * NA, 3, NA, Wc),
        bE(da.gw_type ? sb.ops : sb.ops + 8 * NA, GRAD ? 5 : 0, NA, Wc), bPx(sb.px, 3, N, W), bPy(sb.py, 3, N, W),
        bG(sb.g, 1, N, W), bCov(sb.coverage, 1, N, W), bPxo(sb.pxout, 3, N, W), bPyo(sb.pyout, 3, N, W),
        bUn(sb.unew, 3, N, W), bUq(sb.uq_relax, 3, N, W), bGo(sb.gout, 3, N, W), bNm(sb.norm_mask, 1, N, W);
    const int first = y0 - LAG, yend = y1 + LAG;  // rows of U

    // the loads of one row: U's new row, the operator one row behind the box sums, the output row's own
    struct Loads {
        float u[3], f[1 + G][5], b[3], p[PD ? 6 : 1], g, cov;
    } ld[NB];
    auto fetch = [&](Loads &l, int yn) __attribute__((always_inline)) {
        const int yq = yn - G - 1, yo = yn - LAG;
        const int vu = yn >= 0 && yn < min(H, yend) ? vx : kOutside;
        const int vq = yq >= max(0, y0 - 1) && yq < Hc && yn < yend ? vc : kOutside;
        const int vp = yo >= max(0, y0 - 1) && yo < y1 ? vx : kOutside;
#pragma unroll
        for (int c = 0; c < 3; c++) l.u[c] = bU.load(c, yn, vu);
#pragma unroll
        for (int k = 0; k < 5; k++) {
            l.f[0][k] = bC.load(k, yq, vq);
            if constexpr (GRAD) l.f[G][k] = bE.load(k, yq, vq);
        }
#pragma unroll
        for (int c = 0; c < 3; c++) l.b[c] = bB.load(c, yq, vq);
        l.cov = bCov.load(0, yo, vp);
        if constexpr (PD) {
#pragma unroll
            for (int c = 0; c < 3; c++) {
                l.p[c] = bPx.load(c, yo, vp);
                l.p[3 + c] = bPy.load(c, yo, vp);
            }
            l.g = bG.load(0, yo, vp);
        }
    };
    float u[RING][3];                       // U's last rows
    float bc[1 + G][3][D - 1];              // column chains of U's and lap U's row sums
    // BU, BL of the two rows before the newest, at the lane's left, own and right anchor
    float bm[1 + G][3][3], b0[1 + G][3][3];
    // the operator row above: its south, the left neighbour's south-east, the right one's south-west
    float s1[1 + G], s2[1 + G], s3[1 + G];
    float qc[3][D - 1], py1[3];             // column chains of the residuals' row sums; the duals of the row above
#pragma unroll
    for (int c = 0; c < 3; c++) {
#pragma unroll
        for (int k = 0; k < RING; k++) u[k][c] = 0.0f;
#pragma unroll
        for (int t = 0; t <= G; t++) {
#pragma unroll
            for (int d = 0; d < 3; d++) bm[t][c][d] = b0[t][c][d] = 0.0f;
#pragma unroll
            for (int d = 0; d < D - 1; d++) bc[t][c][d] = 0.0f;
        }
#pragma unroll
        for (int d = 0; d < D - 1; d++) qc[c][d] = 0.0f;
        py1[c] = 0.0f;
    }
#pragma unroll
    for (int t = 0; t <= G; t++) s1[t] = s2[t] = s3[t] = 0.0f;
    // the sum of the last D rows' values, added from the oldest on
    auto chain = [](float(&ch)[D - 1], float v) __attribute__((always_inline)) {
        const float sum = ch[D - 2] + v;
#pragma unroll
        for (int d = D - 2; d > 0; d--) ch[d] = ch[d - 1] + v;
        ch[0] = v;
        return sum;
    };
    // Row first + i with k = i modulo RING.  PHASE 0: box sums only; 1: and the residuals; 2: and the duals of
    // row y0 - 1; 3: an output row.
    auto row = [&](auto K, auto PHASE, int i) __attribute__((always_inline)) {
        constexpr int k = decltype(K)::value, ph = decltype(PHASE)::value;
        constexpr int ku = k % RING, k1 = (k + RING - 1) % RING, k2 = (k + RING - 2) % RING,
                      ko = (k + RING - LAG) % RING;
        const int yn = first + i, yb = yn - G, yo = yn - LAG;
        const Loads &l = ld[k % NB];
        fetch(ld[(k + 2) % NB], yn + 2);
#pragma unroll
        for (int c = 0; c < 3; c++) u[ku][c] = l.u[c];
        // row sums of U and lap U at row yb, BU and BL of the anchor row yb
        float bp[1 + G][3][3];
        // (+: of the values; a choice between the captured variables would keep them all in memory)
        const bool inner = yb > 0 && yb < H - 1;
        const float n4 = inner ? +n_inner : +n_edge, r4 = inner ? +r_inner : +r_edge;
        const bool bin = xin && yb >= 0 && yb < H;
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const float uc = GRAD ? u[k1][c] : u[ku][c];
            if constexpr (GRAD) {
                const float sum = ((from_left(uc) + u[k2][c]) + from_right(uc)) + u[ku][c];
                float t = small_quotient(sum, n4, r4) - uc;
                t = bin ? t : 0.0f;
                float rs = t;
#pragma unroll
                for (int d = 1; d < D; d++) rs = t + from_left(rs);
                bp[G][c][1] = chain(bc[G][c], rs);
            }
            float rs = uc;
#pragma unroll
            for (int d = 1; d < D; d++) rs = uc + from_left(rs);
            bp[0][c][1] = chain(bc[0][c], rs);
#pragma unroll
            for (int t = 0; t <= G; t++) {
                bp[t][c][0] = from_left(bp[t][c][1]);
                bp[t][c][2] = from_right(bp[t][c][1]);
            }
        }
        float up[3] = {0, 0, 0}, acc[3] = {0, 0, 0};
        if constexpr (ph >= 1) {
            // residuals of the anchor row yb - 1, and back onto the pixels of row yo
            float fw[1 + G];  // west: the left neighbour's own east
#pragma unroll
            for (int t = 0; t <= G; t++) fw[t] = from_left(l.f[t][1]);
#pragma unroll
            for (int c = 0; c < 3; c++) {
                float st[1 + G];
#pragma unroll
                for (int t = 0; t <= G; t++) {
                    const float *f = l.f[t], *m = bm[t][c], *z = b0[t][c], *p = bp[t][c];  // (left, own, right)
                    float w = fmaf(f[0], z[1], f[1] * z[2]);
                    w = fmaf(f[2], p[1], fmaf(fw[t], z[0], w));
                    w = fmaf(f[3], p[2], fmaf(s1[t], m[1], w));
                    w = fmaf(f[4], p[0], fmaf(s2[t], m[0], w));
                    st[t] = fmaf(s3[t], m[2], w);
                }
                const float q = (GRAD ? fmaf(ci, st[0], cgd * st[G]) : st[0]) - l.b[c];
                float rs = q, qr = q;
#pragma unroll
                for (int d = 1; d < D; d++) {
                    qr = from_right(qr);
                    rs += qr;
                }
                acc[c] = chain(qc[c], rs);
                up[c] = u[ko][c];  // LAG rows ago
            }
        }
        float a[3] = {0, 0, 0}, b[3] = {0, 0, 0};
        if constexpr (PD && ph >= 2) {
            // the duals (vtv_rof.cu:118-147, 280-321)
            const int has_below = mask_below(yo, H - 1);
            float nn = 0.0f;
#pragma unroll
            for (int c = 0; c < 3; c++) {
                const float gx = from_right(up[c]) - up[c], gy = u[(ko + 1) % RING][c] - up[c];
                a[c] = fmaf(pa.sigma, where(has_right, gx), l.p[c]);
                b[c] = fmaf(pa.sigma, where(has_below, gy), l.p[3 + c]);
                nn += fmaf(a[c], a[c], b[c] * b[c]);
            }
            nn = sqrtf(nn);
            const float gr = l.g + gnone, ratio = gr / nn, sc = nn > gr ? ratio : 1.0f;
#pragma unroll
            for (int c = 0; c < 3; c++) {
                a[c] = product(a[c], sc);
                b[c] = product(b[c], sc);
            }
        }
        if constexpr (ph == 3) {
            // the step of vtv_sr_ista_step_unstructured, and the primal (cuda_kernels.cu:504-532)
            const int vo = yo < y1 ? vs : kOutside;
            // (a lane with a coverage that a division would have to scale is rare: the wave divides then)
            const float cov = l.cov != 0.0f ? l.cov : 1.0f;
            float quot[3];
            if (__all(Divisor::plain(cov))) {
                const Divisor by(cov, 1.0f);
#pragma unroll
                for (int c = 0; c < 3; c++) quot[c] = by.of_scaled(acc[c]);
            } else {
#pragma unroll
                for (int c = 0; c < 3; c++) quot[c] = acc[c] / cov;
            }
#pragma unroll
            for (int c = 0; c < 3; c++) {
                float Gv = quot[c];
                if constexpr (!GRAD) Gv = da.alpha > 0.0f ? da.alpha * (Gv * da.sigma2) : 0.0f;
                Gv = fminf(1.0f, fmaxf(-1.0f, Gv));
                const float F = fminf(1.0f, fmaxf(0.0f, fmaf(Gv, da.prox_factor, up[c])));
                float rel = up[c];
                if constexpr (PD) {
                    // (left of the image U and the duals read 0)
                    const float step = a[c] + b[c] - from_left(a[c]) - py1[c];
                    const float un = fmaf(pa.tau, step, up[c]);
                    const float v = vden.of_scaled(fmaf(vtau, F, vlam * un));
                    rel = fmaf(pa.theta, v - up[c], up[c]);
                    bPxo.store(a[c], c, yo, vo);
                    bPyo.store(b[c], c, yo, vo);
                    bUn.store(v, c, yo, vo);
                }
                if constexpr (EXTRA) {
                    bUq.store(rel, c, yo, vo);
                    bGo.store(F, c, yo, vo);
                }
            }
            if constexpr (EXTRA) bNm.store(l.cov, 0, yo, vo);
        }
        if constexpr (PD && ph >= 2) {
#pragma unroll
            for (int c = 0; c < 3; c++) py1[c] = b[c];
        }
#pragma unroll
        for (int t = 0; t <= G; t++) {
            s1[t] = l.f[t][2];
            s2[t] = from_left(l.f[t][3]);
            s3[t] = from_right(l.f[t][4]);
#pragma unroll
            for (int c = 0; c < 3; c++)
#pragma unroll
                for (int d = 0; d < 3; d++) {
                    bm[t][c][d] = b0[t][c][d];
                    b0[t][c][d] = bp[t][c][d];
                }
        }
    };
#pragma unroll
    for (int k = 0; k < 2; k++) fetch(ld[k], first + k);
    constexpr int WARM = 2 * LAG;  // rows before the first output
    static_for<WARM>([&](auto K) __attribute__((always_inline)) {
        constexpr int i = decltype(K)::value;
        row(K, std::integral_constant<int, (i == WARM - 1 ? 2 : i > D + 2 * G ? 1 : 0)>(), i);
    });
    // whole groups of kStripGroup rows, those past y1 without bytes: a branch between rows would cost the state's
    // registers a move each.  A ring of two groups changes halves after each, so that its indices stay the same.
    for (int j0 = 0; j0 < y1 - y0; j0 += kStripGroup) {
        static_for<kStripGroup>([&](auto J) __attribute__((always_inline)) {
            constexpr int j = decltype(J)::value;
            row(std::integral_constant<int, WARM + j>(), std::integral_constant<int, 3>(), WARM + j0 + j);
        });
        if constexpr (RING == 2 * kStripGroup)
#pragma unroll
            for (int k = 0; k < kStripGroup; k++)
#pragma unroll
                for (int c = 0; c < 3; c++) {
                    const float t = u[k][c];
                    u[k][c] = u[k + kStripGroup][c];
                    u[k + kStripGroup][c] = t;
                }
    }
}

template <int D, bool GRAD, bool PD, bool EXTRA, bool WIDE>
__device__ __forceinline__ void sr_block(int b, StripGeom sg, int W, int H, int Wc, int Hc, size_t NA,
                                         const DataTermArgs &da, const PdArgs &pa, const StepBufs &sb)
{
    const int strip = __builtin_amdgcn_readfirstlane(4 * b + (int)(threadIdx.x >> 6));
    const int sy = strip / sg.nx, sx = strip - sy * sg.nx, y0 = sy * sg.rows;
    if (y0 >= H) return;
    sr_strip<D, GRAD, PD, EXTRA, WIDE>(sx * Strip<D, GRAD>::OW, y0, min(y0 + sg.rows, H), W, H, Wc, Hc, NA, da, pa, sb);
}

// One outer step for dsf >= 2 (PD), or its data term alone.  U is only read.
// uq_relax and norm_mask are nullable: a run of fixed steps reads neither
// between its steps (the next step starts from the new primal, and the mask
// is the coverage again), so only its last step writes them.
template <int KS, bool GRAD, bool PD, bool EXTRA, bool WIDE>
__global__ void __launch_bounds__(256) k_sr_step_st(int W, int H, int Wc, int Hc, StripGeom sg, DataTermArgs da, PdArgs pa,
                                                    size_t NA, StepBufs sb, const int *halt)
{
    if (halt && *halt) return;  // a step enqueued behind a stopping rule that fired
    sr_block<KS - 1, GRAD, PD, EXTRA, WIDE>(xcd_tile(blockIdx.x, sg.nblocks), sg, W, H, Wc, Hc, NA, da, pa, sb);
}

// Step s of every IBR_color solve of a batch in one launch: block b runs block
// xcd_tile(j, nblocks) of solve k, (k, j) = work[b], as in that solve's own
// k_sr_step_st launch (the same arithmetic), on the buffers of step parity
// s & 1; a solve with fewer steps returns.  Only a solve's last step writes Uq
// and the norm mask, as in its own run.
template <int KS, bool GRAD>
__global__ void __launch_bounds__(256) k_sr_step_st_batch(const SrBatchItem *__restrict__ items,
                                                          const int2 *__restrict__ work, int s)
{
    const int2 wk = work[blockIdx.x];
    const SrBatchItem &it = items[wk.x];
    if (s >= it.steps) return;
    const int p = s & 1;
    PdArgs pa = it.pa;
    pa.theta = it.theta[s];
    const bool last = s == it.steps - 1;
    const StepBufs sb{it.U[p],         it.ops,       it.coverage, it.PX[p], it.PY[p], it.g, it.PX[p ^ 1], it.PY[p ^ 1],
                      it.U[p ^ 1], last ? it.uq : nullptr, nullptr,     last ? it.norm_mask : nullptr};
    const StripGeom sg = it.sg;
    if (last)
        sr_block<KS - 1, GRAD, true, true, false>(xcd_tile(wk.y, sg.nblocks), sg, it.W, it.H, it.Wc, it.Hc, it.NA, it.da, pa, sb);
    else
        sr_block<KS - 1, GRAD, true, false, false>(xcd_tile(wk.y, sg.nblocks), sg, it.W, it.H, it.Wc, it.Hc, it.NA, it.da, pa, sb);
}

// ---- further primal-dual iterations -------------------------------------------
//
// Inner iterations of vtv_sr_ista_step_unstructured (optimization.cu:1817-1828):
//   dual:   p_c <- p_c + sigma grad+ Uq_c           (vtv_rof.cu:118-147)
//   proj:   joint TV_F projection onto |p| <= g      (vtv_rof.cu:280-321; radius 1 without g, :237-275)
//   primal: Uq_c <- (tau F_c + lam (Uq_c + tau div- p_c)) / (tau + lam)   (cuda_kernels.cu:504-532)
// K of them in one pass of the marching strips: iteration j takes row y of the
// iteration before it as soon as that row and the next are there, one row and
// one column behind, so U, the duals, F and g cross memory once per K
// iterations.  One pass of 431 x 322: 3 iterations in 12 us, where a pass per
// iteration (64 x 4 tiles) took 8.2 us each.
// With u_final (the last iterations of an outer step) the over-relaxation of
// the outer step is fused in (vtv_rof.cu:28-45): u_final <- the new primal,
// uout <- u_final_old + theta (new primal - u_final_old).
struct PdBufs {
    const float *uin, *px, *py, *F, *g;
    float *uout, *pxout, *pyout, *u_final;
};

template <int K, bool WIDE>
__device__ __forceinline__ void pd_strip(int x0, int y0, int y1, int W, int H, const PdArgs &pa, const PdBufs &pb)
{
    const size_t N = (size_t)W * H;
    const int lane = threadIdx.x & 63, x = x0 - K + lane;
    const bool xin = x >= 0 && x < W;
    const int vx = xin ? 4 * x : kOutside, vs = lane >= K && lane < 64 - K ? vx : kOutside;
    const Divisor vden(pa.tau + pa.lam);
    const float vtau = pa.tau * vden.scale, vlam = pa.lam * vden.scale;
    const int has_right = lane_mask(xin && x < W - 1);
    const float gnone = pb.g ? 0.0f : 1.0f;
    const Planes<WIDE> bU(pb.uin, 3, N, W), bPx(pb.px, 3, N, W), bPy(pb.py, 3, N, W), bF(pb.F, 3, N, W), bG(pb.g, 1, N, W),
        bUo(pb.uout, 3, N, W), bPxo(pb.pxout, 3, N, W), bPyo(pb.pyout, 3, N, W), bUf(pb.u_final, 3, N, W);
    const int first = y0 - K, yend = y1 + K;  // rows of U
    struct Loads {
        float u[3], p[6], F[3], g, uf[3];
    } ld[3];
    auto fetch = [&](Loads &l, int yn) __attribute__((always_inline)) {
        const int yp = yn - 1, yo = yn - K;
        const int vu = yn >= 0 && yn < min(H, yend) ? vx : kOutside;
        const int vp = yp >= 0 && yp < H && yn < yend ? vx : kOutside;
        const int vf = yo >= y0 && yo < y1 ? vs : kOutside;
#pragma unroll
        for (int c = 0; c < 3; c++) {
            l.u[c] = bU.load(c, yn, vu);
            l.p[c] = bPx.load(c, yp, vp);
            l.p[3 + c] = bPy.load(c, yp, vp);
            l.F[c] = bF.load(c, yp, vp);
            l.uf[c] = bUf.load(c, yo, vf);
        }
        l.g = bG.load(0, yp, vp);
    };
    // iteration j: U's last row, and for j > 0 the duals, F and g of that row, as iteration j - 1 left them a turn
    // ago; the y part of its own duals a row up
    float u[K][3], p[K][6], F[K][3], g[K], py[K][3];
#pragma unroll
    for (int j = 0; j < K; j++) {
        g[j] = 0.0f;
#pragma unroll
        for (int c = 0; c < 3; c++) u[j][c] = p[j][c] = p[j][3 + c] = py[j][c] = F[j][c] = 0.0f;
    }
    auto row = [&](auto B, int yn) __attribute__((always_inline)) {
        constexpr int k = decltype(B)::value;
        const Loads &l = ld[k % 3];
        fetch(ld[(k + 2) % 3], yn + 2);
        float un[3], cp[6], cF[3], cg = l.g + gnone;  // to iteration j: its new row of U; duals, F, g of the row above
#pragma unroll
        for (int c = 0; c < 3; c++) {
            un[c] = l.u[c];
            cF[c] = l.F[c];
            cp[c] = l.p[c];
            cp[3 + c] = l.p[3 + c];
        }
#pragma unroll
        for (int j = 0; j < K; j++) {
            const int y = yn - 1 - j;  // the row this iteration completes
            const bool yin = y >= 0 && y < H;
            const int has_below = mask_below(y, H - 1);
            if (j > 0) {
                // what came from iteration j - 1 is for the next turn
                const float tg = g[j];
                g[j] = cg;
                cg = tg;
#pragma unroll
                for (int c = 0; c < 6; c++) {
                    const float t = p[j][c];
                    p[j][c] = cp[c];
                    cp[c] = t;
                }
#pragma unroll
                for (int c = 0; c < 3; c++) {
                    const float t = F[j][c];
                    F[j][c] = cF[c];
                    cF[c] = t;
                }
            }
            float nn = 0.0f;
#pragma unroll
            for (int c = 0; c < 3; c++) {
                const float gx = from_right(u[j][c]) - u[j][c], gy = un[c] - u[j][c];
                cp[c] = fmaf(pa.sigma, where(has_right, gx), cp[c]);
                cp[3 + c] = fmaf(pa.sigma, where(has_below, gy), cp[3 + c]);
                nn += fmaf(cp[c], cp[c], cp[3 + c] * cp[3 + c]);
            }
            nn = sqrtf(nn);
            const float ratio = cg / nn, sc = nn > cg ? ratio : 1.0f;  // (outside the image the duals read and stay 0)
#pragma unroll
            for (int c = 0; c < 3; c++) {
                cp[c] = product(cp[c], sc);
                cp[3 + c] = product(cp[3 + c], sc);
                const float step = cp[c] + cp[3 + c] - from_left(cp[c]) - py[j][c];
                const float v = vden.of_scaled(fmaf(vtau, cF[c], vlam * fmaf(pa.tau, step, u[j][c])));
                py[j][c] = cp[3 + c];
                u[j][c] = un[c];
                un[c] = xin && yin ? +v : 0.0f;
            }
        }
        const int yo = yn - K, vo = yo >= y0 && yo < y1 ? vs : kOutside;
#pragma unroll
        for (int c = 0; c < 3; c++) {
            bPxo.store(cp[c], c, yo, vo);
            bPyo.store(cp[3 + c], c, yo, vo);
            const float rel = fmaf(pa.theta, un[c] - l.uf[c], l.uf[c]);
            bUo.store(pb.u_final ? rel : un[c], c, yo, vo);
            bUf.store(un[c], c, yo, vo);
        }
    };
#pragma unroll
    for (int k = 0; k < 2; k++) fetch(ld[k], first + k);
    for (int yn = first; yn < yend; yn += kStripGroup)
        static_for<kStripGroup>([&](auto B) __attribute__((always_inline)) { row(B, yn + decltype(B)::value); });
}

template <int K, bool WIDE>
__global__ void __launch_bounds__(256) k_pd_steps(int W, int H, StripGeom sg, PdArgs pa, PdBufs pb, const int *halt)
{
    if (halt && *halt) return;  // a step enqueued behind a stopping rule that fired
    const int strip = __builtin_amdgcn_readfirstlane(4 * xcd_tile(blockIdx.x, sg.nblocks) + (int)(threadIdx.x >> 6));
    const int sy = strip / sg.nx, sx = strip - sy * sg.nx, y0 = sy * sg.rows;
    if (y0 >= H) return;
    pd_strip<K, WIDE>(sx * (64 - 2 * K), y0, min(y0 + sg.rows, H), W, H, pa, pb);
}

// theta over-relaxation (vtv_rof.cu:28-45): uq <- u + theta (uq - u); u <- uq_old
__global__ void k_overrelax(size_t n3, float theta, float *__restrict__ uq, float *__restrict__ u, const int *halt)
{
    if (halt && *halt) return;
    const size_t k = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n3) return;
    const float uv = u[k], uqv = uq[k];
    uq[k] = uv + theta * (uqv - uv);
    u[k] = uqv;
}

// E_TV over pixels whose 3x3 neighbourhood is visible, and the ungated Sobel
// of Y(U) for the gradient term (optimization.cu:1505-1534, 1622-1625).
// With prev2 (two 3N buffers, the loop state L saying which one holds the
// previous solution), the same pass also counts the pixels of U that moved
// against it (the count of k_count_moving, block partials at pmove) and
// writes U into the other buffer: if the step's rules keep it, that buffer
// becomes the previous solution (k_sr_loop_step flips L->cur).
__global__ void __launch_bounds__(256) k_sr_energy_tv(int W, int H, const float *__restrict__ U,
                                                      const float *__restrict__ vis, float *__restrict__ ugx,
                                                      float *__restrict__ ugy, double *partials, const int *halt,
                                                      float *__restrict__ prev2, const SrLoop *L, float thr,
                                                      double *pmove)
{
    if (halt && *halt) return;
    __shared__ double red[16], red_m[16];
    const size_t N = (size_t)W * H;
    const int cur = prev2 ? L->cur : 0;
    const float *prev = prev2 ? prev2 + (size_t)cur * 3 * N : nullptr;
    float *next = prev2 ? prev2 + (size_t)(cur ^ 1) * 3 * N : nullptr;
    double v[1] = {0.0}, vm[1] = {0.0};
    for (size_t o = (size_t)blockIdx.x * blockDim.x + threadIdx.x; o < N; o += (size_t)gridDim.x * blockDim.x) {
        if (prev2) {
            double mx = 0.0;
            for (int c = 0; c < 3; c++) {
                const float u = U[c * N + o];
                mx = fmax(mx, fabs((double)u - (double)prev[c * N + o]));
                next[c * N + o] = u;
            }
            if (!(mx < (double)thr)) vm[0] += 1.0;
        }
        const int ox = (int)(o % W), oy = (int)(o / W);
        float GX = 0.0f, GY = 0.0f;
        bool ok = false;
        if (0 < ox && ox < W - 1 && 0 < oy && oy < H - 1) {
            const float *r = U, *g = U + N, *b = U + 2 * N;
            auto Y = [&](long d) { return 0.2126f * r[o + d] + 0.7152f * g[o + d] + 0.0722f * b[o + d]; };
            const float Ypp = Y(-W - 1), Ypc = Y(-W), Ypn = Y(-W + 1);
            const float Ycp = Y(-1), Ycn = Y(1);
            const float Ynp = Y(W - 1), Ync = Y(W), Ynn = Y(W + 1);
            GX = (Ypn + 2.0f * Ycn + Ynn - Ypp - 2.0f * Ycp - Ynp) * 0.125f;
            GY = (Ynp + 2.0f * Ync + Ynn - Ypp - 2.0f * Ypc - Ypn) * 0.125f;
            ok = true;
            for (int dy = -1; dy <= 1 && ok; dy++)
                for (int dx = -1; dx <= 1; dx++)
                    if (vis[o + (long)dy * W + dx] == 0.0f) ok = false;
        }
        ugx[o] = GX;
        ugy[o] = GY;
        if (ok) v[0] += fabs((double)GX) + fabs((double)GY);
    }
    block_partials<1>(v, partials, red);
    if (prev2) block_partials<1>(vm, pmove, red_m);
}

// E_int and E_grad over every (view, pixel) with gather validity
// (optimization.cu:1549-1606, 1611-1704).
template <int KS>
__global__ void __launch_bounds__(256) k_sr_energy_views(int V, int W, int H, int w, int h,
                                                         const float *__restrict__ tx, const float *__restrict__ ty,
                                                         const float *__restrict__ omega, const float *__restrict__ views,
                                                         const float *__restrict__ vgrad, const float *__restrict__ U,
                                                         const float *__restrict__ ugx, const float *__restrict__ ugy,
                                                         float sigma2, int gw_type, double *partials,
                                                         const int *halt)
{
    if (halt && *halt) return;
    __shared__ double red[2 * 16];
    const size_t n = (size_t)w * h, N = (size_t)W * H;
    double v[2] = {0.0, 0.0};
    for (size_t k = (size_t)blockIdx.x * blockDim.x + threadIdx.x; k < (size_t)V * n;
         k += (size_t)gridDim.x * blockDim.x) {
        const size_t vi = k / n, m = k - vi * n;
        const float t0 = tx[k], t1 = ty[k];
        float s[5] = {0, 0, 0, 0, 0};
        int x0, y0;
        float wx[KS], wy[KS];
        if (gather_valid(t0, t1, W, H) && footprint<KS>(t0, t1, W, H, x0, y0, wx, wy)) {
            for (int i = 0; i < KS; i++) {
                const int y = y0 + i;
                if (y < 0 || y > H - 1) continue;
                for (int j = 0; j < KS; j++) {
                    const int x = x0 + j;
                    if (x < 0 || x > W - 1) continue;
                    const float a = wy[i] * wx[j];
                    const size_t o = (size_t)y * W + x;
                    s[0] += a * U[o];
                    s[1] += a * U[N + o];
                    s[2] += a * U[2 * N + o];
                    s[3] += a * ugx[o];
                    s[4] += a * ugy[o];
                }
            }
        }
        const float om = omega[k];
        for (int c = 0; c < 3; c++) {
            const float r = s[c] - views[vi * 3 * n + c * n + m];
            v[0] += (double)(r * r) * (double)om * (double)sigma2;
        }
        float a = s[3] - vgrad[vi * 2 * n + m], b = s[4] - vgrad[vi * 2 * n + n + m];
        a *= a;
        b *= b;
        if (gw_type != 0) {
            a = a * om * sigma2;
            b = b * om * sigma2;
        }
        v[1] += (double)a + (double)b;
    }
    block_partials<2>(v, partials, red);
}

__global__ void __launch_bounds__(256) k_count_moving(size_t N, const float *__restrict__ U,
                                                      const float *__restrict__ prev, float thr,
                                                      double *partials, const int *halt)
{
    if (halt && *halt) return;
    __shared__ double red[16];
    double v[1] = {0.0};
    for (size_t o = (size_t)blockIdx.x * blockDim.x + threadIdx.x; o < N; o += (size_t)gridDim.x * blockDim.x) {
        // the difference in double, as sr_compare_images takes it of its double planes
        double mx = 0.0;
        for (int c = 0; c < 3; c++) mx = fmax(mx, fabs((double)U[c * N + o] - (double)prev[c * N + o]));
        if (!(mx < (double)thr)) v[0] += 1.0;
    }
    block_partials<1>(v, partials, red);
}

unsigned int rblocks(size_t N)
{
    const size_t b = (N + kBlock - 1) / kBlock;
    return (unsigned int)(b < 2048 ? (b == 0 ? 1 : b) : 2048);
}

// The energy's block partials: E_TV at partials[0, 2048), E_int and E_grad
// at partials + 2048 (2 x up to 2048 blocks).
constexpr size_t kViewPartials = 2048;

struct EnergyCoef {
    double lambda, alpha, beta;
};

// The energy of the driver, E = lambda E_TV + dt_alpha E_int + dt_beta E_grad
// (optimization.cu:1710), from the block partials; the driver keeps it in
// float (super-resolution.cpp:181, 230).  The sum in the host's order,
// without contraction into FMAs.
__device__ __forceinline__ float sr_loop_energy(const double (&tv)[1], const double (&dv)[2], const EnergyCoef &c)
{
    return (float)__dadd_rn(__dadd_rn(__dmul_rn(c.lambda, tv[0]), __dmul_rn(c.alpha, dv[0])),
                            __dmul_rn(c.beta, dv[1]));
}

// The pass's starting energy (super-resolution.cpp:207-209), which also opens
// the pass.
__global__ void __launch_bounds__(kFinalizeThreads) k_sr_loop_begin(SrLoop *L, const double *__restrict__ ptv, int Gtv,
                                                                  const double *__restrict__ pviews, int Gv,
                                                                  EnergyCoef c)
{
    __shared__ double red[2 * 16];
    double tv[1], dv[2];
    reduce_partials<1>(ptv, Gtv, tv, red);
    reduce_partials<2>(pviews, Gv, dv, red);
    if (threadIdx.x != 0) return;
    const float E = sr_loop_energy(tv, dv, c);
    L->parts[0] = tv[0];
    L->parts[1] = dv[0];
    L->parts[2] = dv[1];
    L->energy = E;
    L->halt = 0;
    L->steps = 0;
    L->stop = LFRV_SR_STOP_MAXIT;
    L->prev_energy = E;
}

// The rules after a FISTA step, in the driver's order: E < 1e-4 stops;
// |(E - E_prev) / E| < 1e-4 stops; else E_prev = E (super-resolution.cpp:
// 230-244), and fewer than pct of the pixels moved against the previous
// step's solution stops (:246-257), on the count the step's energy pass took
// (k_sr_energy_tv with prev2; its block partials at pmove); a step the rules
// keep becomes the previous solution.
__global__ void __launch_bounds__(kFinalizeThreads) k_sr_loop_step(SrLoop *L, const double *__restrict__ ptv, int Gtv,
                                                                 const double *__restrict__ pviews, int Gv,
                                                                 EnergyCoef c, float eps,
                                                                 const double *__restrict__ pmove, int Gm,
                                                                 float npix, float pct)
{
    if (L->halt) return;
    __shared__ double red[2 * 16];
    double tv[1], dv[2], m[1];
    reduce_partials<1>(ptv, Gtv, tv, red);
    reduce_partials<2>(pviews, Gv, dv, red);
    reduce_partials<1>(pmove, Gm, m, red);
    if (threadIdx.x != 0) return;
    const float E = sr_loop_energy(tv, dv, c);
    L->parts[0] = tv[0];
    L->parts[1] = dv[0];
    L->parts[2] = dv[1];
    L->energy = E;
    L->steps += 1;
    if (E < eps) {
        L->halt = 1;
        L->stop = LFRV_SR_STOP_ENERGY;
    } else if (fabsf((E - L->prev_energy) / E) < eps) {
        L->halt = 1;
        L->stop = LFRV_SR_STOP_RELATIVE;
    } else {
        L->prev_energy = E;
        if ((float)m[0] / npix < pct) {
            L->halt = 1;
            L->stop = LFRV_SR_STOP_MOVING;
        } else {
            L->cur ^= 1;  // prev <- U (super-resolution.cpp:255): the energy pass wrote it
        }
    }
}

}  // namespace

namespace {

DataTermArgs data_term_args(const lfrv_ctx *ctx)
{
    DataTermArgs da;
    da.alpha = ctx->p.dt_alpha;
    da.beta = ctx->p.dt_beta;
    da.sigma2 = ctx->p.sigma_sensor * ctx->p.sigma_sensor;
    da.grad_step = ctx->p.gradient_step;
    da.dsf2 = (float)(ctx->dsf * ctx->dsf);
    const float L = (float)(1.0 / (double)ctx->p.lambda);  // optimization.cu:1741
    da.prox_factor = (float)(-1.0 / ((double)ctx->p.lambda * (double)L));
    da.gw_type = ctx->p.gw_type;
    return da;
}

// The normalisation buffer that a step leaves the coverage in, as its data
// terms do (optimization.cu:1835-2116): without either term it stays as it is.
float *step_norm_mask(const lfrv_ctx *ctx)
{
    return ctx->p.dt_alpha > 0.0f || ctx->p.dt_beta > 0.0f ? ctx->norm_mask : nullptr;
}

// FISTA weights (optimization.cu:1744-1746): alpha_new is a cuflt (float)
// there, theta the float of the double quotient.  Returns theta of the step
// that starts at alpha; `an` receives alpha_new.
float fista_theta(double alpha, float &an)
{
    an = (float)(0.5 * (1.0 + std::sqrt(1.0 + 4.0 * std::pow(alpha, 2.0))));
    return (float)((alpha - 1.0) / (double)an);
}

// The primal-dual constants of the step fused with the data term
// (vtv_rof.cu:118-147), theta left for the caller.
PdArgs pd_args(const lfrv_ctx *ctx)
{
    PdArgs pa;
    pa.tau = pa.sigma = (float)(0.3 / std::sqrt(8.0));
    const float Lp = (float)(1.0 / (double)ctx->p.lambda);
    pa.lam = (float)(1.0 / (double)Lp);
    pa.theta = 0.0f;
    return pa;
}

// The assembled anchor-grid operator of the data term (dsf >= 2), rebuilt
// when the weights or the entries changed.
lfrv_status ensure_sr_ops(lfrv_ctx *ctx)
{
    if (ctx->sr_ops_epoch == ctx->epoch) return LFRV_OK;
    const TileGeom g = tile_geom(ctx);
    const TileEntries te = tile_entries(ctx);
    const int Wc = ctx->W + ctx->ks - 1, Hc = ctx->H + ctx->ks - 1;
    const size_t NA = (size_t)Wc * Hc;
    const int grad = ctx->p.dt_beta > 0.0f ? 1 : 0;
    const DataTermArgs da = data_term_args(ctx);
    TileGeom ga = g;
    ga.ntx = (Wc + g.tw - 1) / g.tw;
    ga.ntiles = ga.ntx * ((Hc + g.th - 1) / g.th);
    const int wh = g.th + 1, ncw = (g.tw + 1) * wh;
    const int cap = std::min(1024, kStagePer * ctx->pull_bs);
    const size_t lds = sizeof(int) * (2 * wh + 2) + sizeof(float) * std::max<size_t>(44 * (size_t)ncw, 9 * (size_t)cap);
    TimedRegion tr(ctx, 5);
#define AS(K) k_sr_assemble<K><<<ga.ntiles, ctx->pull_bs, lds, ctx->stream>>>(ga, te, cap, grad, ctx->p.gw_type != 0, dt_intensity_weight(da), dt_gradient_weight(da), NA, ctx->sr_ops)
    switch (ctx->ks) {
    case 3: AS(3); break;
    case 4: AS(4); break;
    case 5: AS(5); break;
    default: return fail(ctx, LFRV_E_ARG, "dsf out of range");
    }
#undef AS
    LFRV_LAUNCH(ctx, "data-term assembly");
    ctx->sr_ops_epoch = ctx->epoch;
    return LFRV_OK;
}

// Whether the step's planes outgrow one buffer descriptor (the five planes of a coupling set are the largest).
bool sr_wide(const lfrv_ctx *ctx)
{
    return strip_wide(5, ctx->W + ctx->ks - 1, ctx->H + ctx->ks - 1, ctx->narrow_bytes);
}

}  // namespace

int sr_lag(int ks, bool grad) { return ks - 1 + (grad ? 1 : 0); }

// Rows per strip for targets stepped in one launch.  A wave costs its rows and
// the 2 LAG before the first output, and 2 waves per SIMD, 2048 in all, run at
// once: the height (whole groups of rows) with the least rows per slot.  2048^2,
// dsf 4 (38 strips across): 42 rows, 1862 waves, 141 us per step; 36 rows, 2166
// waves, 173 us; 256^2, dsf 2: 3 rows 6.6 us, 12 rows 12.6 us.  Two waves are
// what the steps with the gradient term and the PCG iteration have registers
// for; the steps without it and the primal-dual passes would fit three to seven,
// and take the same rule without a measurement of theirs at other heights.
int strip_rows(int lag, const StripSize *sizes, int n)
{
    int best = kStripGroup;
    long best_cost = LONG_MAX;
    for (int rows = kStripGroup; rows <= 96; rows += kStripGroup) {
        long waves = 0;
        for (int i = 0; i < n; i++) waves += 4L * strips(lag, sizes[i], rows).nblocks;
        const long cost = (waves + 2047) / 2048 * (rows + 2 * lag);
        if (cost < best_cost) {
            best_cost = cost;
            best = rows;
        }
    }
    return best;
}

StripGeom strips(int lag, StripSize size, int rows)
{
    const int ow = 64 - 2 * lag;
    StripGeom sg;
    sg.nx = (size.W + ow - 1) / ow;
    sg.rows = rows;
    sg.nblocks = (sg.nx * ((size.H + rows - 1) / rows) + 3) / 4;
    return sg;
}

namespace {

// `iters` primal-dual iterations on F, up to four per pass, as even as they
// come; with `overrelax` the last also does the over-relaxation.
lfrv_status run_pd_steps(lfrv_ctx *ctx, int iters, const float *F, bool overrelax, float theta, const int *halt)
{
    const StripSize size{ctx->W, ctx->H};
    PdArgs pa = pd_args(ctx);
    pa.theta = theta;
    const bool wide = strip_wide(3, ctx->W, ctx->H, ctx->narrow_bytes);
    int left = iters;
    for (int passes = (iters + 3) / 4; passes > 0; passes--) {
        const int k = (left + passes - 1) / passes;
        left -= k;
        const StripGeom sg = strips(k, size, strip_rows(k, &size, 1));
        const PdBufs pb{ctx->Uq, ctx->PX,  ctx->PY,  F, ctx->has_reg_g ? ctx->reg_g : nullptr,
                        ctx->U2, ctx->P2X, ctx->P2Y, overrelax && left == 0 ? ctx->U : nullptr};
        const KernelEvents ev = kernel_events(ctx, 2);  // stamped by the dispatch itself
#define PD1(K, WI) hipExtLaunchKernelGGL(k_pd_steps<K, WI>, dim3(sg.nblocks), dim3(256), 0, ctx->stream, ev.a, ev.b, 0, ctx->W, ctx->H, sg, pa, pb, halt)
#define PD(K) case K: if (wide) PD1(K, true); else PD1(K, false); break
        switch (k) {
            PD(1);
            PD(2);
            PD(3);
            PD(4);
        }
#undef PD
#undef PD1
        record_kernel_events(ctx, 2, ev);
        std::swap(ctx->Uq, ctx->U2);
        std::swap(ctx->PX, ctx->P2X);
        std::swap(ctx->PY, ctx->P2Y);
    }
    LFRV_LAUNCH(ctx, "pd step");
    return LFRV_OK;
}

// One FISTA step on the stream; with `halt` every launch of the step is a
// no-op once a stopping rule has fired on the device.  A step that is not the
// last of a fixed run (last = false) leaves Uq and the norm mask to the run's
// last step where one pass does the whole step (dsf >= 2, one inner iteration).
lfrv_status enqueue_fista(lfrv_ctx *ctx, const int *halt, bool last = true)
{
    if (!ctx->prepared) return fail(ctx, LFRV_E_STATE, "FISTA step before lfrv_prepare");
    lfrv_status st = run_refresh_entry_weights(ctx, 1.0f);
    if (st != LFRV_OK) return st;
    const TileGeom g = tile_geom(ctx);
    const TileEntries te = tile_entries(ctx);
    const DataTermArgs da = data_term_args(ctx);
    // the over-relaxation is fused into the last primal-dual step
    float an;
    const float theta = fista_theta(ctx->fista_alpha, an);
    const int inner = ctx->p.inner_iterations;
    bool pd_done = false;  // the first primal-dual iteration ran with the data term
    const int HAL = ctx->ks - 1;
    if (ctx->ks == 2) {
        const size_t up = (size_t)(ctx->tile_w + 2 * HAL + 2) * (ctx->tile_h + 2 * HAL + 2);
        const size_t lpp = (size_t)(ctx->tile_w + 2 * HAL) * (ctx->tile_h + 2 * HAL);
        const size_t tiles = sizeof(float) * (3 * up + 3 * lpp);
        const int cap = pull_cap(ctx, 6, tiles, ctx->pull_budget, PullKind::Cell);
        const size_t lds = tiles + pull_lds(ctx, 6, cap, PullKind::Cell);
        const KernelEvents ev = kernel_events(ctx, 3);
        hipExtLaunchKernelGGL(k_sr_dataterm<2>, dim3(ctx->ntiles), dim3(ctx->pull_bs), lds, ctx->stream, ev.a, ev.b, 0,
                              g, te, cap, ctx->n, da, (const float *)ctx->U, (const float *)ctx->views,
                              (const float *)ctx->view_lap, (const float *)ctx->coverage, ctx->G, ctx->Uq,
                              ctx->norm_mask, halt);
        record_kernel_events(ctx, 3, ev);
        LFRV_LAUNCH(ctx, "data term");
    } else {
        // assembled operator on the anchor grid, rebuilt when the weights or
        // the entries changed; the step itself is a stencil
        const int Wc = ctx->W + ctx->ks - 1, Hc = ctx->H + ctx->ks - 1;
        const size_t NA = (size_t)Wc * Hc;
        st = ensure_sr_ops(ctx);
        if (st != LFRV_OK) return st;
        const StripSize size{ctx->W, ctx->H};
        const bool grad = da.beta > 0.0f;
        const StripGeom sg = strips(sr_lag(ctx->ks, grad), size, strip_rows(sr_lag(ctx->ks, grad), &size, 1));
        const KernelEvents ev = kernel_events(ctx, 3);  // stamped by the dispatch itself
#define STEP2(K, GR, PD, EX, WI) hipExtLaunchKernelGGL(k_sr_step_st<K, GR, PD, EX, WI>, dim3(sg.nblocks), dim3(256), 0, ctx->stream, ev.a, ev.b, 0, ctx->W, ctx->H, Wc, Hc, sg, da, pa, NA, sb, halt)
#define STEP1(K, GR, PD, EX) do { if (sr_wide(ctx)) STEP2(K, GR, PD, EX, true); else STEP2(K, GR, PD, EX, false); } while (0)
#define STEP(PD, EX)                                                              \
    do {                                                                          \
        if (ctx->ks == 3) { if (grad) STEP1(3, true, PD, EX); else STEP1(3, false, PD, EX); }      \
        else if (ctx->ks == 4) { if (grad) STEP1(4, true, PD, EX); else STEP1(4, false, PD, EX); } \
        else if (ctx->ks == 5) { if (grad) STEP1(5, true, PD, EX); else STEP1(5, false, PD, EX); } \
        else return fail(ctx, LFRV_E_ARG, "dsf out of range");                    \
    } while (0)
        if (inner > 0) {
            // the data term and the first primal-dual iteration in one pass: U is
            // read, the new primal goes to U2 (with one inner iteration the
            // over-relaxed one to Uq), the duals to P2X / P2Y
            PdArgs pa = pd_args(ctx);
            pa.theta = theta;
            const float *gw = ctx->has_reg_g ? ctx->reg_g : nullptr;
            const StepBufs sb{ctx->U,    ctx->sr_ops, ctx->coverage, ctx->PX, ctx->PY, gw, ctx->P2X, ctx->P2Y, ctx->U2,
                              (inner == 1 && last) ? ctx->Uq : nullptr, inner > 1 ? ctx->G : nullptr,
                              (inner > 1 || last) ? step_norm_mask(ctx) : nullptr};
            if (sb.uq_relax || sb.gout || sb.norm_mask) STEP(true, true);
            else STEP(true, false);
            record_kernel_events(ctx, 3, ev);
            LFRV_LAUNCH(ctx, "data term + primal-dual step");
            std::swap(ctx->PX, ctx->P2X);
            std::swap(ctx->PY, ctx->P2Y);
            if (inner == 1)
                std::swap(ctx->U, ctx->U2);  // U the new primal, Uq the over-relaxed one
            else
                std::swap(ctx->Uq, ctx->U2);  // the remaining iterations start from Uq
            pd_done = true;
        } else {
            const PdArgs pa{};
            const StepBufs sb{ctx->U,  ctx->sr_ops, ctx->coverage, nullptr, nullptr, nullptr,       nullptr, nullptr,
                              nullptr, ctx->Uq,     ctx->G,        step_norm_mask(ctx)};
            STEP(false, true);
            record_kernel_events(ctx, 3, ev);
            LFRV_LAUNCH(ctx, "data term");
        }
    }
#undef STEP
#undef STEP1
#undef STEP2
    if (pd_done) {
        if (inner > 1) {
            st = run_pd_steps(ctx, inner - 1, ctx->G, true, theta, halt);
            if (st != LFRV_OK) return st;
        }
    } else if (inner > 0) {
        st = run_pd_steps(ctx, inner, ctx->G, true, theta, halt);
        if (st != LFRV_OK) return st;
    } else {
        k_overrelax<<<blocks_for(3 * ctx->N), kBlock, 0, ctx->stream>>>(3 * ctx->N, theta, ctx->Uq, ctx->U, halt);
        LFRV_LAUNCH(ctx, "overrelaxation");
    }
    ctx->fista_alpha = an;
    return LFRV_OK;
}

// The energy's block partials (tv at partials[0], views at
// partials + kViewPartials); ugx / ugy in tmp3N.
lfrv_status enqueue_sr_energy(lfrv_ctx *ctx, const int *halt, float *prev2 = nullptr, float thr = 0.0f,
                              double *pmove = nullptr)
{
    const size_t N = ctx->N;
    float *ugx = ctx->tmp3N, *ugy = ctx->tmp3N + N;
    k_sr_energy_tv<<<rblocks(N), 256, 0, ctx->stream>>>(ctx->W, ctx->H, ctx->U, ctx->visibility, ugx, ugy,
                                                        ctx->partials, halt, prev2, ctx->sr_loop, thr, pmove);
    const size_t tot = (size_t)ctx->V * ctx->n;
    const float s2 = ctx->p.sigma_sensor * ctx->p.sigma_sensor;
    double *pv = ctx->partials + kViewPartials;
#define EV(K) k_sr_energy_views<K><<<rblocks(tot), 256, 0, ctx->stream>>>(ctx->V, ctx->W, ctx->H, ctx->w, ctx->h, ctx->tau_x, ctx->tau_y, ctx->omega, ctx->views, ctx->view_grad, ctx->U, ugx, ugy, s2, ctx->p.gw_type, pv, halt)
    switch (ctx->ks) {
    case 2: EV(2); break;
    case 3: EV(3); break;
    case 4: EV(4); break;
    case 5: EV(5); break;
    default: return fail(ctx, LFRV_E_ARG, "dsf out of range");
    }
#undef EV
    LFRV_LAUNCH(ctx, "sr energy");
    return LFRV_OK;
}

EnergyCoef energy_coef(const lfrv_ctx *ctx)
{
    return EnergyCoef{(double)ctx->p.lambda, (double)ctx->p.dt_alpha, (double)ctx->p.dt_beta};
}

}  // namespace

lfrv_status run_fista(lfrv_ctx *ctx, bool last)
{
    return enqueue_fista(ctx, nullptr, last);
}

bool sr_batchable(const lfrv_ctx *ctx)
{
    return ctx->p.mode == LFRV_MODE_COLOR_SR && ctx->ks >= 3 && ctx->ks <= 5 && ctx->p.inner_iterations == 1 &&
           !sr_wide(ctx);
}

lfrv_status sr_batch_begin(lfrv_ctx *ctx, int steps, SrBatchItem *it, float *theta_host)
{
    if (!ctx->prepared) return fail(ctx, LFRV_E_STATE, "FISTA step before lfrv_prepare");
    if (!sr_batchable(ctx)) return fail(ctx, LFRV_E_ARG, "batched FISTA steps need dsf >= 2 and one inner iteration");
    lfrv_status st = run_refresh_entry_weights(ctx, 1.0f);
    if (st == LFRV_OK) st = ensure_sr_ops(ctx);
    if (st != LFRV_OK) return st;
    const int Wc = ctx->W + ctx->ks - 1, Hc = ctx->H + ctx->ks - 1;
    it->W = ctx->W;
    it->H = ctx->H;
    it->Wc = Wc;
    it->Hc = Hc;
    it->steps = steps;
    it->da = data_term_args(ctx);
    it->pa = pd_args(ctx);
    it->theta = nullptr;
    it->ops = ctx->sr_ops;
    it->NA = (size_t)Wc * Hc;
    it->coverage = ctx->coverage;
    it->g = ctx->has_reg_g ? ctx->reg_g : nullptr;
    it->U[0] = ctx->U;
    it->U[1] = ctx->U2;
    it->PX[0] = ctx->PX;
    it->PX[1] = ctx->P2X;
    it->PY[0] = ctx->PY;
    it->PY[1] = ctx->P2Y;
    it->uq = ctx->Uq;
    it->norm_mask = step_norm_mask(ctx);
    double a = ctx->fista_alpha;
    for (int k = 0; k < steps; k++) {
        float an;
        theta_host[k] = fista_theta(a, an);
        a = an;
    }
    ctx->u_zero = false;
    return LFRV_OK;
}

void sr_batch_end(lfrv_ctx *ctx, int steps)
{
    double a = ctx->fista_alpha;
    for (int k = 0; k < steps; k++) {
        float an;
        (void)fista_theta(a, an);
        a = an;
    }
    ctx->fista_alpha = a;
    if (steps & 1) {  // the solve's own steps swap after every step
        std::swap(ctx->U, ctx->U2);
        std::swap(ctx->PX, ctx->P2X);
        std::swap(ctx->PY, ctx->P2Y);
    }
}

hipError_t launch_sr_batch_step(int ks, bool grad, const SrBatchItem *items, const int2 *work, int nblocks, int s,
                                hipStream_t stream)
{
#define SB(K, G) k_sr_step_st_batch<K, G><<<nblocks, 256, 0, stream>>>(items, work, s)
    switch (ks * 2 + (grad ? 1 : 0)) {
    case 6: SB(3, false); break;
    case 7: SB(3, true); break;
    case 8: SB(4, false); break;
    case 9: SB(4, true); break;
    case 10: SB(5, false); break;
    case 11: SB(5, true); break;
    default: return hipErrorInvalidValue;
    }
#undef SB
    return hipGetLastError();
}

lfrv_status run_sr_energy(lfrv_ctx *ctx, double *e, double *parts)
{
    lfrv_status st = enqueue_sr_energy(ctx, nullptr);
    if (st != LFRV_OK) return st;
    const size_t tot = (size_t)ctx->V * ctx->n;
    k_reduce_out<1><<<1, kFinalizeThreads, 0, ctx->stream>>>(ctx->partials, (int)rblocks(ctx->N), ctx->scal + 8);
    k_reduce_out<2><<<1, kFinalizeThreads, 0, ctx->stream>>>(ctx->partials + kViewPartials, (int)rblocks(tot),
                                                             ctx->scal + 9);
    LFRV_LAUNCH(ctx, "sr energy");
    LFRV_HIP(ctx, hipMemcpyAsync(ctx->scal_host + 8, ctx->scal + 8, 3 * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    LFRV_HIP(ctx, hipStreamSynchronize(ctx->stream));
    const double etv = ctx->scal_host[8], eint = ctx->scal_host[9], egrad = ctx->scal_host[10];
    if (parts) {
        parts[0] = etv;
        parts[1] = eint;
        parts[2] = egrad;
    }
    *e = (double)ctx->p.lambda * etv + (double)ctx->p.dt_alpha * eint + (double)ctx->p.dt_beta * egrad;
    return LFRV_OK;
}

lfrv_status run_count_moving(lfrv_ctx *ctx, const float *prev_dev, float max_diff, int64_t *moving)
{
    k_count_moving<<<rblocks(ctx->N), 256, 0, ctx->stream>>>(ctx->N, ctx->U, prev_dev, max_diff, ctx->partials,
                                                             nullptr);
    k_reduce_out<1><<<1, kFinalizeThreads, 0, ctx->stream>>>(ctx->partials, (int)rblocks(ctx->N), ctx->scal + 12);
    LFRV_LAUNCH(ctx, "count moving");
    LFRV_HIP(ctx, hipMemcpyAsync(ctx->scal_host + 12, ctx->scal + 12, sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    LFRV_HIP(ctx, hipStreamSynchronize(ctx->stream));
    *moving = (int64_t)std::llround(ctx->scal_host[12]);
    return LFRV_OK;
}

// The re-weighted least-squares loop of super-resolution.cpp:177-300.  Each
// FISTA step is followed on the stream by its energy pass (which also counts
// the moving pixels against the previous step's solution and writes U into
// the spare one of the two previous-step buffers) and one rule kernel (the
// energy rules, then the moving rule; when the step is kept it flips
// SrLoop::cur, so the spare buffer becomes the previous solution without a
// copy); once a rule fires, the launches enqueued after it return at once.  The host enqueues kSrPollSteps steps at
// a time and reads the loop state of the chunk before the one it has just
// enqueued, so the device runs ahead of the poll.
lfrv_status run_sr_solve(lfrv_ctx *ctx, int niter, int nmeta, lfrv_sr_stats *out)
{
    constexpr int kSrPollSteps = 8;
    const float EPSILON_TOL = 1e-4f, MAX_DIFF_THRESHOLD = 1e-3f, PERCENT_MOVING = 0.01f;
    const auto t0 = std::chrono::steady_clock::now();
    const size_t N = ctx->N, n3 = 3 * N;
    // the previous step's solution (two buffers, SrLoop::cur picks) and the previous pass's
    if (!ctx->sr_prev) LFRV_HIP(ctx, hipMalloc((void **)&ctx->sr_prev, 3 * n3 * sizeof(float)));
    float *prev2 = ctx->sr_prev, *prev_meta = ctx->sr_prev + 2 * n3;
    LFRV_HIP(ctx, hipMemcpyAsync(prev2, ctx->U, n3 * sizeof(float), hipMemcpyDeviceToDevice, ctx->stream));
    LFRV_HIP(ctx, hipMemsetAsync(&ctx->sr_loop->cur, 0, sizeof(int), ctx->stream));
    LFRV_HIP(ctx, hipMemcpyAsync(prev_meta, ctx->U, n3 * sizeof(float), hipMemcpyDeviceToDevice, ctx->stream));
    const int *halt = &ctx->sr_loop->halt;
    const EnergyCoef ec = energy_coef(ctx);
    const int Gtv = (int)rblocks(N), Gv = (int)rblocks((size_t)ctx->V * ctx->n), Gm = (int)rblocks(N);
    const float npix = (float)N;
    // the moving count's block partials, after the energy's (E_TV: 2048, views: 2 x 2048)
    double *pmove = ctx->partials + 3 * kViewPartials;
    if (3 * kViewPartials + (size_t)Gm > ctx->partials_cap) return fail(ctx, LFRV_E_STATE, "partials buffer too small");
    lfrv_sr_stats s{};
    float energy = 0.0f, previous_energy_reweight = 0.0f;
    int r;
    for (r = 0; r < nmeta; r++) {
        lfrv_status st = run_compute_weights(ctx);
        if (st == LFRV_OK) st = run_regularizer_weight(ctx);
        if (st == LFRV_OK) st = enqueue_sr_energy(ctx, nullptr);
        if (st != LFRV_OK) return st;
        k_sr_loop_begin<<<1, kFinalizeThreads, 0, ctx->stream>>>(ctx->sr_loop, ctx->partials, Gtv,
                                                                 ctx->partials + kViewPartials, Gv, ec);
        LFRV_LAUNCH(ctx, "sr loop begin");
        // alpha and the ping-pong buffers after each enqueued step, to undo the
        // host-side effects of the steps the device skipped
        struct StepState {
            double alpha;
            float *U, *Uq, *U2, *PX, *PY, *P2X, *P2Y;
        };
        auto snap = [ctx]() {
            return StepState{ctx->fista_alpha, ctx->U, ctx->Uq, ctx->U2, ctx->PX, ctx->PY, ctx->P2X, ctx->P2Y};
        };
        std::vector<StepState> states{snap()};
        int enq = 0, polls = 0;
        bool halted = false;
        while (enq < niter && !halted) {
            const int chunk = std::min(kSrPollSteps, niter - enq);
            for (int j = 0; j < chunk; j++) {
                st = enqueue_fista(ctx, halt);
                // the energy pass also takes the moving count (rblocks(N) == Gm block partials)
                if (st == LFRV_OK) st = enqueue_sr_energy(ctx, halt, prev2, MAX_DIFF_THRESHOLD, pmove);
                if (st != LFRV_OK) return st;
                states.push_back(snap());
                k_sr_loop_step<<<1, kFinalizeThreads, 0, ctx->stream>>>(
                    ctx->sr_loop, ctx->partials, Gtv, ctx->partials + kViewPartials, Gv, ec, EPSILON_TOL, pmove, Gm,
                    npix, PERCENT_MOVING);
                LFRV_LAUNCH(ctx, "sr loop step");
            }
            enq += chunk;
            const int slot = polls & 1;
            LFRV_HIP(ctx, hipMemcpyAsync(ctx->sr_loop_host + slot, ctx->sr_loop, sizeof(SrLoop), hipMemcpyDeviceToHost,
                                         ctx->stream));
            LFRV_HIP(ctx, hipEventRecord(ctx->sr_ev[slot], ctx->stream));
            if (++polls >= 2) {
                LFRV_HIP(ctx, hipEventSynchronize(ctx->sr_ev[slot ^ 1]));
                halted = ctx->sr_loop_host[slot ^ 1].halt != 0;
            }
        }
        LFRV_HIP(ctx, hipMemcpyAsync(ctx->sr_loop_host + 2, ctx->sr_loop, sizeof(SrLoop), hipMemcpyDeviceToHost,
                                     ctx->stream));
        LFRV_HIP(ctx, hipStreamSynchronize(ctx->stream));
        const SrLoop L = ctx->sr_loop_host[2];
        if (L.steps < 0 || L.steps > enq) return fail(ctx, LFRV_E_STATE, "FISTA loop state out of range");
        const StepState &ss = states[L.steps];
        ctx->fista_alpha = ss.alpha;
        ctx->U = ss.U;
        ctx->Uq = ss.Uq;
        ctx->U2 = ss.U2;
        ctx->PX = ss.PX;
        ctx->PY = ss.PY;
        ctx->P2X = ss.P2X;
        ctx->P2Y = ss.P2Y;
        energy = L.energy;
        s.fista_steps += L.steps;
        s.last_stop = L.stop;
        // the re-weighting rules (super-resolution.cpp:272-297)
        if (energy < EPSILON_TOL) {
            if (previous_energy_reweight < EPSILON_TOL) {
                s.converged = 1;
                break;
            }
            previous_energy_reweight = energy;
            continue;
        }
        int64_t moving = 0;
        st = run_count_moving(ctx, prev_meta, MAX_DIFF_THRESHOLD, &moving);
        if (st != LFRV_OK) return st;
        if ((float)moving / npix < PERCENT_MOVING) {
            s.converged = 1;
            break;
        }
        LFRV_HIP(ctx, hipMemcpyAsync(prev_meta, ctx->U, n3 * sizeof(float), hipMemcpyDeviceToDevice, ctx->stream));
    }
    LFRV_HIP(ctx, hipStreamSynchronize(ctx->stream));
    s.meta_iterations = r < nmeta ? r + 1 : nmeta;
    s.energy = energy;
    s.ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    if (out) *out = s;
    return LFRV_OK;
}

}  // namespace lfrv
