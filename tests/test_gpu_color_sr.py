"""GPU parity of the IBR_color path (TV primal-dual with warped data terms)
against the FP64 oracle, step by step through sr_synthesize_view."""
import numpy as np
import pytest

import lfrv
import oracle
from lfrv import pipelines
from lfrv.batch import Batch
from conftest import rel_err

pytestmark = pytest.mark.gpu


def _scene(dsf=2, kind=1, w=48):
    d = lfrv.synth_desc(1, 5)
    d.w = d.h = w
    d.dsf = dsf
    d.render_scale = dsf
    d.focal = float(w)
    d.baseline = 0.7 * 4.0 / (w * dsf)
    if kind == 2:
        d.kind = 2
        d.baseline = 2.0 * 4.0 / (w * dsf)
    return lfrv.synth(d)


@pytest.mark.parametrize("dsf,beta,gw,inner", [(2, 0.0, 0, 10), (2, 0.5, 1, 10), (3, 0.3, 0, 10), (1, 0.5, 1, 10),
                                              (2, 0.5, 0, 1), (4, 0.3, 0, 1), (4, 0.0, 1, 2), (3, 0.3, 0, 0)])
def test_sr_steps_match_oracle(dsf, beta, gw, inner):
    """inner = 1: for dsf >= 2 the data term and the only primal-dual iteration
    (with the over-relaxation) run as one kernel; inner > 1 fuses the first
    iteration; inner = 0 leaves the data term alone."""
    _steps_match_oracle(_scene(dsf=dsf, kind=2 if dsf == 1 else 1), beta, gw, inner)


def _c3_scene(w=96, seed=7):
    """The 5x5-view generator of the 512^2 -> 2048^2 workload (8 tilted planes,
    disparity -2..+2 px per grid step through the principal-point shift,
    views box-averaged x4) at w x w views: the focal length scales with w and
    f * baseline stays 10, so the disparities in view pixels are the same."""
    d = lfrv.synth_desc(3, seed)
    d.w = d.h = w
    d.focal = float(w)
    d.baseline = 10.0 / w
    return lfrv.synth(d)


@pytest.mark.parametrize("beta,inner", [(1.0, 1), (0.3, 2)])
def test_sr_steps_match_oracle_25_views_dsf4(beta, inner):
    """25 views and dsf 4 (the 512^2 -> 2048^2 configuration's generator, at
    96^2 -> 384^2): the pull kernels' per-window caps and the assembled
    anchor-grid operator at 25 views."""
    s = _c3_scene()
    assert s["V"] == 25 and s["dsf"] == 4
    _steps_match_oracle(s, beta, 0, inner, metas=2, steps=3)


def test_sr_full_size_128_to_256_matches_oracle():
    """The 3x3 128^2 -> 256^2 configuration at its full size: 20 FISTA steps of
    the benchmark's parameters (one primal-dual iteration, lambda 0.05,
    lambda_max_factor 100) against the oracle, U within 5e-4 and the energy
    within 1e-4 relative at the end."""
    s = lfrv.synth(1, seed=2024)
    _steps_match_oracle(s, 0.0, 0, 1, metas=1, steps=20, u_tol=5e-4, dual_tol=5e-4)


def _steps_match_oracle(s, beta, gw, inner, metas=2, steps=3, u_tol=2e-4, dual_tol=2e-4):
    dsf = s["dsf"]
    print(f"IBR_color V={s['V']} {s['w']}x{s['h']} dsf={dsf} beta={beta} gw={gw} inner={inner}", flush=True)
    V, h, w, H, W = s["V"], s["h"], s["w"], s["H"], s["W"]
    sig, lam, lmf = 1.0 / 255.0, 0.05, 100.0
    prm = pipelines.color_sr_params(s, lambda_=lam, lambda_max_factor=lmf, inner_iterations=inner, dt_beta=beta,
                                    gw_type=gw, gradient_step=1.0)
    with lfrv.Context(prm) as ctx:
        pipelines.load_scene(ctx, s)
        ctx.warps_from_depth()
        ctx.prepare()
        tx = ctx.get_buffer("TAU_X").reshape(V, h, w)
        ty = ctx.get_buffer("TAU_Y").reshape(V, h, w)
        dpx = ctx.get_buffer("DPART_X").reshape(V, h, w)
        dpy = ctx.get_buffer("DPART_Y").reshape(V, h, w)
        # oracle state mirrors coco_vtv_workspace
        st = oracle.SrState(W, H, np.zeros((3, H, W)))
        vis0 = np.zeros((H, W), np.uint8)
        ctx.compute_weights()
        om, gx, gy = oracle.sr_weights(W, H, dsf, tx, ty, dpx, dpy, st.U, vis0, st.PX[0], st.PY[0], sig, 1.0)
        st.PX[0], st.PY[0] = gx, gy
        assert rel_err(ctx.get_buffer("OMEGA").reshape(V, h, w), om) < 1e-6
        ctx.setup_visibility()
        cov = oracle.coverage(W, H, dsf, tx, ty)
        vis = (cov >= 1.0).astype(np.uint8)
        st.norm_mask += cov
        gvis = ctx.get_buffer("VISIBILITY").reshape(H, W)
        near = np.abs(cov - 1.0) < 1e-5
        assert np.array_equal(gvis[~near].astype(np.uint8), vis[~near])
        vis = np.where(near, gvis.astype(np.uint8), vis)
        ctx.compute_initial_image()
        U0, nm = oracle.initial_image(W, H, dsf, tx, ty, s["views"], om)
        st.norm_mask = nm
        U0 = oracle.push_pull(U0, vis)
        st.U = U0.copy()
        st.Uq = U0.copy()
        assert np.max(np.abs(ctx.get_solution() - U0)) < 1e-5
        for meta in range(metas):
            ctx.compute_weights()
            om, gx, gy = oracle.sr_weights(W, H, dsf, tx, ty, dpx, dpy, st.U, vis, st.PX[0], st.PY[0], sig, 1.0)
            st.PX[0], st.PY[0] = gx, gy
            assert rel_err(ctx.get_buffer("OMEGA").reshape(V, h, w), om) < 1e-5
            ctx.sr_init_regularizer_weight()
            g, st.norm_mask = oracle.regularizer_weight(W, H, dsf, tx, ty, om, sig, lmf * lam, lam, st.norm_mask)
            assert np.max(np.abs(ctx.get_buffer("REG_G").reshape(H, W) - g)) < 1e-5 * lmf * lam
            assert rel_err(ctx.get_buffer("NORM_MASK").reshape(H, W), st.norm_mask) < 1e-5
            e, parts = ctx.sr_primal_energy()
            oe, oparts = oracle.sr_energy(W, H, dsf, tx, ty, s["views"], om, sig, lam, 1.0, beta, gw, vis, st.U)
            assert abs(e - oe) / oe < 1e-4
            for k in range(steps):
                ctx.sr_iteration_fista()
                oracle.fista_step(W, H, dsf, tx, ty, s["views"], om, sig, 1.0, beta, 1.0, gw, lam, inner, g, st)
            U = ctx.get_solution()
            assert np.max(np.abs(U - st.U)) < u_tol, np.max(np.abs(U - st.U))
            assert np.max(np.abs(ctx.get_buffer("UQ").reshape(3, H, W) - st.Uq)) < 2 * u_tol
            assert np.max(np.abs(ctx.get_buffer("PX").reshape(3, H, W) - st.PX)) < dual_tol
            assert np.max(np.abs(ctx.get_buffer("PY").reshape(3, H, W) - st.PY)) < dual_tol
            assert rel_err(ctx.get_buffer("NORM_MASK").reshape(H, W), st.norm_mask) < 1e-5
        # the energy of the final iterate
        e, _ = ctx.sr_primal_energy()
        oe, _ = oracle.sr_energy(W, H, dsf, tx, ty, s["views"], om, sig, lam, 1.0, beta, gw, vis, st.U)
        assert abs(e - oe) / oe < 1e-4, (e, oe)


def test_sr_count_moving():
    s = _scene()
    prm = pipelines.color_sr_params(s)
    with lfrv.Context(prm) as ctx:
        pipelines.load_scene(ctx, s)
        pipelines.color_sr_setup(ctx)
        U = ctx.get_solution()
        prev = U.copy()
        rng = np.random.default_rng(0)
        idx = rng.choice(s["H"] * s["W"], 100, replace=False)
        prev.reshape(3, -1)[1, idx] += 2e-3
        prev.reshape(3, -1)[0, idx[:10]] += 5e-4
        assert ctx.sr_count_moving(prev, 1e-3) == 100


@pytest.mark.parametrize("dsf,inner,beta", [(2, 1, 0.3), (3, 1, 0.0), (1, 3, 0.3)])
def test_sr_iterate_equals_single_steps(dsf, inner, beta):
    """lfrv_sr_iterate(k) gives the solution, duals, over-relaxed solution and
    normalisation buffer of k lfrv_sr_iteration_fista calls, bit for bit (a
    fixed run writes the last two only in its last step)."""
    s = _scene(dsf=dsf, kind=2 if dsf == 1 else 1)
    prm = pipelines.color_sr_params(s, inner_iterations=inner, dt_beta=beta, gradient_step=1.0)
    out = []
    for batched in (False, True):
        with lfrv.Context(prm) as ctx:
            pipelines.load_scene(ctx, s)
            ctx.clear_solution()
            pipelines.color_sr_setup(ctx)
            ctx.sr_init_regularizer_weight()
            if batched:
                ctx.sr_iterate(7)
            else:
                for _ in range(7):
                    ctx.sr_iteration_fista()
            out.append((ctx.get_solution(), ctx.get_buffer("PX"), ctx.get_buffer("PY"), ctx.get_buffer("UQ"),
                        ctx.get_buffer("NORM_MASK")))
    for a, b in zip(*out):
        assert np.array_equal(a, b)
    assert np.abs(out[0][3].ravel() - out[0][0].ravel()).max() > 0  # the over-relaxed solution is not the solution


@pytest.mark.parametrize("w,h,dsf,beta", [(29, 7, 2, 0.3),   # one strip to its last column, rows short of a group
                                          (30, 8, 2, 0.0),
                                          (31, 3, 2, 0.0),   # a second strip of two columns
                                          (19, 16, 3, 0.3),  # a second strip of one column
                                          (14, 5, 4, 0.3), (70, 4, 4, 0.0)])
def test_sr_steps_at_strip_edges(w, h, dsf, beta):
    """The marching step where its 64-column strips and 3-row groups end, against the oracle."""
    d = lfrv.synth_desc(1, 3)
    d.grid, d.w, d.h, d.dsf, d.render_scale = 3, w, h, dsf, dsf
    d.focal, d.baseline = float(w), 0.7 * 4.0 / (w * dsf)
    _steps_match_oracle(lfrv.synth(d), beta, 0, 1, metas=1, steps=3)


@pytest.mark.parametrize("w,h,dsf,inner", [(62, 5, 1, 1),    # one strip of a pass of one iteration, exactly
                                           (57, 7, 1, 4),    # four iterations per pass: a second strip of one column
                                           (59, 9, 1, 5),    # three and two
                                           (30, 4, 2, 4), (33, 3, 2, 9)])  # three after the first; four and four
def test_pd_passes_at_strip_edges(w, h, dsf, inner):
    """Several primal-dual iterations per pass where the strips end, against the oracle."""
    d = lfrv.synth_desc(1, 3)
    d.grid, d.w, d.h, d.dsf, d.render_scale = 3, w, h, dsf, dsf
    d.focal, d.baseline = float(w), 0.7 * 4.0 / (w * dsf)
    _steps_match_oracle(lfrv.synth(d), 0.3, 0, inner, metas=1, steps=2)


@pytest.mark.parametrize("dsf,inner", [(1, 1), (2, 1), (2, 0), (2, 3), (4, 1)])
def test_step_without_data_terms_keeps_the_norm_mask(dsf, inner):
    """dt_alpha = dt_beta = 0: no data term runs, so the normalisation buffer stays, in single steps, in a fixed run
    and in a batch (whose set-up leaves the mask that the same calls leave here)."""
    s = _scene(dsf=dsf, kind=2 if dsf == 1 else 1)
    print(f"norm mask without data terms dsf={dsf} inner={inner}", flush=True)
    prm = pipelines.color_sr_params(s, inner_iterations=inner, dt_alpha=0.0, dt_beta=0.0)
    with lfrv.Context(prm) as ctx, lfrv.Context(prm) as other:
        for c in (ctx, other):
            pipelines.load_scene(c, s)
        pipelines.color_sr_setup(ctx)
        ctx.sr_init_regularizer_weight()
        before = ctx.get_buffer("NORM_MASK")
        assert rel_err(before, ctx.get_buffer("COVERAGE")) > 0.1
        ctx.sr_iteration_fista()
        ctx.sr_iterate(3)
        assert np.array_equal(ctx.get_buffer("NORM_MASK"), before)
        b = Batch()
        b.add_pd(other, 4)
        b.run()
        b.close()
        assert np.array_equal(other.get_buffer("NORM_MASK"), before)
        assert np.array_equal(other.get_solution(), ctx.get_solution())


def _step_from_buffers(ctx, s, U0, alpha, beta, inner):
    """One step of the oracle from the context's own warps, weights and duals and the solution U0."""
    V, w, h, W, H = s["V"], s["w"], s["h"], s["W"], s["H"]
    tx, ty, om = [ctx.get_buffer(k).reshape(V, h, w) for k in ("TAU_X", "TAU_Y", "OMEGA")]
    st = oracle.SrState(W, H, U0)
    st.PX[:], st.PY[:] = [ctx.get_buffer(k).reshape(3, H, W) for k in ("PX", "PY")]
    with np.errstate(all="ignore"):
        oracle.fista_step(W, H, s["dsf"], tx, ty, s["views"], om, 1 / 255.0, alpha, beta, 1.0, 0, 0.05, inner,
                          ctx.get_buffer("REG_G").reshape(H, W), st)
    return st


@pytest.mark.parametrize("value", [np.inf, -np.inf])
@pytest.mark.parametrize("dsf,inner", [(2, 1), (2, 3), (3, 0), (4, 1)])
def test_step_with_an_infinite_view_pixel(dsf, inner, value):
    """An infinite view pixel makes its target pixels' gradient infinite: the clamp takes it to +-1, not to NaN."""
    s = _scene(dsf=dsf)
    s["views"] = s["views"].copy()
    s["views"][0, :, 20, 17] = value  # (a corner camera: its footprints have no weight of 0, whose product is NaN)
    print(f"infinite view pixel {value} dsf={dsf} inner={inner}", flush=True)
    with lfrv.Context(pipelines.color_sr_params(s, inner_iterations=inner)) as ctx:
        pipelines.load_scene(ctx, s)
        pipelines.color_sr_setup(ctx)
        U0 = np.random.default_rng(dsf).uniform(0.2, 0.8, (3, s["H"], s["W"])).astype(np.float32)
        ctx.set_solution(U0)
        ctx.sr_init_regularizer_weight()
        st = _step_from_buffers(ctx, s, U0, 1.0, 0.0, inner)
        ctx.sr_iteration_fista()
        key = "G" if inner == 0 else "U"
        got, want = ctx.get_buffer(key).reshape(U0.shape), st.G if inner == 0 else st.U
        assert np.all(np.isfinite(want)) and np.max(np.abs(got - want)) < 1e-4


@pytest.mark.parametrize("dsf,inner", [(1, 1), (1, 4), (2, 1), (2, 2), (4, 1)])
@pytest.mark.parametrize("at", ["right", "bottom", "corner", "left", "top"])
def test_duals_beside_an_infinite_pixel(dsf, inner, at):
    """Forward differences end at the image's edge: an infinite pixel there is not multiplied by a weight of 0, and
    what is not a number is so in the same places as in the oracle."""
    s = _scene(dsf=dsf, kind=2 if dsf == 1 else 1)
    H, W = s["H"], s["W"]
    y, x = {"right": (9, W - 1), "bottom": (H - 1, 9), "corner": (H - 1, W - 1), "left": (9, 0), "top": (0, 9)}[at]
    print(f"infinite solution pixel {y},{x} dsf={dsf} inner={inner}", flush=True)
    with lfrv.Context(pipelines.color_sr_params(s, inner_iterations=inner, dt_alpha=0.0)) as ctx:
        pipelines.load_scene(ctx, s)
        pipelines.color_sr_setup(ctx)
        U0 = np.random.default_rng(dsf).uniform(0.2, 0.8, (3, H, W)).astype(np.float32)
        U0[1, y, x] = np.inf
        ctx.set_solution(U0)
        ctx.sr_init_regularizer_weight()
        st = _step_from_buffers(ctx, s, U0, 0.0, 0.0, inner)
        ctx.sr_iteration_fista()
        for key, want in (("U", st.U), ("PX", st.PX), ("PY", st.PY)):
            got = ctx.get_buffer(key).reshape(want.shape)
            assert np.array_equal(np.isfinite(got), np.isfinite(want)), key
            ok = np.isfinite(want)
            assert np.max(np.abs(got[ok] - want[ok])) < 1e-4, key


def _fma(a, b, c):
    """a b + c of FP32 values, rounded once."""
    return np.float32(np.longdouble(a) * np.longdouble(b) + np.longdouble(c))


@pytest.mark.parametrize("dsf,inner", [(1, 1), (1, 4), (2, 1), (2, 3), (4, 1)])
def test_primal_is_formed_from_the_stored_duals(dsf, inner):
    """Where the projection scales the duals, the divergence is that of the rounded duals, as they are two passes in
    the reference: the last iteration's primal restated operation by operation, bit for bit."""
    s = _scene(dsf=dsf, kind=2 if dsf == 1 else 1)
    H, W = s["H"], s["W"]
    print(f"primal from the stored duals dsf={dsf} inner={inner}", flush=True)
    rng = np.random.default_rng(dsf)
    U0 = rng.uniform(0.2, 0.8, (3, H, W)).astype(np.float32)
    P0 = rng.uniform(-0.5, 0.5, (2, 3, H, W)).astype(np.float32)

    def step(iterations):  # (without data terms F is the solution itself)
        with lfrv.Context(pipelines.color_sr_params(s, inner_iterations=iterations, dt_alpha=0.0)) as ctx:
            pipelines.load_scene(ctx, s)
            pipelines.color_sr_setup(ctx)
            ctx.sr_init_regularizer_weight()
            ctx.set_buffer("REG_G", np.full((H, W), 0.3, np.float32))
            ctx.set_buffer("PX", P0[0])
            ctx.set_buffer("PY", P0[1])
            ctx.set_solution(U0)
            ctx.sr_iteration_fista()
            return [ctx.get_buffer(b).reshape(3, H, W) for b in ("U", "PX", "PY")]

    U, px, py = step(inner)
    before = step(inner - 1)[0] if inner > 1 else U0
    length = np.sqrt((px.astype(np.float64) ** 2 + py.astype(np.float64) ** 2).sum(0))
    assert length.max() < 0.3 * (1 + 1e-6) and (length > 0.299).mean() > 0.1
    left, up = np.zeros_like(px), np.zeros_like(py)
    left[..., 1:], up[..., 1:, :] = px[..., :-1], py[..., :-1, :]
    tau, lam = np.float32(0.3 / np.sqrt(8.0)), np.float32(0.05)
    lam = np.float32(1 / np.float64(np.float32(1 / np.float64(lam))))
    un = _fma(tau, px + py - left - up, before)
    assert np.array_equal(U, _fma(tau, U0, lam * un) / (tau + lam))


@pytest.mark.parametrize("dsf,beta", [(2, 0.0), (3, 0.3), (4, 0.3)])
def test_step_with_coverages_that_need_a_division(dsf, beta):
    """A few coverages beyond the range of the shared reciprocal: their waves divide, with the same bits for the
    ordinary pixels, and theirs are what division gives."""
    s = _scene(dsf=dsf)
    H, W = s["H"], s["W"]
    print(f"extreme coverages dsf={dsf} beta={beta}", flush=True)
    at = {(3, 5): 1e-40, (20, 30): -0.5, (21, 31): 3e38, (40, 7): np.inf, (H - 1, W - 1): 2e-39, (H - 9, 0): 0.0}
    U0 = np.random.default_rng(dsf).uniform(0.2, 0.8, (3, H, W)).astype(np.float32)
    F = []
    for special in (False, True):
        with lfrv.Context(pipelines.color_sr_params(s, inner_iterations=0, dt_beta=beta, gradient_step=1.0)) as ctx:
            pipelines.load_scene(ctx, s)
            pipelines.color_sr_setup(ctx)
            cov = ctx.get_buffer("COVERAGE").reshape(H, W).copy()
            for p, v in at.items():
                cov[p] = v if special else 1.0
            ctx.set_buffer("COVERAGE", cov)
            ctx.set_solution(U0)
            ctx.sr_iteration_fista()
            F.append(ctx.get_buffer("G").reshape(3, H, W))
    rest = np.ones((H, W), bool)
    for (y, x), v in at.items():
        rest[y, x] = False
        step = F[0][:, y, x] - U0[:, y, x]  # minus the clamped gradient at a coverage of 1
        assert np.all(step != 0)
        want = {1e-40: np.where(step > 0, 1, 0), 2e-39: np.where(step > 0, 1, 0), 3e38: U0[:, y, x], np.inf: U0[:, y, x],
                0.0: F[0][:, y, x]}.get(v)
        if want is not None:
            assert np.array_equal(F[1][:, y, x], want.astype(np.float32)), v
        else:
            assert np.all(np.sign(F[1][:, y, x] - U0[:, y, x]) == -np.sign(step))
    assert np.array_equal(F[0][:, rest], F[1][:, rest])


@pytest.mark.parametrize("dsf,beta", [(2, 0.0), (4, 0.3)])
def test_step_whose_quotients_overflow(dsf, beta):
    """Views of 1e33: over a coverage of 1e-3 the gradient overflows to an infinity, which the clamp takes to the same
    +-1 as the finite one over 1, not to NaN."""
    s = _scene(dsf=dsf)
    H, W = s["H"], s["W"]
    s["views"] = ((s["views"] - 0.5) * np.float32(1e33)).astype(np.float32)
    print(f"overflowing quotients dsf={dsf} beta={beta}", flush=True)
    U0 = np.random.default_rng(dsf).uniform(0.2, 0.8, (3, H, W)).astype(np.float32)
    F = []
    for cov in (1.0, 1e-3):
        with lfrv.Context(pipelines.color_sr_params(s, inner_iterations=0, dt_beta=beta, gradient_step=1.0)) as ctx:
            pipelines.load_scene(ctx, s)
            pipelines.color_sr_setup(ctx)
            ctx.set_buffer("COVERAGE", np.full((H, W), cov, np.float32))
            ctx.set_solution(U0)
            ctx.sr_iteration_fista()
            F.append(ctx.get_buffer("G").reshape(3, H, W))
    assert np.isin(F[0], (0, 1)).mean() > 0.9 and 0.2 < (F[0] == 1).mean() < 0.8
    assert np.array_equal(F[0][np.isin(F[0], (0, 1))], F[1][np.isin(F[0], (0, 1))])
