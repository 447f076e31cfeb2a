"""Ragged and degenerate inputs on the GPU against the FP64 oracle: sizes that
are no multiple of any tile, a single view, tiny images, and a view whose depth
is invalid everywhere (import.cpp:292-296 sends all its pixels out of the
target), for both models."""
import ctypes

import numpy as np
import pytest

import lfrv
import oracle
from lfrv import pipelines
from conftest import rel_err

pytestmark = pytest.mark.gpu


def _planes(w, h, dsf, grid, seed, dead_view=None):
    d = lfrv.synth_desc(2, seed)
    d.w, d.h, d.dsf, d.grid = w, h, dsf, grid
    d.focal = float(w)          # disparities of w/200 .. w/40 px per grid step
    d.render_scale = dsf
    s = lfrv.synth(d)
    if dead_view is not None:
        s["depths"][dead_view][:] = 0.0
    return s


GRAD_CASES = [
    (37, 23, 1, 3, None),   # 2x2 footprints: the assembled stencil with partial 64x8 tiles
    (29, 17, 2, 2, None),   # four views, entry-walk operator
    (21, 19, 3, 1, None),   # one view
    (6, 5, 1, 2, None),     # smaller than one tile
    (40, 24, 1, 3, 4),      # the centre view's depth invalid everywhere
]


@pytest.mark.parametrize("w,h,dsf,grid,dead", GRAD_CASES)
def test_gradient_ibr_ragged_inputs(w, h, dsf, grid, dead):
    s = _planes(w, h, dsf, grid, seed=11, dead_view=dead)
    print(f"IBR_gradient w={w} h={h} dsf={dsf} views={s['V']} dead={dead}", flush=True)
    with lfrv.Context(pipelines.gradient_ibr_params(s)) as ctx:
        pipelines.load_scene(ctx, s)
        st = ctx.ibr_gradient(1e-5, 2000)
        U = ctx.get_solution()
        tx = ctx.get_buffer("TAU_X").reshape(s["V"], h, w)
    r = oracle.gibr_pipeline(s["views"], s["depths"], s["P_views"], s["P_target"], dsf, 1 / 255.0, 1.0,
                             1.0, 0.5, 1e-5, 2000)
    if dead is not None:
        assert np.all(tx[dead] < 0) and np.all(r["tx"][dead] < 0)
    assert all(st["converged"])
    assert np.all(np.isfinite(U))
    assert rel_err(U, r["U"]) < 1e-3
    assert abs(oracle.psnr(U, s["target"]) - oracle.psnr(r["U"], s["target"])) < 0.01


COLOR_CASES = [
    (29, 17, 2, 1),   # the data-term / primal-dual pass with partial 32x16 tiles
    (13, 11, 4, 1),   # dsf 4 on a target of 52 x 44
    (7, 5, 3, 2),     # smaller than one tile, two inner iterations
    (23, 19, 1, 3),   # dsf 1: entry pull + separate primal-dual steps
]


@pytest.mark.parametrize("w,h,dsf,inner", COLOR_CASES)
def test_color_sr_ragged_inputs(w, h, dsf, inner):
    s = _planes(w, h, dsf, 3, seed=7)
    V, H, W = s["V"], s["H"], s["W"]
    print(f"IBR_color w={w} h={h} dsf={dsf} inner={inner}", flush=True)
    sig, lam, lmf, beta = 1.0 / 255.0, 0.05, 100.0, 0.5
    prm = pipelines.color_sr_params(s, lambda_=lam, lambda_max_factor=lmf, inner_iterations=inner, dt_beta=beta,
                                    gradient_step=1.0)
    with lfrv.Context(prm) as ctx:
        pipelines.load_scene(ctx, s)
        ctx.clear_solution()
        pipelines.color_sr_setup(ctx)
        tx = ctx.get_buffer("TAU_X").reshape(V, h, w)
        ty = ctx.get_buffer("TAU_Y").reshape(V, h, w)
        dpx = ctx.get_buffer("DPART_X").reshape(V, h, w)
        dpy = ctx.get_buffer("DPART_Y").reshape(V, h, w)
        gvis = ctx.get_buffer("VISIBILITY").reshape(H, W).astype(np.uint8)
        # the oracle's state from the GPU's warps, as sr_synthesize_view sets it up
        st = oracle.SrState(W, H, np.zeros((3, H, W)))
        om, gx, gy = oracle.sr_weights(W, H, dsf, tx, ty, dpx, dpy, st.U, np.zeros((H, W), np.uint8), st.PX[0],
                                       st.PY[0], sig, 1.0)
        st.PX[0], st.PY[0] = gx, gy
        cov = oracle.coverage(W, H, dsf, tx, ty)
        vis = (cov >= 1.0).astype(np.uint8)
        near = np.abs(cov - 1.0) < 1e-5
        assert np.array_equal(gvis[~near], vis[~near])
        vis = np.where(near, gvis, vis)
        st.norm_mask += cov
        U0, st.norm_mask = oracle.initial_image(W, H, dsf, tx, ty, s["views"], om)
        st.U = oracle.push_pull(U0, vis)
        st.Uq = st.U.copy()
        assert np.max(np.abs(ctx.get_solution() - st.U)) < 1e-5
        ctx.sr_init_regularizer_weight()
        g, st.norm_mask = oracle.regularizer_weight(W, H, dsf, tx, ty, om, sig, lmf * lam, lam, st.norm_mask)
        ctx.sr_iterate(4)
        for _ in range(4):
            oracle.fista_step(W, H, dsf, tx, ty, s["views"], om, sig, 1.0, beta, 1.0, 0, lam, inner, g, st)
        U = ctx.get_solution()
        assert np.all(np.isfinite(U))
        assert np.max(np.abs(U - st.U)) < 2e-4
        assert np.max(np.abs(ctx.get_buffer("PX").reshape(3, H, W) - st.PX)) < 2e-4
        e, _ = ctx.sr_primal_energy()
        oe, _ = oracle.sr_energy(W, H, dsf, tx, ty, s["views"], om, sig, lam, 1.0, beta, 0, vis, st.U)
        assert abs(e - oe) <= 1e-4 * max(oe, 1e-12)


@pytest.mark.parametrize("w,h,dead", [(17, 33, (0, 17, 0, 16)),    # holes to three image edges, one tile past the second
                                      (48, 40, (8, 40, 8, 24)),    # whole tiles of holes
                                      (65, 20, (60, 65, 3, 20))])  # one column in the last tile
def test_hole_sweeps_at_tile_edges(w, h, dead):
    """A solve from an image whose holes end at the edges of tiles (the diffusion itself: the next test)."""
    print(f"hole filling {w}x{h} holes {dead}", flush=True)
    d = lfrv.synth_desc(2, 11)
    d.grid, d.w, d.h, d.focal = 2, w, h, 1000.0 * w / 1024.0
    s = lfrv.synth(d)
    s["depths"] = s["depths"].copy()
    s["depths"][:, dead[2]:dead[3], dead[0]:dead[1]] = 0.0
    with lfrv.Context(pipelines.gradient_ibr_params(s)) as ctx:
        pipelines.load_scene(ctx, s)
        pipelines.gradient_ibr_solve(ctx, 1e-5, 3000)
        U = ctx.get_solution()
    r = oracle.gibr_pipeline(s["views"], s["depths"], s["P_views"], s["P_target"], 1, 1 / 255.0, 1.0, 1.0, 0.5, 1e-5, 3000)
    # two solves to a relative residual of 1e-5
    assert rel_err(U, r["U"]) < 1e-3


# (holes to three image edges, one tile past the second; whole tiles of holes; one column in the last tile; a hole
# across all inner tiles; a tile's middle row; more tiles than blocks).  The scale of the views sets when the rule
# fires: at sweeps that end a launch of eight, within one, at the first, and at the 500 of the cap, of which the last
# launch has four.
@pytest.mark.parametrize("w,h,holes,scale,sweeps", [
    (17, 33, (0, 17, 0, 16), 0.4, 5), (17, 33, (0, 17, 0, 16), 1.0, 7), (17, 33, (0, 17, 0, 16), 6.0, 56),
    (48, 40, (8, 40, 8, 24), 0.7, 14), (65, 20, (60, 65, 3, 20), 0.3, 1), (65, 20, (60, 65, 3, 20), 6.0, 11),
    (64, 48, (3, 60, 2, 47), 6.0, 500), (40, 41, (8, 24, 17, 33), 1.0, 16), (40, 41, (8, 24, 17, 33), 2.0, 26),
    (560, 530, (0, 560, 3, 530), 0.1, 60), (560, 530, (0, 560, 3, 530), 1.0, 500)])
def test_hole_sweeps_match_the_oracle(w, h, holes, scale, sweeps):
    """The Poisson diffusion in tiles of 16 x 16 and eight sweeps per launch: the filled image and the sweep at which
    the rule fires, against sweep after sweep in FP64."""
    print(f"hole filling {w}x{h} holes {holes} scale {scale}", flush=True)
    s = _planes(w, h, 1, 2, seed=11)
    s["views"] = (np.float32(scale) * s["views"]).astype(np.float32)
    vis = np.ones((h, w), np.uint8)
    vis[holes[2]:holes[3], holes[0]:holes[1]] = 0
    with lfrv.Context(pipelines.gradient_ibr_params(s)) as ctx:
        pipelines.load_scene(ctx, s)
        ctx.warps_from_depth()
        ctx.prepare()
        ctx.setup_visibility()
        ctx.compute_weights()
        ctx.set_buffer("VISIBILITY", vis.astype(np.float32))
        ctx.compute_initial_image()
        U, stats = ctx.get_solution(), ctx.hole_stats()
        tx, ty, om = [ctx.get_buffer(k).reshape(s["V"], h, w) for k in ("TAU_X", "TAU_Y", "OMEGA")]
    want, _ = oracle.initial_image(w, h, 1, tx, ty, s["views"], om)
    want, k = oracle.hole_filling(want, vis)
    # (the energies of FP32 images: their rounding is a percent at most of how far the rule was from firing)
    assert k == sweeps and stats == (int((vis == 0).sum()), sweeps)
    # a sweep rounds a mean and a sum of values of the image's scale: half an ulp each, averaged over the sweeps
    assert np.max(np.abs(U - want)) < scale * 6e-8 * (4 + sweeps)


@pytest.mark.parametrize("w,h,dsf", [(30, 7, 2), (31, 5, 2),    # one strip of 60 columns exactly, and two columns more
                                     (29, 4, 3), (14, 9, 4), (15, 3, 4)])
def test_box_iterations_at_strip_edges(w, h, dsf):
    """The marching PCG iteration of the box operator where its strips and row groups end, against the oracle."""
    s = _planes(w, h, dsf, 3, 5)
    print(f"PCG {w}x{h} dsf {dsf}", flush=True)
    with lfrv.Context(pipelines.gradient_ibr_params(s)) as ctx:
        pipelines.load_scene(ctx, s)
        st = pipelines.gradient_ibr_solve(ctx, 1e-6, 3000)
        U = ctx.get_solution()
    assert all(st["converged"])
    r = oracle.gibr_pipeline(s["views"], s["depths"], s["P_views"], s["P_target"], dsf, 1 / 255.0, 1.0, 1.0, 0.5, 1e-6, 3000)
    # two solves to a relative residual of 1e-6 of a system whose condition number is below 1e3
    assert rel_err(U, r["U"]) < 1e-3


def _address_row_by_row(ctx):
    """What planes of 2 GiB and more take: a buffer descriptor per row in the marching strips."""
    f = lfrv.lib().lfrv_test_narrow_bytes
    f.restype, f.argtypes = None, [ctypes.c_void_p, ctypes.c_size_t]
    f(ctx._h, 0)


@pytest.mark.parametrize("w,h,dsf,inner,beta", [(62, 5, 1, 1, 0.3), (57, 7, 1, 9, 0.0), (29, 7, 2, 1, 0.3), (61, 8, 2, 1, 0.0),
                                               (31, 3, 2, 0, 0.3), (31, 3, 2, 0, 0.0), (19, 16, 3, 1, 0.3), (40, 9, 3, 4, 0.0),
                                               (33, 6, 3, 0, 0.3), (14, 5, 4, 1, 0.3), (30, 4, 4, 2, 0.0), (20, 7, 4, 0, 0.3)])
def test_color_steps_addressed_row_by_row(w, h, dsf, inner, beta):
    """The forms of the marching step and of the primal-dual passes for planes beyond one descriptor: the same bits."""
    s = _planes(w, h, dsf, 3, seed=7)
    print(f"IBR_color row by row {w}x{h} dsf={dsf} inner={inner} beta={beta}", flush=True)
    out = []
    for wide in (False, True):
        with lfrv.Context(pipelines.color_sr_params(s, inner_iterations=inner, dt_beta=beta, gradient_step=1.0)) as ctx:
            if wide:
                _address_row_by_row(ctx)
            pipelines.load_scene(ctx, s)
            ctx.clear_solution()
            pipelines.color_sr_setup(ctx)
            ctx.sr_init_regularizer_weight()
            ctx.sr_iteration_fista()
            ctx.sr_iterate(4)
            out.append([ctx.get_buffer(k) for k in ("U", "UQ", "PX", "PY", "NORM_MASK") + (("G",) if inner != 1 else ())])
    for a, b in zip(*out):
        assert np.all(np.isfinite(a)) and np.array_equal(a, b)


@pytest.mark.parametrize("w,h,dsf", [(30, 7, 2), (31, 5, 2), (29, 4, 3), (14, 9, 4), (15, 3, 4)])
def test_box_iterations_addressed_row_by_row(w, h, dsf):
    """The marching PCG iteration for planes beyond one descriptor: the same bits."""
    s = _planes(w, h, dsf, 3, 5)
    print(f"PCG row by row {w}x{h} dsf {dsf}", flush=True)
    out = []
    for wide in (False, True):
        with lfrv.Context(pipelines.gradient_ibr_params(s)) as ctx:
            if wide:
                _address_row_by_row(ctx)
            pipelines.load_scene(ctx, s)
            st = pipelines.gradient_ibr_solve(ctx, 1e-6, 3000)
            out.append((ctx.get_solution(), st["iterations"]))
    assert out[0][1] == out[1][1] and np.array_equal(out[0][0], out[1][0])
