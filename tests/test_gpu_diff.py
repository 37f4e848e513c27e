"""GPU differentiable rendering (ft_diff_*) through the C ABI.

  * forward (t*, s) against the oracle's f32 forward of the same parametric scene;
  * adjoint gradient against central finite differences (h = 1e-4) of the oracle's FP64
    forward, every parameter, relative error <= 1e-3 each (8 and 32 spheres), and the
    directional derivative at the benchmark's full size;
  * one sphere: dt*/d(centre, radius) against the analytic derivative of the ray/sphere root;
  * Adam fit lowers the loss; the torch.autograd.Function gives the C-ABI gradient.
"""
import math

import numpy as np
import pytest

from forgedthoughts_amd import synthetic
from forgedthoughts_amd.diff import DiffRenderer, sphere_tree_render
from forgedthoughts_amd.options import RenderOptions
from oracle import ftref

pytestmark = pytest.mark.gpu


def interior(t, max_jump=0.1):
    """Pixels whose 3x3 neighbourhood hits the surface with no depth discontinuity: away
    from silhouettes and occlusion edges, where t is a smooth function of the parameters."""
    from scipy.ndimage import binary_erosion, maximum_filter, minimum_filter
    hit = t >= 0
    out = binary_erosion(hit, structure=np.ones((1, 3, 3)), border_value=0)
    tt = np.where(hit, t, 0.0)
    jump = maximum_filter(tt, size=(1, 3, 3)) - minimum_filter(tt, size=(1, 3, 3))
    return out & (jump < max_jump)


@pytest.fixture(scope="module")
def small():
    return synthetic.adjoint_fit(n_prims=8, n_views=2, size=64, steps=30)


def test_forward_matches_oracle(small):
    w = small
    print(f"[diff forward] n={w.n_prims} views={len(w.views)} {w.options.width}^2", flush=True)
    with DiffRenderer(w.n_prims, w.views, w.options, w.light_dir, w.normal_step) as dr:
        dr.set_params(w.params_true)
        t, s = dr.forward()
    tc, sc = ftref.diff_forward(w.n_prims, np.float32(w.params_true), w.views, w.options, w.light_dir,
                                w.normal_step, precision=0)
    mism = int(((t >= 0) != (tc >= 0)).sum())
    assert mism <= max(1, int(1e-4 * t.size)), mism
    both = (t >= 0) & (tc >= 0)
    assert np.abs(t - tc)[both].max() <= 1e-4
    assert np.abs(s - sc)[both].max() <= 2e-3


def _adjoint_vs_fd(w, p32, h=1e-4):
    """The GPU adjoint g = J^T u for upstream gradients u = dL/d(t, s) of an L2 loss at the
    GPU forward, against central differences (step h) of the FP64 oracle's forward
    projected on the same u: fd_j = u . (F(p + h e_j) - F(p - h e_j)) / 2h, per parameter."""
    import torch
    p = p32.astype(np.float64)
    tt, st = ftref.diff_forward(w.n_prims, w.params_true, w.views, w.options, w.light_dir, w.normal_step, precision=1)
    with DiffRenderer(w.n_prims, w.views, w.options, w.light_dir, w.normal_step) as dr:
        dr.set_params(p32)
        t, s = dr.forward()
        m = interior(t) & interior(tt)
        ut = (2.0 * (t - tt) * m).astype(np.float32)
        us = (2.0 * (s - st) * m).astype(np.float32)
        gt = torch.from_numpy(ut).cuda()
        gs = torch.from_numpy(us).cuda()
        torch.cuda.synchronize()
        g = dr.backward_device(gt.data_ptr(), gs.data_ptr())

    def proj(q):
        a, b = ftref.diff_forward(w.n_prims, q, w.views, w.options, w.light_dir, w.normal_step, precision=1)
        return float((ut * np.where(m, a, 0.0)).sum() + (us * np.where(m, b, 0.0)).sum())

    fd = np.zeros_like(p)
    for j in range(p.size):
        e = np.zeros_like(p)
        e[j] = h
        fd[j] = (proj(p + e) - proj(p - e)) / (2 * h)
    return g, fd


def _perturbed(w):
    return np.float32(w.params_true) + np.float32(0.02) * np.float32(np.sin(np.arange(len(w.params_true))))


def _check_per_parameter(g, fd, label):
    floor = 1e-5 * np.abs(fd).max()
    bad = np.abs(g - fd) > 1e-3 * np.abs(fd) + floor
    rel = np.abs(g - fd) / np.maximum(np.abs(fd), floor)
    print(f"[diff grad {label}] worst per-parameter relative error {rel.max():.2e} (param {int(rel.argmax())}), "
          f"floor {floor:.2e}", flush=True)
    assert not bad.any(), [(int(j), float(g[j]), float(fd[j])) for j in np.nonzero(bad)[0]]


def test_gradient_per_parameter_small(small):
    w = small
    g, fd = _adjoint_vs_fd(w, _perturbed(w))
    _check_per_parameter(g, fd, "8 prims")


def test_gradient_per_parameter_32_prims():
    """All 159 parameters of the 32-sphere workload (centres, radii, every blend radius), 4
    views at 128^2: |g_j - fd_j| <= 1e-3 |fd_j| + 1e-5 max|fd| for every j."""
    w = synthetic.adjoint_fit(n_prims=32, n_views=4, size=128)
    print(f"[diff grad] 32 prims, {len(w.views)} views at 128^2", flush=True)
    g, fd = _adjoint_vs_fd(w, _perturbed(w))
    _check_per_parameter(g, fd, "32 prims")


def test_gradient_directional_full_size():
    """The benchmark's size (32 spheres, 16 views at 512^2): the adjoint's directional
    derivative g . v along a random unit direction against the FP64 oracle's central
    difference of the same projected loss."""
    import torch
    w = synthetic.adjoint_fit()
    p32 = _perturbed(w)
    p = p32.astype(np.float64)
    tt, st = ftref.diff_forward(w.n_prims, w.params_true, w.views, w.options, w.light_dir, w.normal_step, precision=1)
    with DiffRenderer(w.n_prims, w.views, w.options, w.light_dir, w.normal_step) as dr:
        dr.set_params(p32)
        t, s = dr.forward()
        m = interior(t) & interior(tt)
        ut = (2.0 * (t - tt) * m).astype(np.float32)
        us = (2.0 * (s - st) * m).astype(np.float32)
        gt = torch.from_numpy(ut).cuda()
        gs = torch.from_numpy(us).cuda()
        torch.cuda.synchronize()
        g = dr.backward_device(gt.data_ptr(), gs.data_ptr())
    v = np.random.default_rng(7).standard_normal(p.size)
    v /= np.linalg.norm(v)
    h = 1e-4

    def proj(q):
        a, b = ftref.diff_forward(w.n_prims, q, w.views, w.options, w.light_dir, w.normal_step, precision=1)
        return float((ut * np.where(m, a, 0.0)).sum() + (us * np.where(m, b, 0.0)).sum())
    fd = (proj(p + h * v) - proj(p - h * v)) / (2 * h)
    gv = float(np.dot(g, v))
    print(f"[diff grad full] g.v {gv:.6e} fd {fd:.6e}", flush=True)
    assert abs(gv - fd) <= 1e-3 * abs(fd), (gv, fd)


def test_single_sphere_analytic_derivative():
    views = [(0, (0.3, 0.2, 6.0), (0.0, 0.0, 0.0), 30.0)]
    opts = RenderOptions(33, 33, 256, 30.0, 1.0e-5, 0.7, 6.0, 30.0)
    c = np.array([0.1, -0.2, 0.3])
    r = 1.1
    import torch
    with DiffRenderer(1, views, opts, (0.0, 0.0, 1.0), 1.0e-2) as dr:
        dr.set_params(np.float32(list(c) + [r]))
        t, _ = dr.forward()
        for (y, x) in ((16, 16), (10, 20), (22, 13)):
            seed = np.zeros_like(t)
            seed[0, y, x] = 1.0
            gt = torch.from_numpy(seed).cuda()
            torch.cuda.synchronize()
            g = dr.backward_device(gt.data_ptr(), 0)
            # the pixel's ray, from the camera basis of the view (origin o, target 0, fov 30)
            o = np.array(views[0][1])
            fwd = -o / np.linalg.norm(o)
            right = np.cross(fwd, [0, 1, 0]); right /= np.linalg.norm(right)
            up = np.cross(right, fwd); up /= np.linalg.norm(up)
            tanf = math.tan(math.radians(15.0))
            px = ((x + 0.5) / 33) * 2 - 1
            py = 1 - ((y + 0.5) / 33) * 2
            d = fwd + right * px * tanf + up * py * tanf
            d /= np.linalg.norm(d)
            hit = o + d * t[0, y, x]
            n = (hit - c) / np.linalg.norm(hit - c)
            # root of |o + t d - c| = r: dt/dr = 1 / (n . d), dt/dc = n / (n . d)
            nd = float(np.dot(n, d))
            dt_dr = 1.0 / nd
            dt_dc = n / nd
            assert abs(g[3] - dt_dr) <= 1e-3 * abs(dt_dr), (g, dt_dr)
            assert np.abs(g[:3] - dt_dc).max() <= 1e-3 * np.abs(dt_dc).max() + 1e-6, (g, dt_dc)


def test_fit_lowers_loss(small):
    w = small
    tt, st = ftref.diff_forward(w.n_prims, w.params_true, w.views, w.options, w.light_dir, w.normal_step, precision=0)
    with DiffRenderer(w.n_prims, w.views, w.options, w.light_dir, w.normal_step) as dr:
        dr.set_params(w.params_init)
        dr.set_target(tt.astype(np.float32), st.astype(np.float32))
        losses = dr.fit(w.steps, w.lr)
        assert np.isfinite(losses).all()
        assert losses[-1] < 0.5 * losses[0], losses
        p = dr.get_params()
    e0 = np.abs(np.float32(w.params_init) - np.float32(w.params_true)).mean()
    e1 = np.abs(p - np.float32(w.params_true)).mean()
    print(f"[diff fit] loss {losses[0]:.4g} -> {losses[-1]:.4g}; param error {e0:.4f} -> {e1:.4f}", flush=True)


def test_torch_autograd_function(small):
    import torch
    w = small
    tt, st = ftref.diff_forward(w.n_prims, w.params_true, w.views, w.options, w.light_dir, w.normal_step, precision=0)
    with DiffRenderer(w.n_prims, w.views, w.options, w.light_dir, w.normal_step) as dr:
        params = torch.tensor(w.params_init, dtype=torch.float32, device="cuda", requires_grad=True)
        t, s = sphere_tree_render(params, dr)
        m = torch.from_numpy(interior(t.detach().cpu().numpy()) & interior(tt)).cuda()
        T = torch.from_numpy(tt.astype(np.float32)).cuda()
        S = torch.from_numpy(st.astype(np.float32)).cuda()
        loss = (((t - T) ** 2) * m).sum() + (((s - S) ** 2) * m).sum()
        loss.backward()
        gt = (2 * (t.detach() - T) * m).contiguous()
        gs = (2 * (s.detach() - S) * m).contiguous()
        torch.cuda.synchronize()
        ref = dr.backward_device(gt.data_ptr(), gs.data_ptr())
    np.testing.assert_allclose(params.grad.cpu().numpy(), np.float32(ref), rtol=1e-5, atol=1e-6)


def test_counted_kernels_match_and_count(small):
    """The FLOP-counting forward / adjoint give the same loss and gradient as the timed
    kernels, and count at least the march's minimum work (every pixel of every view evaluates
    the tree at least once; a hit adds 10 bisection steps and 6 normal samples)."""
    w = small
    tt, st = ftref.diff_forward(w.n_prims, w.params_true, w.views, w.options, w.light_dir, w.normal_step, precision=0)
    with DiffRenderer(w.n_prims, w.views, w.options, w.light_dir, w.normal_step) as dr:
        dr.set_params(w.params_init)
        dr.set_target(tt.astype(np.float32), st.astype(np.float32))
        l0, g0 = dr.loss_grad()
        dr.set_flop_counting(True)
        l1, g1 = dr.loss_grad()
        flops = dr.stats().sdf_flops
        dr.set_flop_counting(False)
        t, _ = dr.forward()
    assert l0 == l1
    np.testing.assert_array_equal(g0, g1)
    per_eval = 10 * w.n_prims + 13 * (w.n_prims - 1)
    hits = int((t >= 0).sum())
    assert flops >= per_eval * (t.size + 16 * hits)


# losses with every join of the tree evaluated at every point, lengths as fma(z, z, fma(x, x, y y))
WHOLE_TREE_LOSS = {19: 38373.98785014648, 31: 42602.08975846099, 36: 28493.01545299478, 42: 23275.965396354408}


@pytest.mark.parametrize("seed", list(WHOLE_TREE_LOSS))
def test_loss_is_that_of_the_whole_tree(seed):
    """Views with a ray along a silhouette that hits or misses on a last bit of a distance: rounded
    another way, that pixel moves the loss by 3.6e-5 to 5.9e-4.  What the cells leave out cannot
    show, so the distances are the whole tree's bit for bit.  The derivative of the Newton step may
    round another way: a last bit of t* (2^-21 at most 8 away) in any of the N pixels moves
    sum (t* - T)^2 by at most 2^-20 sqrt(N loss), 0.09 to 0.13 here: 4e-6 of the loss and less."""
    rng = np.random.default_rng(seed)
    target = np.concatenate([np.concatenate([rng.uniform(-2, 2, 3), rng.uniform(0.4, 0.9, 1)]) for _ in range(32)]
                            + [rng.uniform(0.1, 0.4, 31)])
    now = target + rng.normal(0, 0.05, target.size)
    views = []
    for _ in range(4):
        z, phi = rng.uniform(-0.5, 0.9), rng.uniform(0, 2 * np.pi)
        r = np.sqrt(1 - z * z)
        views.append((0, (7 * r * np.cos(phi), 7 * z, 7 * r * np.sin(phi)), (0.0, 0.0, 0.0), 45.0))
    opts = RenderOptions(width=320, height=320, max_steps=256, max_dist=30.0, epsilon=1e-5, step_scale=0.7,
                         camera_z=6.0, fov_y_degrees=45.0)
    print(f"[diff loss] seed {seed}, 32 prims, 4 views at 320^2", flush=True)
    with DiffRenderer(32, views, opts) as dr:
        dr.set_params(np.float32(target))
        dr.set_target(*dr.forward())
        dr.set_params(np.float32(now))
        loss, _ = dr.loss_grad()
    want = WHOLE_TREE_LOSS[seed]
    assert abs(loss - want) <= 2.0 ** -20 * math.sqrt(4 * 320 * 320 * want), (loss, want)


def test_adjoint_of_more_tiles_than_waves():
    """Beyond 65536 tiles a wave of the adjoint takes several, the last ones of it none: the gradient is the
    sum of those of its views' halves, to the order of the double sums."""
    import torch
    opts = RenderOptions(width=130, height=130, max_steps=64, max_dist=30.0, epsilon=1e-3, step_scale=0.7,
                         camera_z=6.0, fov_y_degrees=45.0)
    n = 230  # views of 17 x 17 tiles: 66470 in all
    rng = np.random.default_rng(4)
    params = np.float32([-0.4, 0.1, 0.0, 0.7, 0.5, -0.1, 0.2, 0.6, 0.2])
    views = []
    for k in range(n):
        phi = 2 * np.pi * k / n
        views.append((0, (5 * np.cos(phi), 1.0, 5 * np.sin(phi)), (0.0, 0.0, 0.0), 45.0))
    up = np.float32(rng.normal(size=(2, n, 130, 130)))
    print(f"[diff adjoint] {n} views at 130^2", flush=True)

    def gradient(lo, hi):
        with DiffRenderer(2, views[lo:hi], opts) as dr:
            dr.set_params(params)
            dr.forward()
            gt, gs = (torch.from_numpy(np.ascontiguousarray(u[lo:hi])).cuda() for u in up)
            torch.cuda.synchronize()
            return dr.backward_device(gt.data_ptr(), gs.data_ptr())
    whole, parts = gradient(0, n), gradient(0, n // 2) + gradient(n // 2, n)
    assert np.abs(whole).max() > 1.0
    np.testing.assert_allclose(whole, parts, rtol=1e-9, atol=1e-9 * np.abs(whole).max())
