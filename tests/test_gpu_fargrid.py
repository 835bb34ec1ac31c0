"""Grids whose far charges are interpolated (csrc/fargrid.hip) against the FP64 oracle.

Tolerance, derived before the first run: a result is the FP64 sum rounded to float32 (2^-24
of each component) plus what the interpolation misses, at most 1e-9 of each charge's E term
and 1e-10 of its phi term (charges at the far threshold; the interpolation bound is checked
on the CPU below).  So, with A the sum of the terms' magnitudes,
    |E - E64| <= 1.1 * 2^-24 |E64| + 1e-9 A,   |phi - phi64| <= 1.1 * 2^-24 |phi64| + 1e-10 A.
"""
import numpy as np
import pytest

K = 14.3996451


def _mesh(axes):
    return np.stack(np.meshgrid(*axes, indexing="ij"), -1).reshape(-1, 3).astype(np.float32)


def _check(axes, x, q, E, phi, oracle_mod, soften=True):
    pts = _mesh(axes)
    at = np.random.default_rng(0).choice(len(pts), min(len(pts), 2000), replace=False)
    pts, E, phi = pts[at], None if E is None else E[at], None if phi is None else phi[at]
    E64, p64 = oracle_mod.field_f64(pts, x, q, want_phi=True, soften=soften)
    AE = np.empty(len(pts))
    AP = np.empty(len(pts))
    for a in range(0, len(pts), 100):
        d2 = ((pts[a:a + 100, None].astype(np.float64) - x[None]) ** 2).sum(2)
        AE[a:a + 100] = K * (np.abs(q) / np.maximum(d2, 1e-6)).sum(1)
        with np.errstate(divide="ignore"):
            AP[a:a + 100] = K * (np.abs(q) / np.sqrt(d2)).sum(1)
    if E is not None:
        err = np.linalg.norm(E - E64, axis=1)
        assert (err <= 1.1 * 2.0**-24 * np.linalg.norm(E64, axis=1) + 1e-9 * AE).all()
    if phi is not None:
        inf = np.isinf(p64)
        np.testing.assert_array_equal(phi[inf], p64[inf])
        err = np.abs(phi[~inf] - p64[~inf])
        assert (err <= 1.1 * 2.0**-24 * np.abs(p64[~inf]) + 1e-10 * AP[~inf]).all()


def test_interpolation_bound_at_the_threshold():
    """A charge on the ellipse of parameter 7 of a cell, in any direction and for cells of
    unequal sides: 12 Chebyshev nodes per axis miss at most 1e-9 of its E and 1e-10 of its
    phi (numpy, FP64)."""
    P, rho = 12, 7.0
    sigma = (rho + 1 / rho) / 2
    k = np.arange(P)
    node = np.cos((2 * k + 1) * np.pi / (2 * P))
    bary = (-1.0) ** k * np.sin((2 * k + 1) * np.pi / (2 * P))
    t = np.linspace(-1, 1, 8)
    L = bary / (t[:, None] - node[None])
    L /= L.sum(1, keepdims=True)
    rng = np.random.default_rng(1)

    def field(pts, c):
        d = pts - c
        r = np.linalg.norm(d, axis=-1, keepdims=True)
        return np.concatenate([d / r**3, 1 / r], -1)

    for trial in range(40):
        half = np.ones(3) if trial < 20 else rng.uniform(0.2, 1.0, 3)
        u = np.eye(3)[trial] if trial < 3 else rng.standard_normal(3)

        def far(s):
            d = np.abs(s * u)
            g2 = np.maximum(d - half, 0) ** 2
            return all(d[i] ** 2 / sigma**2 + (g2.sum() - g2[i]) / (sigma**2 - 1) >= half[i] ** 2
                       for i in range(3))

        lo, hi = 0.0, 100.0
        for _ in range(60):
            mid = 0.5 * (lo + hi)
            lo, hi = (lo, mid) if far(mid) else (mid, hi)
        c = hi * u
        V = field(np.stack(np.meshgrid(*[h * node for h in half], indexing="ij"), -1), c)
        got = np.einsum("ia,jb,kc,abcd->ijkd", L, L, L, V, optimize=True)
        ref = field(np.stack(np.meshgrid(*[h * t for h in half], indexing="ij"), -1), c)
        eE = np.linalg.norm(got[..., :3] - ref[..., :3], axis=-1)
        assert (eE / np.linalg.norm(ref[..., :3], axis=-1)).max() < 1e-9
        assert (np.abs(got[..., 3] - ref[..., 3]) / ref[..., 3]).max() < 1e-10


# (nx, ny, nz, charges, half width of the longest axis, charge ball radius)
SHAPES = [
    (8, 8, 27, 131_072, 1.3, 22.0),       # the smallest axes, the most charges
    (27, 27, 27, 10_200, 1.3, 10.0),      # one leaf, as large as it gets
    (28, 27, 55, 4_900, 2.7, 12.0),       # 1, 0 and 2 halvings
    (9, 54, 109, 3_800, 5.4, 14.0),       # 0, 1 and 3 halvings
    (8, 8, 432, 7_300, 21.0, 30.0),       # 4 halvings, the longest axis
    (37, 41, 43, 3_137, 2.1, 3.0),        # charges all over the box
]


@pytest.mark.gpu
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s[:4])))
def test_against_oracle(gpu_ctx, oracle_mod, shape):
    from pycpet_amd import ops

    nx, ny, nz, N, half, radius = shape
    rng = np.random.default_rng(N)
    d = rng.standard_normal((N, 3))
    x = (d / np.linalg.norm(d, axis=1, keepdims=True) * radius
         * rng.random((N, 1)) ** (1 / 3)).astype(np.float32)
    q = rng.normal(0, 0.4, N).astype(np.float32)
    step = 2 * half / (max(nx, ny, nz) - 1)
    axes = [np.linspace(-0.5 * (n - 1) * step, 0.5 * (n - 1) * step, n).astype(np.float32)
            for n in (nx, ny, nz)]
    print(f"case {shape}", flush=True)
    E, phi = ops.field_grid(*axes, x, q, want_phi=True, ctx=gpu_ctx)
    assert gpu_ctx.refined_points() == 0
    _check(axes, x, q, E, phi, oracle_mod)
    E1, _ = ops.field_grid(*axes, x, q, ctx=gpu_ctx)
    _, p1 = ops.field_grid(*axes, x, q, want_E=False, want_phi=True, ctx=gpu_ctx)
    _check(axes, x, q, E1, p1, oracle_mod)
    Eh, _ = ops.field_grid(*axes, x, q, soften=False, ctx=gpu_ctx)
    _check(axes, x, q, Eh, None, oracle_mod, soften=False)


def _frame(seed=3, N=5000, n=(41, 30, 43)):
    rng = np.random.default_rng(seed)
    x = rng.uniform(-9, 9, (N, 3)).astype(np.float32)
    q = rng.normal(0, 0.4, N).astype(np.float32)
    axes = [np.linspace(-0.05 * (k - 1), 0.05 * (k - 1), k).astype(np.float32) for k in n]
    return axes, x, q


@pytest.mark.gpu
def test_charges_on_and_beside_grid_points(gpu_ctx, oracle_mod):
    """The r^2 >= 1e-6 floor of E and phi = inf on a charge."""
    from pycpet_amd import ops

    axes, x, q = _frame()
    g = np.array([axes[0][7], axes[1][20], axes[2][11]], np.float32)
    for i, off in enumerate((0.0, 4e-4, 9e-4, 2e-3)):
        x[i] = g + np.float32(off) * np.eye(3, dtype=np.float32)[i % 3]
    E, phi = ops.field_grid(*axes, x, q, want_phi=True, ctx=gpu_ctx)
    assert np.isfinite(E).all() and np.isinf(phi).sum() == 1
    _check(axes, x, q, E, phi, oracle_mod)


@pytest.mark.gpu
def test_axes_in_any_order(gpu_ctx, oracle_mod):
    """Unsorted, repeated and unevenly spaced axis values."""
    from pycpet_amd import ops

    axes, x, q = _frame(seed=4)
    rng = np.random.default_rng(0)
    axes[0] = rng.permutation(axes[0])
    axes[1][:] = np.repeat(axes[1][::10], 10)
    axes[2] = np.sort(rng.uniform(-2, 2, axes[2].size)).astype(np.float32)[::-1].copy()
    E, phi = ops.field_grid(*axes, x, q, want_phi=True, ctx=gpu_ctx)
    _check(axes, x, q, E, phi, oracle_mod)


@pytest.mark.gpu
def test_values_that_are_not_finite(gpu_ctx):
    """Infinite, NaN and huge inputs give what the direct kernel gives: nothing for a charge
    beyond the FP32 range, the same components NaN for a charge, or at the points of an axis
    value, that is not finite."""
    from pycpet_amd import ops

    axes, x, q = _frame(seed=5)

    def both():
        far = ops.field_grid(*axes, x, q, want_phi=True, ctx=gpu_ctx)
        gpu_ctx.set_tuning(0, 2, 0)
        try:
            direct = ops.field_grid(*axes, x, q, want_phi=True, ctx=gpu_ctx)
        finally:
            gpu_ctx.set_tuning(0, 0, 0)
        for a, b in zip(far, direct):
            np.testing.assert_array_equal(np.isnan(a), np.isnan(b))
            ok = np.isfinite(b)
            scale = np.sqrt(np.mean(b[ok].astype(float) ** 2)) if ok.any() else 1.0
            np.testing.assert_allclose(a[ok], b[ok], rtol=1e-4, atol=1e-5 * scale)
        return far

    keep = x[0].copy()
    x[0] = (1e25, 0, 0)
    assert np.isfinite(both()[0]).all()
    for bad in (np.inf, np.nan):
        x[0] = (bad, 0, 0)
        assert np.isnan(both()[0]).any()
        x[0] = keep
        q0, q[0] = q[0], bad
        both()
        q[0] = q0
    for bad in (np.inf, np.nan):
        v, axes[1][4] = axes[1][4], bad
        E = both()[0].reshape(41, 30, 43, 3)
        assert np.isnan(E[:, 4]).any() and np.isfinite(np.delete(E, 4, 1)).all()
        axes[1][4] = v


@pytest.mark.gpu
def test_batch_equals_single(gpu_ctx):
    """Frames of both paths in one batch: the interpolated ones equal the frame run alone to
    FP64 rounding of the node sums (one float32 rounding), host or device arrays alike."""
    import torch

    from pycpet_amd import batch, ops

    frames = []
    for k, (N, n) in enumerate([(5000, (41, 30, 43)), (300, (9, 9, 9)), (9000, (60, 27, 28)),
                                (4000, (41, 41, 41))]):
        axes, x, q = _frame(seed=10 + k, N=N, n=n)
        frames.append({"axes": axes, "x": x, "q": q})
    outs = batch.batch_volume(frames, want_phi=True, ctx=gpu_ctx)
    for f, (E, phi) in zip(frames, outs):
        E1, p1 = ops.field_grid(*f["axes"], f["x"], f["q"], want_phi=True, ctx=gpu_ctx)
        for a, b in ((E, E1), (phi, p1)):
            scale = np.sqrt(np.mean(b.astype(float) ** 2))
            np.testing.assert_allclose(a, b, rtol=5e-6, atol=1e-7 * scale)
    T = lambda a: torch.from_numpy(a).cuda()
    dev = [{"axes": tuple(T(a) for a in f["axes"]), "x": T(f["x"]), "q": T(f["q"])}
           for f in frames]
    for (E, phi), (Et, pt) in zip(outs, batch.batch_volume(dev, want_phi=True, ctx=gpu_ctx)):
        np.testing.assert_array_equal(E, Et.cpu().numpy())
        np.testing.assert_array_equal(phi, pt.cpu().numpy())


@pytest.mark.gpu
@pytest.mark.parametrize("batched", [False, True])
def test_captured_replays(gpu_ctx, batched):
    """In a HIP graph: every replay equals the eager call, with other inputs in between."""
    import torch

    from pycpet_amd import batch, graphs, ops

    T = lambda a: torch.from_numpy(a).cuda()
    fr = []
    for k in range(2):
        axes, x, q = _frame(seed=20 + k, N=5000 + 700 * k)
        fr.append({"axes": tuple(T(a) for a in axes), "x": T(x), "q": T(q)})
    if batched:
        fn = lambda ctx: torch.cat([E for E, _ in batch.batch_volume(fr, ctx=ctx)])
    else:
        fn = lambda ctx: ops.field_grid(*fr[0]["axes"], fr[0]["x"], fr[0]["q"], ctx=ctx)[0]
    step = graphs.CapturedStep(fn)
    for k in range(3):
        fr[0]["x"].add_(0.01 * k)
        got = step.replay()
        torch.cuda.synchronize()
        want = fn(gpu_ctx)
        torch.cuda.synchronize()
        assert torch.equal(got, want)
    step.close()


@pytest.mark.gpu
@pytest.mark.parametrize("what", ["E", "E unsoftened", "phi"])
def test_one_output_of_values_that_are_not_finite(gpu_ctx, what):
    """E alone (with and without the floor) and phi alone of infinite and NaN charges and axis
    values: the same components are NaN as in the direct kernel, the others agree.  E alone is
    NaN in all three components for a NaN coordinate: no charge is within the floor's reach."""
    from pycpet_amd import ops

    axes, x, q = _frame(seed=6)
    kw = {"want_E": what != "phi", "want_phi": what == "phi", "soften": what != "E unsoftened"}

    def same():
        far = [a for a in ops.field_grid(*axes, x, q, ctx=gpu_ctx, **kw) if a is not None][0]
        gpu_ctx.set_tuning(0, 2, 0)
        try:
            direct = [a for a in ops.field_grid(*axes, x, q, ctx=gpu_ctx, **kw)
                      if a is not None][0]
        finally:
            gpu_ctx.set_tuning(0, 0, 0)
        np.testing.assert_array_equal(np.isnan(far), np.isnan(direct))
        ok = np.isfinite(direct)
        scale = np.sqrt(np.mean(direct[ok].astype(float) ** 2)) if ok.any() else 1.0
        np.testing.assert_allclose(far[ok], direct[ok], rtol=1e-4, atol=1e-5 * scale)
        return far

    keep = x[0].copy()
    for bad in (np.inf, np.nan):
        for k in range(3):
            x[0, k] = bad
            far = same()
            x[0] = keep
            if np.isnan(bad):
                assert np.isnan(far).all()
        q0, q[0] = q[0], bad
        same()
        q[0] = q0
        v, axes[1][4] = axes[1][4], bad
        same()
        axes[1][4] = v


@pytest.mark.gpu
def test_captured_batch_of_several_scratch_groups(gpu_ctx):
    """A batch whose node sums and near lists need more than the 1 GiB that one launch may take
    (8 frames, 512 leaves each, 65,536 charges: 134 MB of near list a frame) runs in several; it
    can be captured, its replays follow the inputs, and its frames equal the frames run alone
    to one float32 rounding."""
    import torch

    from pycpet_amd import batch, graphs, ops

    rng = np.random.default_rng(31)
    T = lambda a: torch.from_numpy(a).cuda()
    axis = T(np.linspace(-2.7, 2.7, 109).astype(np.float32))
    fr = [{"axes": (axis, axis, axis),
           "x": T(rng.uniform(-40, 40, (65536, 3)).astype(np.float32)),
           "q": T(rng.normal(0, 0.4, 65536).astype(np.float32))} for _ in range(8)]
    fn = lambda ctx: torch.cat([E for E, _ in batch.batch_volume(fr, ctx=ctx)])
    step = graphs.CapturedStep(fn)
    for k in range(3):
        fr[k]["x"].add_(0.05)
        got = step.replay()
        torch.cuda.synchronize()
        want = fn(gpu_ctx)
        torch.cuda.synchronize()
        assert torch.equal(got, want)
    step.close()
    M = 109 ** 3
    for k in (0, 7):
        one, _ = ops.field_grid(axis, axis, axis, fr[k]["x"], fr[k]["q"], ctx=gpu_ctx)
        b = want[k * M:(k + 1) * M]
        scale = float(one.double().square().mean().sqrt())
        assert float((one - b).abs().max()) <= 1e-7 * scale + 5e-6 * float(one.abs().max())


@pytest.mark.gpu
@pytest.mark.parametrize("n, charges", [((217, 217, 217), 200), ((217, 218, 217), 45000)])
def test_largest_plan(oracle_mod, n, charges):
    """Four halvings on every axis (4,681 cells, 100 KB of LDS in the classification), with few
    charges, and with so many that the near lists of all leaves would need 740 MB: right, and
    within 1 GiB of scratch (and the quarter that the context adds)."""
    import torch

    from pycpet_amd import _native as nat, batch, ops

    rng = np.random.default_rng(charges)
    x = rng.uniform(-25, 25, (charges, 3)).astype(np.float32)
    q = rng.normal(0, 0.4, charges).astype(np.float32)
    x[:40] *= np.float32(0.15)  # in the box
    axes = [np.linspace(-5.4, 5.4, k).astype(np.float32) for k in n]
    T = lambda a: torch.from_numpy(a).cuda()
    xd, qd, ad = T(x), T(q), [T(a) for a in axes]
    out = torch.empty((int(np.prod(n)), 3), device="cuda")  # what the call's result will use
    del out
    ctx = nat.Context(0)
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    E, _ = ops.field_grid(*ad, xd, qd, ctx=ctx)
    torch.cuda.synchronize()
    assert free - torch.cuda.mem_get_info()[0] <= 1.3 * 2**30
    _check(axes, x, q, E.cpu().numpy(), None, oracle_mod)
    few = {"x": xd[:9000], "q": qd[:9000], "axes": [a[::5].contiguous() for a in ad]}
    big = {"x": xd, "q": qd, "axes": ad}
    out = batch.batch_volume([few, big, few], ctx=ctx)  # in a batch: a launch of its own
    scale = float(E.double().square().mean().sqrt())
    assert float((out[1][0] - E).abs().max()) <= 1e-7 * scale + 5e-6 * float(E.abs().max())
    for k in (0, 2):
        _check([a[::5] for a in axes], x[:9000], q[:9000], out[k][0].cpu().numpy(), None,
               oracle_mod)
    del E, out
    ctx.close()


@pytest.mark.gpu
@pytest.mark.parametrize("batched", [False, True])
@pytest.mark.parametrize("name", ["shell", "mirror"])
def test_points_where_the_field_cancels(gpu_ctx, oracle_mod, name, batched):
    """Layouts whose interpolation misses add up while the field itself cancels (E of 1e-6 of
    the terms' magnitudes A and less): points below 2e-5 of it are summed directly, whose pair
    terms are good to 1e-14, so 1e-13 A beside the rounding is allowed there."""
    from pycpet_amd import batch, ops

    rng = np.random.default_rng(4)
    if name == "shell":  # equal charges on a sphere: E ~ 0 inside
        k = np.arange(6000) + 0.5
        ph, th = np.arccos(1 - 2 * k / 6000), np.pi * (1 + 5 ** 0.5) * k
        x = 9 * np.stack([np.cos(th) * np.sin(ph), np.sin(th) * np.sin(ph), np.cos(ph)], 1)
        q = np.full(6000, 0.3)
    else:  # point symmetric: E = 0 at the centre
        h = rng.uniform(-12, 12, (3000, 3))
        h = h[(np.abs(h) > 3.5).any(1)]
        x = np.concatenate([h, -h])
        q = np.tile(rng.normal(0, 0.4, len(h)), 2)
    x, q = x.astype(np.float32), q.astype(np.float32)
    axes = [np.linspace(-2, 2, 41).astype(np.float32)] * 3
    if batched:
        E = batch.batch_volume([{"axes": axes, "x": x, "q": q}] * 2, ctx=gpu_ctx)[1][0]
    else:
        E, _ = ops.field_grid(*axes, x, q, ctx=gpu_ctx)
    E2, _ = ops.field_grid(*axes, x, q, want_phi=True, ctx=gpu_ctx)
    pts = _mesh(axes)
    at = np.unique(np.concatenate([[len(pts) // 2], rng.choice(len(pts), 1500, replace=False)]))
    pts = pts[at]
    E64, _ = oracle_mod.field_f64(pts, x, q)
    A = np.empty(len(pts))
    for a in range(0, len(pts), 100):
        d2 = ((pts[a:a + 100, None].astype(np.float64) - x[None]) ** 2).sum(2)
        A[a:a + 100] = K * (np.abs(q) / d2).sum(1)
    nE = np.linalg.norm(E64, axis=1)
    low = nE <= 1e-5 * A
    assert low[at == 41 ** 3 // 2].all() and (name == "mirror" or low.all())
    for e in (E[at], E2[at]):
        err = np.linalg.norm(e - E64, axis=1)
        assert (err <= 1.1 * 2.0**-24 * nE + np.where(low, 1e-13, 1e-9) * A).all()
