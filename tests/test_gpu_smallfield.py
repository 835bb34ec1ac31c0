"""The one-launch path of small field calls against the FP64 oracle and, where
results are not finite or the floor of the softened field binds, against the
all-FP64-pair-term ("mixed") precision of the direct path.

Tolerance: the sums are FP64 with pair terms good to 1e-13, so a float32 result
is the rounding (2^-24) of a value within 1e-12 of the sum of the terms'
magnitudes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

K = 14.3996451


def _charges(N, seed):
    from pycpet_amd import workloads as W

    x, q = W.ball_exclusion(N, 30.0, 1.0, 1.5, seed)
    if N == 1:
        q = np.array([0.5], np.float32)
    return x, q


def _check(pts, x, q, E, phi, oracle_mod):
    E64, p64 = oracle_mod.field_f64(pts, x, q, want_phi=True)
    d = pts[:, None, :].astype(np.float64) - x[None].astype(np.float64)
    r2 = (d ** 2).sum(2)
    aq = K * np.abs(q.astype(np.float64))[None]
    if E is not None:
        assert (np.abs(E - E64) <= 2.0 ** -24 * np.abs(E64)
                + 1e-12 * (aq / r2).sum(1)[:, None]).all()
    if phi is not None:
        assert (np.abs(phi - p64) <= 2.0 ** -24 * np.abs(p64)
                + 1e-12 * (aq / np.sqrt(r2)).sum(1)).all()


# points on both sides of each workgroup shape (3, 12 and 48 points per CU of
# 256), charges around a stage's 1,024 and a workgroup's splits
@pytest.mark.parametrize("M,N", [(1, 1), (1, 7890), (2, 1023), (768, 1025), (769, 1024),
                                 (3072, 63), (3073, 65), (12288, 17), (12289, 33), (5, 70001)])
def test_points(gpu_ctx, oracle_mod, M, N):
    from pycpet_amd import ops

    x, q = _charges(N, seed=N)
    pts = np.random.default_rng(M).uniform(-1, 1, (M, 3)).astype(np.float32)
    sel = np.unique(np.linspace(0, M - 1, 60).astype(int))
    for kw in ({}, {"soften": False}, {"want_phi": True}, {"want_E": False, "want_phi": True}):
        E, phi = ops.field_points(pts, x, q, ctx=gpu_ctx, **kw)
        _check(pts[sel], x, q, None if E is None else E[sel], None if phi is None else phi[sel],
               oracle_mod)


@pytest.mark.parametrize("shape,N", [((1, 1, 1), 500), ((3, 1, 7), 1500), ((13, 9, 8), 2048),
                                     ((21, 21, 21), 2001), ((29, 31, 37), 700)])
def test_grids(gpu_ctx, oracle_mod, shape, N):
    from pycpet_amd import ops

    x, q = _charges(N, seed=N)
    axes = [np.linspace(-1.0, 0.7 + 0.1 * i, n).astype(np.float32) for i, n in enumerate(shape)]
    pts = np.stack(np.meshgrid(*axes, indexing="ij"), -1).reshape(-1, 3)
    sel = np.unique(np.linspace(0, len(pts) - 1, 60).astype(int))
    for kw in ({}, {"want_phi": True}, {"want_E": False, "want_phi": True}):
        E, phi = ops.field_grid(*axes, x, q, ctx=gpu_ctx, **kw)
        _check(pts[sel], x, q, None if E is None else E[sel], None if phi is None else phi[sel],
               oracle_mod)


def test_special_values(gpu_ctx):
    """A charge on a point, charges inside the r^2 floor, beyond the FP32 range
    of r^2, infinite, not a number, and of zero and of no charge."""
    from pycpet_amd import ops

    ax = np.linspace(-1, 1, 5).astype(np.float32)
    pts = np.stack(np.meshgrid(ax, ax, ax, indexing="ij"), -1).reshape(-1, 3).copy()
    x0, q0 = _charges(40, seed=4)
    cases = {"on a point": ([0.5, 0.0, -0.5], 0.4), "in the floor": ([0.5004, 0.0, -0.5], 0.4),
             "uncharged on a point": ([0.5, 0.0, -0.5], 0.0), "far": ([1e25, -1e20, 3.0], 0.4),
             "infinite": ([np.inf, 0.0, 0.0], 0.4), "nan": ([0.1, np.nan, 0.0], 0.4),
             "infinite charge": ([2.0, 2.0, 2.0], np.inf)}
    for name, (p, c) in cases.items():
        x = np.concatenate([x0, np.array([p], np.float32)])
        q = np.concatenate([q0, np.array([c], np.float32)])
        print(name, flush=True)
        for kw in ({}, {"soften": False}, {"want_phi": True}, {"want_E": False, "want_phi": True}):
            for run in (lambda x, q, **k: ops.field_points(pts, x, q, ctx=gpu_ctx, **k),
                        lambda x, q, **k: ops.field_grid(ax, ax, ax, x, q, ctx=gpu_ctx, **k)):
                got = run(x, q, **kw)
                if name == "infinite":
                    # as the FP32 sums of the direct path have it (FP64 outputs take
                    # it): not a number along x and in phi, and nothing added to
                    # the others ("mixed" clamps 1 / r there)
                    direct, without = run(x, q, out_f64=True, **kw), run(x0, q0, **kw)
                    for a, b, w in zip(got, direct, without):
                        if a is not None:
                            bad = ~np.isfinite(b)
                            np.testing.assert_array_equal(~np.isfinite(a), bad)
                            np.testing.assert_allclose(a[~bad], w[~bad], rtol=2.0 ** -22,
                                                       atol=1e-6)
                    continue
                for a, b in zip(got, run(x, q, prec="mixed", **kw)):
                    if a is not None:
                        np.testing.assert_allclose(a, b, rtol=2.0 ** -22, atol=1e-6)


def test_batch(gpu_ctx, oracle_mod):
    """Frames of a batch, of different sizes, as the same frames alone."""
    from pycpet_amd import batch, ops

    frames = []
    for i, (shape, N) in enumerate([((3, 1, 7), 65), ((13, 9, 8), 2048), ((5, 5, 5), 1),
                                    ((17, 16, 21), 1023)]):
        x, q = _charges(N, seed=70 + i)
        axes = tuple(np.linspace(-1.0, 0.7 + 0.1 * k, n).astype(np.float32)
                     for k, n in enumerate(shape))
        frames.append({"axes": axes, "x": x, "q": q})
    for kw in ({}, {"want_phi": True}, {"want_E": False, "want_phi": True}):
        for f, (E, phi) in zip(frames, batch.batch_volume(frames, ctx=gpu_ctx, **kw)):
            pts = np.stack(np.meshgrid(*f["axes"], indexing="ij"), -1).reshape(-1, 3)
            _check(pts, f["x"], f["q"], E, phi, oracle_mod)


@pytest.mark.parametrize("kw", [{}, {"want_E": False, "want_phi": True}, {"want_phi": True}],
                         ids=["E", "phi", "both"])
def test_small_frames_are_judged_together(gpu_ctx, oracle_mod, kw):
    """Small frames of a batch: few take the FP64 pair terms; of many, the larger grids are
    interpolated and the smallest, and those with few charges, take the direct batch kernel, bit
    for bit the one asked for by tuning.  refined_points() tells the three apart (all points,
    none, those with cancellation)."""
    from pycpet_amd import batch

    def frame(n, N, seed):
        rng = np.random.default_rng(seed)
        axes = [np.linspace(-0.1 * (n - 1), 0.1 * (n - 1), n).astype(np.float32)] * 3
        return {"axes": axes, "x": rng.uniform(-15, 15, (N, 3)).astype(np.float32),
                "q": rng.normal(0, 0.4, N).astype(np.float32)}

    E = kw.get("want_E", True)
    few = [frame(9, 1000, k) for k in range(20)]
    batch.batch_volume(few, ctx=gpu_ctx, **kw)
    assert gpu_ctx.refined_points() == (20 * 729 if E else 0)

    tiny = [frame(9, 1000, k) for k in range(400)] + [frame(16, 60, k) for k in range(5)]
    got = batch.batch_volume(tiny, ctx=gpu_ctx, **kw)
    assert gpu_ctx.refined_points() < (400 * 729 + 5 * 4096) / 2
    gpu_ctx.set_tuning(4, 2, 0)
    try:
        want = batch.batch_volume(tiny, ctx=gpu_ctx, **kw)
    finally:
        gpu_ctx.set_tuning(4, 0, 0)
    for a, b in zip(got, want):
        for u, v in zip(a, b):
            if u is not None:
                np.testing.assert_array_equal(u, v)

    mixed = [frame(21, 2000, k) for k in range(4)] + [frame(9, 700, 9), frame(16, 191, 10),
                                                      frame(15, 200, 11)]
    got = batch.batch_volume(mixed, ctx=gpu_ctx, **kw)
    assert gpu_ctx.refined_points() == (729 if E else 0)  # 16^3 x 191 has 192 padded charges
    for f, (e, phi) in zip(mixed, got):
        pts = np.stack(np.meshgrid(*f["axes"], indexing="ij"), -1).reshape(-1, 3)
        at = np.unique(np.linspace(0, len(pts) - 1, 80).astype(int))
        pts, e, phi = pts[at], None if e is None else e[at], None if phi is None else phi[at]
        E64, p64 = oracle_mod.field_f64(pts, f["x"], f["q"], want_phi=True)
        r2 = ((pts[:, None].astype(np.float64) - f["x"][None]) ** 2).sum(2)
        for u, v, mag, miss in ((e, E64, r2, 1e-9), (phi, p64, np.sqrt(r2), 1e-10)):
            if u is not None:  # the interpolation's bounds: see test_gpu_fargrid.py
                A = K * (np.abs(f["q"].astype(np.float64)) / mag).sum(1)
                err = np.abs(u - v).reshape(len(pts), -1).max(1)
                assert (err <= 2.0**-24 * np.abs(v).reshape(len(pts), -1).max(1) + miss * A).all()
