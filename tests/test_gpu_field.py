"""GPU parity of the field / potential kernels against the FP64 oracle.

Tolerance (stated once): pointwise relative error
    |E_gpu(p) - E_64(p)| / max(|E_64(p)|, 1e-3 * RMS_p |E_64|) <= 1e-5
for E (vector norm) and phi, with E_64 the FP64 oracle on the same float32
inputs.  The denominator floor keeps points where the field nearly cancels
from turning FP32 rounding into unbounded relative error.
"""
import numpy as np
import pytest

from conftest import GOLDEN

pytestmark = pytest.mark.gpu

TOL = 1e-5


def rel_err(a, b, floor_frac=1e-3):
    a = np.asarray(a, float)
    b = np.asarray(b, float)
    if b.ndim == 1:
        a, b = a[:, None], b[:, None]
    nb = np.linalg.norm(b, axis=1)
    d = np.linalg.norm(a - b, axis=1)
    rms = np.sqrt(np.mean(nb ** 2))
    return float((d / np.maximum(nb, floor_frac * rms)).max()), float(np.sqrt(np.mean(d ** 2)) / rms)


def mesh(axes):
    return np.stack(np.meshgrid(*axes, indexing="ij"), -1).reshape(-1, 3).astype(np.float32)


def test_volume_2k_grid_vs_oracle(gpu_ctx, oracle_mod):
    from pycpet_amd import ops, workloads as W

    c = W.volume_2k()
    print(f"case volume_2k N={c.N} M={c.M}", flush=True)
    E, phi = ops.field_grid(*c.axes, c.x, c.q, want_E=True, want_phi=True, ctx=gpu_ctx)
    E64, phi64 = oracle_mod.field_f64(mesh(c.axes), c.x, c.q, want_phi=True)
    assert rel_err(E, E64)[0] <= TOL
    assert rel_err(phi, phi64)[0] <= TOL


def test_points_path_matches_grid_path(gpu_ctx):
    from pycpet_amd import ops, workloads as W

    c = W.volume_2k()
    Eg, pg = ops.field_grid(*c.axes, c.x, c.q, want_phi=True, ctx=gpu_ctx)
    Ep, pp = ops.field_points(mesh(c.axes), c.x, c.q, want_phi=True, ctx=gpu_ctx)
    assert rel_err(Ep, Eg)[0] < 1e-6
    assert rel_err(pp, pg)[0] < 1e-6


def test_volume_30k_precision_modes(gpu_ctx, oracle_mod):
    """Clustered 30k-charge case (net -3 e): every precision mode vs FP64 on
    a seeded 3,000-point sample of the full 101^3 grid.  The default (auto)
    and the compensated/mixed/FP64 modes meet the bound for E and phi; the
    all-FP32 modes meet it for E only (phi cancels between charges of both
    signs), and naive FP32 is reported for comparison."""
    from pycpet_amd import ops, workloads as W

    c = W.volume_30k()
    print(f"case volume_30k N={c.N} M={c.M}", flush=True)
    pts = mesh(c.axes)
    idx = np.random.default_rng(0).choice(pts.shape[0], 3000, replace=False)
    E64, phi64 = oracle_mod.field_f64(pts[idx], c.x, c.q, want_phi=True)
    errs = {}
    for prec in ("auto", "tiled", "kahan", "naive", "mixed", "f64"):
        E, phi = ops.field_grid(*c.axes, c.x, c.q, want_phi=True, prec=prec,
                                out_f64=True, ctx=gpu_ctx)
        errs[prec] = (rel_err(E[idx], E64), rel_err(phi[idx], phi64))
        print(prec, errs[prec], flush=True)
    for prec in ("auto", "mixed", "f64"):
        assert errs[prec][0][0] <= TOL and errs[prec][1][0] <= TOL, (prec, errs[prec])
    for prec in ("tiled", "kahan"):
        assert errs[prec][0][0] <= TOL, (prec, errs[prec])
    assert errs["mixed"][0][0] < 1e-9 and errs["mixed"][1][0] < 1e-9
    assert errs["f64"][0][0] < 1e-11 and errs["f64"][1][0] < 1e-11
    # float32 outputs of the default mode
    E32, p32 = ops.field_grid(*c.axes, c.x, c.q, want_phi=True, ctx=gpu_ctx)
    assert rel_err(E32[idx], E64)[0] <= TOL and rel_err(p32[idx], phi64)[0] <= TOL


def test_reference_golden_vectors(gpu_ctx):
    from pycpet_amd import ops

    g = np.load(GOLDEN / "ref_volume_500.npz")
    E, phi = ops.field_grid(g["ax"], g["ay"], g["az"], g["x"], g["q"], want_phi=True,
                            ctx=gpu_ctx)
    assert rel_err(E, g["E"])[0] < 5e-5  # reference is FP32 -ffast-math
    assert rel_err(phi, g["phi"])[0] < 5e-5
    f = np.load(GOLDEN / "ref_volume_floor.npz")
    E, _ = ops.field_grid(f["ax"], f["ay"], f["az"], f["x"], f["q"], ctx=gpu_ctx)
    assert rel_err(E, f["E"])[0] < 5e-5


def test_dropin_entry_points(gpu_ctx, oracle_mod):
    from pycpet_amd.c_ops import Math_ops

    g = np.load(GOLDEN / "ref_volume_500.npz")
    m = Math_ops()
    pts = mesh([g["ax"], g["ay"], g["az"]])
    E = m.compute_looped_field(pts, g["x"], g["q"].reshape(-1, 1))
    assert E.dtype == np.float32 and E.shape == pts.shape
    E64, phi64 = oracle_mod.field_f64(pts, g["x"], g["q"], want_phi=True)
    assert rel_err(E, E64)[0] <= TOL
    esp = m.calc_esp_base(pts[7], g["x"], g["q"])
    assert esp.shape == (1,) and abs(esp[0] - phi64[7]) <= TOL * abs(phi64[7])
    pf = m.calc_field(np.zeros(3, np.float32), g["x"], g["q"])
    np.testing.assert_allclose(pf, g["point_field"], rtol=5e-5, atol=1e-6)
    Eb = m.calc_field_base(np.zeros(3, np.float32), g["x"], g["q"])
    np.testing.assert_allclose(Eb, pf, rtol=1e-6)


def test_compute_batched_field_through_reference_binding(gpu_ctx, oracle_mod):
    """compute_batched_field bound with the reference's argtypes (ndpointer
    float32, CPET/utils/c_ops.py:140-149) equals the unsoftened FP64 field
    and, within its FP32 rounding, the reference C of the same name."""
    import ctypes

    from pycpet_amd import _native as nat
    from pycpet_amd.c_ops import Math_ops
    from test_abi import _bind_like_reference

    g = np.load(GOLDEN / "ref_volume_500.npz")
    pts = mesh([g["ax"], g["ay"], g["az"]])
    lib, _ = _bind_like_reference(nat.LIB_PATH)
    E = np.zeros_like(pts)
    x = np.ascontiguousarray(g["x"], np.float32)
    q = np.ascontiguousarray(g["q"], np.float32).ravel()
    lib.compute_batched_field(pts.shape[0], 100, q.size, pts, x, q, E)
    E64, _ = oracle_mod.field_f64(pts, x, q, soften=False)
    assert rel_err(E, E64)[0] <= TOL
    Eb = Math_ops().compute_batch_field(pts, x, q.reshape(-1, 1), 37)
    np.testing.assert_array_equal(Eb, E)  # the chunk length changes nothing
    if oracle_mod.REF_SO.exists():
        ref = ctypes.CDLL(str(oracle_mod.REF_SO))
        ref.compute_batched_field.restype = None
        Er = np.zeros_like(pts)
        P = ctypes.c_void_p
        ref.compute_batched_field(ctypes.c_int(pts.shape[0]), ctypes.c_int(100),
                                  ctypes.c_int(q.size), pts.ctypes.data_as(P),
                                  x.ctypes.data_as(P), q.ctypes.data_as(P), Er.ctypes.data_as(P))
        assert rel_err(E, Er)[0] < 5e-5  # the reference is FP32 -ffast-math
    assert nat.load().compute_batched_field(4, 0, q.size, pts.ctypes.data, x.ctypes.data,
                                            q.ctypes.data, E.ctypes.data) == nat.CPET_ERR_ARG


def test_edge_cases(gpu_ctx, oracle_mod):
    from pycpet_amd import ops
    from pycpet_amd._native import CpetError

    rng = np.random.default_rng(1)
    # one charge, one point; ragged charge counts around the 64-charge tile
    for N in (1, 63, 64, 65, 130):
        x = rng.uniform(-4, 4, (N, 3)).astype(np.float32)
        q = rng.normal(0, 0.5, N).astype(np.float32)
        for axes in ([np.array([0.1], np.float32)] * 3,
                     [np.linspace(-1, 1, 7, dtype=np.float32), np.linspace(-1, 1, 3, dtype=np.float32),
                      np.linspace(-1, 1, 5, dtype=np.float32)]):
            E, phi = ops.field_grid(*axes, x, q, want_phi=True, ctx=gpu_ctx)
            E64, p64 = oracle_mod.field_f64(mesh(axes), x, q, want_phi=True)
            assert rel_err(E, E64)[0] <= TOL and rel_err(phi, p64)[0] <= TOL, N
    # a charge exactly on a grid point: phi is +-inf like 1/sqrt(0); E floored
    x = np.array([[0.0, 0.0, 0.0], [2.0, 1.0, 0.5]], np.float32)
    q = np.array([0.5, -0.3], np.float32)
    axes = [np.array([-0.5, 0.0, 0.5], np.float32)] * 3
    E, phi = ops.field_grid(*axes, x, q, want_phi=True, ctx=gpu_ctx)
    c = 13  # the (0,0,0) grid point
    assert np.isposinf(phi[c]) and np.all(np.isfinite(E))
    # invalid sizes are rejected with an error, not a crash
    with pytest.raises(CpetError):
        ops.field_points(np.zeros((0, 3), np.float32), x, q, ctx=gpu_ctx)
    with pytest.raises(CpetError):
        ops.field_grid(np.zeros(0, np.float32), axes[1], axes[2], x, q, ctx=gpu_ctx)


def _random_grids():
    """Ten seeded frames across the shapes the grid kernels branch on:
    z-lines of 1 to 101 points (points per lane), single points and
    single lines, 1 to 3,000 charges (64-charge tiles, the charge split
    over workgroups, the padding), anisotropic boxes of half-widths
    0.3-2.5 A, charges anywhere around the grid or at least 0.5 or 2 A
    outside it."""
    from pycpet_amd import workloads as W

    rng = np.random.default_rng(2027)
    shapes = [(1, 1, 1), (1, 1, 101), (2, 3, 7), (13, 1, 40), (7, 21, 41), (21, 21, 21),
              (3, 64, 65), (40, 13, 3), (65, 9, 64), (11, 17, 101)]
    counts = [1, 3, 64, 65, 257, 1000, 3000, 130, 2048, 511]
    frames = []
    for k, (shape, N) in enumerate(zip(shapes, counts)):
        half = rng.uniform(0.3, 2.5, 3)
        axes = [np.linspace(-half[i], half[i], shape[i]).astype(np.float32) if shape[i] > 1
                else np.array([rng.uniform(-0.5, 0.5)], np.float32) for i in range(3)]
        excl = float(rng.choice([0.0, 0.5, 2.0]))
        x, q = W.ball_exclusion(N, float(half.max()) + excl + 10.0, float(half.max()), excl,
                                seed=900 + k)
        if N == 1:  # the mean-free charge of one would be 0
            q = np.array([0.9], np.float32)
        frames.append({"axes": axes, "x": x, "q": q})
    return frames


def test_random_grids_vs_oracle(gpu_ctx, oracle_mod):
    """E and phi of ten random frames in the default (auto) precision, each
    alone and all ten as one batch, against the FP64 oracle within the
    pointwise bound above."""
    from pycpet_amd import batch, ops

    frames = _random_grids()
    refs = []
    for i, f in enumerate(frames):
        label = f"random grid {i}: shape {tuple(len(a) for a in f['axes'])} N={len(f['q'])}"
        print(label, flush=True)
        E64, p64 = oracle_mod.field_f64(mesh(f["axes"]), f["x"], f["q"], want_phi=True)
        refs.append((E64, p64))
        E, phi = ops.field_grid(*f["axes"], f["x"], f["q"], want_phi=True, ctx=gpu_ctx)
        eE, eP = rel_err(E, E64)[0], rel_err(phi, p64)[0]
        print(f"{label}: E {eE:.2e} phi {eP:.2e}", flush=True)
        assert eE <= TOL and eP <= TOL
    print("random grids batched", flush=True)
    for (E, phi), (E64, p64) in zip(batch.batch_volume(frames, want_phi=True, ctx=gpu_ctx), refs):
        assert rel_err(E, E64)[0] <= TOL and rel_err(phi, p64)[0] <= TOL


def test_floor_near_grid_points(gpu_ctx, oracle_mod):
    """The volume field's r^2 >= 1e-6 floor (math_module.c:405-451) with E
    alone: the grid kernel skips the floor only when no charge is within
    1.01e-3 A of a grid point, so results must match the floored oracle both
    when a charge sits on or next to a grid point and when none does."""
    from pycpet_amd import ops

    rng = np.random.default_rng(5)
    axes = [np.linspace(-1, 1, 21, dtype=np.float32)] * 3
    far = rng.uniform(-3, 3, (200, 3)).astype(np.float32)
    q = rng.normal(0, 0.5, 201).astype(np.float32)
    g = np.array([0.1, 0.2, -0.3], np.float32)  # a grid point (step 0.1)
    for offset in (0.0, 5e-4, 9.9e-4, 1.2e-3, 2e-3):
        x = np.concatenate([far, (g + np.float32(offset) * np.array([1, 0, 0], np.float32))[None]])
        E, _ = ops.field_grid(*axes, x, q, ctx=gpu_ctx)
        E64, _ = oracle_mod.field_f64(mesh(axes), x, q)
        assert np.all(np.isfinite(E)), offset
        assert rel_err(E, E64)[0] <= TOL, offset
    # no charge near the grid: the unfloored sum equals the floored oracle
    x = np.concatenate([far, np.array([[0.15, 0.25, -0.35]], np.float32)])
    E, _ = ops.field_grid(*axes, x, q, ctx=gpu_ctx)
    E64, _ = oracle_mod.field_f64(mesh(axes), x, q)
    assert rel_err(E, E64)[0] <= TOL


def test_charge_split_invariance(gpu_ctx):
    """Splitting the charge sum over workgroups only regroups FP64 partials."""
    from pycpet_amd import ops, workloads as W

    c = W.volume_2k()
    out = []
    for splits in (1, 3, 16):
        gpu_ctx.set_tuning(0, 4, splits)
        E, phi = ops.field_grid(*c.axes, c.x, c.q, want_phi=True, out_f64=True, ctx=gpu_ctx)
        out.append((E, phi))
    gpu_ctx.set_tuning(0, 0, 0)
    for E, phi in out[1:]:
        np.testing.assert_allclose(E, out[0][0], rtol=1e-12, atol=1e-12)
        np.testing.assert_allclose(phi, out[0][1], rtol=1e-12, atol=1e-12)


def test_points_per_lane_invariance(gpu_ctx):
    from pycpet_amd import ops, workloads as W

    c = W.volume_2k()
    ref = None
    for k in (1, 2, 3, 4, 6, 8):
        gpu_ctx.set_tuning(0, k, 1)
        E, _ = ops.field_grid(*c.axes, c.x, c.q, out_f64=True, ctx=gpu_ctx)
        if ref is None:
            ref = E
        else:
            np.testing.assert_array_equal(E, ref)  # same charge tiling: bitwise
    gpu_ctx.set_tuning(0, 0, 0)


def test_device_tensor_path(gpu_ctx):
    import torch

    from pycpet_amd import ops, workloads as W

    c = W.volume_2k()
    En, pn = ops.field_grid(*c.axes, c.x, c.q, want_phi=True, ctx=gpu_ctx)
    dev = torch.device("cuda:0")
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)
    Et, pt = ops.field_grid(*(t(a) for a in c.axes), t(c.x), t(c.q), want_phi=True, ctx=gpu_ctx)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(Et.cpu().numpy(), En)
    np.testing.assert_array_equal(pt.cpu().numpy(), pn)


def _cancelling_frame():
    """771 charges at >= 1.5 A from a +-0.6 A box holding a 2,535-point grid:
    at some points the field cancels to a few % of its RMS, where FP32 pair
    rounding alone (even summed exactly) exceeds 1e-5 relative."""
    from pycpet_amd import workloads as W

    x, q = W.ball_exclusion(771, 12.0, 0.6, 1.5, seed=100)
    ax = np.linspace(-0.5, 0.5, 13).astype(np.float32)
    ay = np.linspace(-0.3, 0.4, 15).astype(np.float32)
    return x, q, (ax, ay, ax)


def test_auto_recomputes_cancelling_points(gpu_ctx, oracle_mod):
    """auto = FP32 tiles plus an FP64 recompute of the points whose error
    estimate u * sum|q|/r^2 exceeds 6e-6 |E|: the bound holds pointwise even
    where the plain FP32 tiling (prec="tiled") is allowed to miss it, and the
    recomputed points equal the all-"mixed" result to FP64 rounding."""
    from pycpet_amd import ops

    x, q, axes = _cancelling_frame()
    pts = mesh(axes)
    E64, _ = oracle_mod.field_f64(pts, x, q, want_phi=True)
    for grid in (True, False):
        run = (lambda **kw: ops.field_grid(*axes, x, q, out_f64=True, ctx=gpu_ctx, **kw)[0]) \
            if grid else (lambda **kw: ops.field_points(pts, x, q, out_f64=True, ctx=gpu_ctx,
                                                        **kw)[0])
        E = run()
        n_fixed = gpu_ctx.refined_points()
        Et = run(prec="tiled")
        assert gpu_ctx.refined_points() == 0
        Em = run(prec="mixed")
        err_auto, err_tiled = rel_err(E, E64, 0.0)[0], rel_err(Et, E64, 0.0)[0]
        print(f"grid={grid} refined {n_fixed}/{len(pts)} err auto {err_auto:.2e} "
              f"tiled {err_tiled:.2e}", flush=True)
        assert 0 < n_fixed < len(pts)
        assert err_auto <= TOL
        fixed = np.any(E != Et, axis=1)
        assert fixed.sum() <= n_fixed
        assert rel_err(E[fixed], Em[fixed], 0.0)[0] < 1e-11  # summation order only
        # E together with phi (volume semantics) takes the same check
        E2, phi2 = ops.field_grid(*axes, x, q, want_phi=True, out_f64=True, ctx=gpu_ctx) \
            if grid else ops.field_points(pts, x, q, want_phi=True, out_f64=True, ctx=gpu_ctx)
        assert gpu_ctx.refined_points() == n_fixed
        np.testing.assert_array_equal(E2, E)


def _adversarial(name):
    """Charge layouts whose FP32 roundings correlate: (axes, x, q)."""
    rng = np.random.default_rng(3)
    g = np.linspace(-2.5, 2.5, 9).astype(np.float32)
    if name == "rocksalt":  # 10^3 lattice of alternating +-1 e, 2.82 A spacing
        idx = np.stack(np.meshgrid(*[np.arange(10)] * 3, indexing="ij"), -1).reshape(-1, 3)
        x = ((idx - 4.5) * 2.82 + 0.37).astype(np.float32)
        q = np.where(idx.sum(1) % 2 == 0, 1.0, -1.0).astype(np.float32)
        return (g, g, g), x, q
    if name == "shell":  # 3,000 equal charges on a 9 A sphere: E ~ 0 inside
        m = 3000
        k = np.arange(m) + 0.5
        phi = np.arccos(1 - 2 * k / m)
        th = np.pi * (1 + 5 ** 0.5) * k
        x = 9.0 * np.stack([np.cos(th) * np.sin(phi), np.sin(th) * np.sin(phi), np.cos(phi)], 1)
        return (g, g, g), x.astype(np.float32), np.full(m, 0.3, np.float32)
    if name.startswith("mirror"):  # same-sign clusters on both sides of a field zero
        mult = int(name[6:])
        c1, c2 = np.array([3.0, 0.0, 0.0]), np.array([-3.0, 0.0, 0.0])
        jit = 0.05 if mult < 64 else 0.0
        s1 = c1 + jit * rng.standard_normal((64 // mult, 3))
        s2 = c2 + jit * rng.standard_normal((64 // mult, 3))
        x = np.concatenate([np.repeat(s1, mult, 0), np.repeat(s2, mult, 0)]).astype(np.float32)
        q = np.concatenate([np.full(64, 0.37), np.full(64, 0.37 * 1.1)]).astype(np.float32)
        ax = np.linspace(0.0715 - 0.03, 0.0715 + 0.03, 61).astype(np.float32)
        ay = np.linspace(-0.2, 0.2, 5).astype(np.float32)
        return (ax, ay, ay), x, q
    from pycpet_amd import workloads as W

    x, q = W.clustered(600, 10, 20.0, 1.5, -3.0, 5)
    return (g, g, g), x, q


@pytest.mark.parametrize("name", ["rocksalt", "shell", "mirror1", "mirror2", "mirror4",
                                  "mirror16", "clustered"])
def test_auto_precision_adversarial(gpu_ctx, oracle_mod, name):
    """The auto mode's accepted FP32 points stay within 1e-5 of |E| (strict,
    no RMS floor) on layouts built to correlate rounding: a rock-salt
    lattice, a shell of equal charges, same-sign clusters (up to 16
    coincident copies of a charge) on both sides of a field zero, and a
    clustered frame.  Points whose FP64 estimate u A / |E| is within 10 % of
    the check's 4e-6 are certainly unflagged and are held to the strict
    bound; every point meets the usual 1e-5 pointwise metric."""
    from pycpet_amd import ops

    axes, x, q = _adversarial(name)
    print(f"case adversarial {name} N={q.size} M={np.prod([a.size for a in axes])}", flush=True)
    E, _ = ops.field_grid(*axes, x, q, ctx=gpu_ctx)
    refined = gpu_ctx.refined_points()
    pts = mesh(axes)
    E64, _ = oracle_mod.field_f64(pts, x, q)
    d = pts[:, None, :].astype(np.float64) - x[None].astype(np.float64)
    A = 14.3996451 * (np.abs(q.astype(np.float64))[None] / (d ** 2).sum(2)).sum(1)
    nE = np.linalg.norm(E64, axis=1)
    err = np.linalg.norm(E - E64, axis=1)
    sure = 2.0 ** -24 * A <= 0.9 * 4e-6 * nE
    print(f"{name}: refined {refined}, strict points {sure.sum()}, "
          f"max rel {(err[sure] / nE[sure]).max() if sure.any() else 0:.2e}", flush=True)
    assert sure.any() or refined == pts.shape[0]  # a shell cancels everywhere: all refined
    assert (err[sure] <= 1e-5 * nE[sure]).all()
    assert rel_err(E, E64)[0] <= TOL


def _check_recompute(pts, x, q, E, refined, oracle_mod):
    """E within the auto mode's bounds, and as many points recomputed as its check's line allows:
    all whose estimate u A / |E| is 10 % above 4e-6, none that is 10 % below."""
    E64, _ = oracle_mod.field_f64(pts, x, q)
    nE = np.linalg.norm(E64, axis=1)
    err = np.linalg.norm(E - E64, axis=1)
    A = np.empty(len(pts))
    for a in range(0, len(pts), 2000):
        d = pts[a:a + 2000, None, :].astype(np.float64) - x[None].astype(np.float64)
        A[a:a + 2000] = 14.3996451 * (np.abs(q.astype(np.float64))[None] / (d ** 2).sum(2)).sum(1)
    sure = 2.0 ** -24 * A <= 0.9 * 4e-6 * nE
    flagged = 2.0 ** -24 * A >= 1.1 * 4e-6 * nE
    print(f"refined {refined} of {len(pts)}, flagged {flagged.sum()}, sure {sure.sum()}", flush=True)
    assert flagged.sum() <= refined <= len(pts) - sure.sum()
    assert (err[sure] <= 1e-5 * nE[sure]).all()
    assert rel_err(E, E64)[0] <= TOL


@pytest.mark.parametrize("out_f64", [False, True])
@pytest.mark.parametrize("name", ["rocksalt", "shell", "mirror1", "mirror16", "clustered"])
def test_auto_precision_adversarial_direct(gpu_ctx, oracle_mod, name, out_f64):
    """The layouts of test_auto_precision_adversarial on the FP32 tiles with their check, which
    small float32 grids take when a launch shape is asked for."""
    from pycpet_amd import ops

    axes, x, q = _adversarial(name)
    gpu_ctx.set_tuning(0, 2, 0)
    try:
        E, _ = ops.field_grid(*axes, x, q, out_f64=out_f64, ctx=gpu_ctx)
        refined = gpu_ctx.refined_points()
    finally:
        gpu_ctx.set_tuning(0, 0, 0)
    _check_recompute(mesh(axes), x, q, E, refined, oracle_mod)


def test_default_grids_on_the_direct_kernel(gpu_ctx, oracle_mod):
    """A float32 grid too large for the FP64 pair terms and, with an axis of five values, not
    interpolated: the direct kernel by default, some points recomputed and others not."""
    from pycpet_amd import ops

    x, q, _ = _cancelling_frame()
    axes = (np.linspace(-0.5, 0.5, 5).astype(np.float32),
            np.linspace(-0.3, 0.4, 130).astype(np.float32),
            np.linspace(-0.5, 0.5, 110).astype(np.float32))
    E, _ = ops.field_grid(*axes, x, q, ctx=gpu_ctx)
    refined = gpu_ctx.refined_points()
    assert 0 < refined < 5 * 130 * 110
    _check_recompute(mesh(axes), x, q, E, refined, oracle_mod)
