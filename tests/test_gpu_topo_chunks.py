"""The chunk-lane form of the 16-wave streamline kernel (four slots x 16
slices' chunks per wave, where few slots are in use) adds the same terms in
the same order as the one-wave walk, which has the slice form only: every
result is equal, with no tolerance."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DIMS = np.array([0.6, 0.5, 0.55], np.float32)


def _frame(N, L, seed):
    from pycpet_amd import workloads as W

    x, q = W.ball_exclusion(N, 20.0, 0.6, 1.5, seed=seed)
    st, it, _ = W.topo_starts(L, DIMS, 0.01, 40, seed=seed + 1, start_seed=seed + 2)
    q[::7] = -0.0          # terms that are zero of either sign
    q[3::11] = 1e-40       # denormal charges
    x[N // 2] = [0.1, -0.2, 0.05]   # a charge inside the box ...
    x[N // 3] = st[0]               # ... and one on a start (r = 0)
    x[N // 5] = [1e-40, 0.0, -0.3]
    return x, q, st, it


def _equal(a, b):
    np.testing.assert_array_equal(a.feats, b.feats)
    np.testing.assert_array_equal(a.steps, b.steps)
    np.testing.assert_array_equal(a.exited, b.exited)


# slices of less than one chunk, of whole chunks, of one more source group, of
# a ragged last chunk; more chunk groups than one pass of the sums in LDS holds
@pytest.mark.parametrize("N,L", [(300, 5), (1023, 3), (1024, 64), (1025, 700), (1089, 255),
                                 (2052, 1), (5003, 2500), (9999, 3300), (21001, 1500)])
def test_chunk_lanes_equal_the_slice_form(gpu_ctx, N, L):
    from pycpet_amd import ops

    x, q, st, it = _frame(N, L, seed=N)
    mu = np.random.default_rng(N).standard_normal((N, 3)).astype(np.float32)
    mu[::5] = -0.0
    try:
        runs = []
        for S in (16, 1):
            gpu_ctx.set_tuning(2, S, 0)
            runs.append([ops.topo(st, it, 0.01, DIMS, x, q, ctx=gpu_ctx),
                         ops.topo(st, it, 0.01, DIMS, x, q, integrator="rk4", ctx=gpu_ctx),
                         ops.topo_dipole(st, it, 0.01, DIMS, x, mu, ctx=gpu_ctx),
                         ops.topo_dipole(st, it, 0.01, DIMS, x, mu, physical=True, ctx=gpu_ctx)])
    finally:
        gpu_ctx.set_tuning(2, 0, 0)
    for a, b in zip(*runs):
        _equal(a, b)


# few workgroups: 64 slots that empty one by one, from the queue and at its end
@pytest.mark.parametrize("G", [1, 3])
def test_chunk_lanes_from_a_queue(gpu_ctx, G):
    from pycpet_amd import ops

    x, q, st, it = _frame(1500, 400, seed=5)
    try:
        gpu_ctx.set_tuning(2, 16, G)
        a = ops.topo(st, it, 0.01, DIMS, x, q, ctx=gpu_ctx)
        gpu_ctx.set_tuning(2, 1, 0)
        b = ops.topo(st, it, 0.01, DIMS, x, q, ctx=gpu_ctx)
    finally:
        gpu_ctx.set_tuning(2, 0, 0)
    _equal(a, b)


def test_chunk_lanes_of_a_batch(gpu_ctx):
    """Frames of different sizes: each frame's chunk groups lie where the
    kernel looks for them."""
    from pycpet_amd import batch, ops

    frames = []
    for i, (N, L) in enumerate([(40, 30), (1024, 7), (3000, 130), (64, 1), (9001, 260),
                                (1025, 65)]):
        x, q, st, it = _frame(N, L, seed=50 + i)
        frames.append({"x": x, "q": q, "starts": st, "n_iter": it, "h": 0.01, "dims": DIMS})
    outs = batch.batch_topo(frames, ctx=gpu_ctx)
    try:
        gpu_ctx.set_tuning(2, 1, 0)
        for f, r in zip(frames, outs):
            _equal(r, ops.topo(f["starts"], f["n_iter"], f["h"], f["dims"], f["x"], f["q"],
                               ctx=gpu_ctx))
    finally:
        gpu_ctx.set_tuning(2, 0, 0)


@pytest.mark.gpu
def test_asked_for_workgroups_are_bounded(gpu_ctx):
    """More workgroups asked for than fit the chip, on so many streamlines that 64 places for
    each would pass 2^31: the results of the library's own choice."""
    import torch

    from pycpet_amd import ops

    L = 2**31 // 63 + 1000
    g = torch.Generator("cuda").manual_seed(1)
    rng = np.random.default_rng(1)
    starts = torch.rand((L, 3), device="cuda", generator=g).sub_(0.5)
    n_iter = torch.ones(L, dtype=torch.int32, device="cuda")
    x = torch.from_numpy((rng.standard_normal((200, 3)) * 9).astype(np.float32)).cuda()
    q = torch.from_numpy(rng.normal(0, 0.4, 200).astype(np.float32)).cuda()
    args = (starts, n_iter, 0.01, np.ones(3, np.float32), x, q)
    want = ops.topo(*args, ctx=gpu_ctx).feats
    gpu_ctx.set_tuning(2, 16, L)
    try:
        got = ops.topo(*args, ctx=gpu_ctx).feats
    finally:
        gpu_ctx.set_tuning(2, 0, 0)
    assert torch.equal(got.view(torch.int64), want.view(torch.int64))


# both sides of the lines between the forms of the 16-wave kernel: one group of charges a
# slice, too few records or too many streamlines for the chunk-lane form, two workgroups a CU
@pytest.mark.parametrize("N,L,G", [(64, 300, 0), (65, 300, 0), (149, 200, 0), (150, 200, 0),
                                   (299, 200, 0), (300, 200, 0), (460, 30000, 0),
                                   (470, 30000, 0), (700, 20000, 300)])
def test_forms_are_equal(gpu_ctx, N, L, G):
    from pycpet_amd import batch, ops

    x, q, st, it = _frame(N, L, seed=N + L)
    it = np.minimum(it, 6)
    mu = np.random.default_rng(N).standard_normal((N, 3)).astype(np.float32)
    frames = [{"x": x[k:], "q": q[k:], "starts": st[k::2], "n_iter": it[k::2], "h": 0.01,
               "dims": DIMS} for k in (0, 1)]
    try:
        runs = []
        for shape in ((16, G), (1, 0)):
            for kind in (2, 3):
                gpu_ctx.set_tuning(kind, *shape)
            runs.append([ops.topo(st, it, 0.01, DIMS, x, q, ctx=gpu_ctx),
                         ops.topo(st, it, 0.01, DIMS, x, q, integrator="rk4", ctx=gpu_ctx),
                         ops.topo_dipole(st, it, 0.01, DIMS, x, mu, ctx=gpu_ctx),
                         *batch.batch_topo(frames, ctx=gpu_ctx)])
    finally:
        for kind in (2, 3):
            gpu_ctx.set_tuning(kind, 0, 0)
    for a, b in zip(*runs):
        _equal(a, b)
