"""Learned CG preconditioner on the GPU against its CPU restatement.

Tolerances: the GPU stores activations and weights in bfloat16 (8-bit
significand) and accumulates in FP32.  The restatement applies the same
bf16 roundings to weights, inputs and activations, so the forward output
agrees to 2e-2 of its largest value (a rounding tie can still fall the
other way on an FP32 difference).  The backward kernels also round the
layer gradients dy, dz to bf16, which the FP64 restatement does not, so
each parameter group's gradient agrees to 5e-2 in norm.
"""
import numpy as np
import pytest

from oracle import lpc_oracle as lo
from rsdft_develop_amd import lpc, systems

pytestmark = pytest.mark.gpu

SHAPE = (20, 14, 12)  # n1, n2, n3 (x fastest)


@pytest.fixture(scope="module")
def setup():
    from rsdft_develop_amd import gpu

    rng = np.random.default_rng(11)
    n1, n2, n3 = SHAPE
    aa = np.diag([10.0, 7.5, 6.8])
    ctx = gpu.Context()
    ctx.set_grid(SHAPE, aa, 6)
    N = n1 * n2 * n3
    v = 0.3 * np.sin(np.arange(N) * 0.01) + 0.1 * rng.standard_normal(N)
    ctx.set_vloc(v)
    ctx.lpc_set_potential(v)
    vn = ((v - v.mean()) / (np.sqrt(np.mean((v - v.mean()) ** 2)) + 1e-30)).astype(np.float32)
    p = lpc.init_params(5)
    d = lpc.unpack(p)
    d["W3"] = rng.standard_normal(d["W3"].shape) * 0.2
    d["b1"] = rng.standard_normal(16) * 0.1
    d["b3"] = np.array([0.05])
    p = lpc.pack(d)
    ctx.lpc_set_params(p)
    return ctx, p, vn, rng


def _grid(a):
    n1, n2, n3 = SHAPE
    return np.asarray(a).reshape(n3, n2, n1)


def test_params_round_trip(setup):
    ctx, p, _, _ = setup
    np.testing.assert_array_equal(ctx.lpc_get_params(), p)
    assert ctx.lpc_param_count() == lpc.NPARAM == 8241


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_forward_matches_restatement(setup, dtype):
    from rsdft_develop_amd import hip

    ctx, p, vn, rng = setup
    N = int(np.prod(SHAPE))
    nb = 3
    g = rng.standard_normal((N, nb)) * np.array([1.0, 1e-3, 40.0])
    dg = hip.DeviceArray.from_numpy(g, dtype=dtype)
    dp = hip.DeviceArray((N, nb), dtype=dtype)
    ctx.lpc_apply_device(dg.ptr, dp.ptr, N, nb, dtype=dtype)
    ctx.synchronize()
    got = dp.to_numpy().astype(np.float64)
    gq = dg.to_numpy().astype(np.float64)
    op = lpc.to_oracle(p)
    for b in range(nb):
        want, c = lo.forward(op, _grid(gq[:, b]), _grid(vn), bf16_storage=True)
        y_got = got[:, b] / c["s"]
        y_want = c["y"].reshape(-1)
        scale = np.abs(y_want).max()
        assert np.abs(y_got - y_want).max() < 2e-2 * scale, b
        assert np.mean(np.abs(y_got - y_want)) < 2e-3 * scale, b
    dg.free()
    dp.free()


def test_gradients_match_restatement(setup):
    from rsdft_develop_amd import hip

    ctx, p, vn, rng = setup
    N = int(np.prod(SHAPE))
    ns = 2
    g = rng.standard_normal((N, ns)).astype(np.float32)
    t = (0.5 * g + 0.2 * rng.standard_normal((N, ns))).astype(np.float32)
    dg = hip.DeviceArray.from_numpy(g)
    dt = hip.DeviceArray.from_numpy(t)
    loss, grads = ctx.lpc_train_step(dg.ptr, dt.ptr, ns, lr=0.0, want_grads=True, kappa=1.7)
    op = lpc.to_oracle(p)
    L_sum, G_sum = 0.0, None
    for b in range(ns):
        L, G = lo.loss_and_grads(op, _grid(g[:, b]), _grid(vn), _grid(t[:, b]), bf16_storage=True, kappa=1.7)
        L_sum += L / ns
        G = {k: v / ns for k, v in G.items()}
        G_sum = G if G_sum is None else {k: G_sum[k] + G[k] for k in G}
    assert loss == pytest.approx(L_sum, rel=2e-3)
    gd = lpc.unpack(grads)
    for k in ("W1", "b1", "W2", "b2", "W3", "b3"):
        want = G_sum[k].reshape(gd[k].shape)
        err = np.linalg.norm(gd[k] - want) / (np.linalg.norm(want) + 1e-30)
        assert err < 5e-2, (k, err)
    dg.free()
    dt.free()


def test_output_is_scale_equivariant(setup):
    from rsdft_develop_amd import hip

    ctx, p, vn, rng = setup
    N = int(np.prod(SHAPE))
    g = rng.standard_normal((N, 1))
    out = []
    for c in (1.0, 64.0):
        dg = hip.DeviceArray.from_numpy(c * g)
        dp = hip.DeviceArray((N, 1))
        ctx.lpc_apply_device(dg.ptr, dp.ptr, N, 1)
        ctx.synchronize()
        out.append(dp.to_numpy()[:, 0])
        dg.free()
        dp.free()
    # a power-of-two scale leaves every bf16 rounding unchanged
    np.testing.assert_allclose(out[1], 64.0 * out[0], rtol=1e-6, atol=0)


def test_training_lowers_the_loss(setup):
    from rsdft_develop_amd import hip

    ctx, p, vn, rng = setup
    N = int(np.prod(SHAPE))
    ns = 4
    g = rng.standard_normal((N, ns)).astype(np.float32)
    dg = hip.DeviceArray.from_numpy(g)
    dt = hip.DeviceArray((N, ns), dtype=np.float32)
    ctx.lpc_target_device(dg.ptr, dt.ptr, ns, steps=30, shift=0.5)
    ctx.lpc_set_params(p)
    ctx.lpc_reset_optimizer()
    first, _ = ctx.lpc_train_step(dg.ptr, dt.ptr, ns, lr=0.0)
    for _ in range(40):
        ctx.lpc_train_step(dg.ptr, dt.ptr, ns, lr=3e-3)
    last, _ = ctx.lpc_train_step(dg.ptr, dt.ptr, ns, lr=0.0)
    assert last < 0.7 * first, (first, last)
    ctx.lpc_set_params(p)
    dg.free()
    dt.free()


def test_target_solves_the_shifted_operator(setup):
    """t = A^-1 g for A = -1/2 lap_7 + (V - min V + shift): check A t = g."""
    from rsdft_develop_amd import gpu, hip

    ctx, p, vn, rng = setup
    n1, n2, n3 = SHAPE
    N = n1 * n2 * n3
    g = rng.standard_normal((N, 1)).astype(np.float32)
    dg = hip.DeviceArray.from_numpy(g)
    dt = hip.DeviceArray((N, 1), dtype=np.float32)
    ctx.lpc_target_device(dg.ptr, dt.ptr, 1, steps=300, shift=0.5, vweight=1.0)
    t = _grid(dt.to_numpy()[:, 0].astype(np.float64))
    h = np.array([10.0 / n1, 7.5 / n2, 6.8 / n3])
    lap = sum((np.roll(t, 1, ax) + np.roll(t, -1, ax) - 2 * t) / hh ** 2 for ax, hh in zip((2, 1, 0), h))
    V = _grid(ctx.get_field(gpu.FIELD_VLOC))
    r = -0.5 * lap + (V - V.min() + 0.5) * t - _grid(g[:, 0])
    assert np.linalg.norm(r) < 1e-3 * np.linalg.norm(g)
    dg.free()
    dt.free()


def test_cg_with_learned_preconditioner_lowers_energies():
    from rsdft_develop_amd import gpu

    cell = systems.silicon_supercell(1, ngrid_per_cell=24, nband=12, displacement=0.05, seed=4)
    v = systems.model_vloc(cell)
    ctx = gpu.Context().setup(cell, v)
    ctx.lpc_set_params(lpc.init_params(0))
    ctx.lpc_set_potential(v)
    ctx.alloc_bands(cell.nband)
    ctx.upload_bands(systems.random_bands(cell.npoints, cell.nband, seed=1))
    ctx.gram_schmidt()
    e0 = ctx.subspace_diag()
    for prec in (64, 32):
        e1, res = ctx.conjugate_gradient(ncg=4, pc_kind=5, mloop=3, precision=prec)
        assert np.all(np.isfinite(e1)) and np.all(np.isfinite(res))
        assert np.all(e1 <= e0 + (1e-10 if prec == 64 else 1e-5))
        e0 = e1
    assert ctx.lpc_fallbacks() >= 0


def test_hybrid_with_a_silent_network_is_hprsdft():
    """pc_kind 6 with a network whose output is zero is hprsdft scaled by
    the hybrid factor; CG is invariant to a positive scale of its
    preconditioner, so both factors give the pc_kind 4 result (to the
    rounding of the recomputed <Pg, g>)."""
    from rsdft_develop_amd import gpu

    cell = systems.silicon_supercell(1, ngrid_per_cell=24, nband=12, displacement=0.05, seed=4)
    v = systems.model_vloc(cell)
    ctx = gpu.Context().setup(cell, v)
    d = lpc.unpack(lpc.init_params(0))
    d["W3"] = np.zeros_like(d["W3"])
    d["b3"] = np.zeros_like(d["b3"])
    ctx.lpc_set_params(lpc.pack(d))
    ctx.lpc_set_potential(v)
    ctx.alloc_bands(cell.nband)
    u0 = systems.random_bands(cell.npoints, cell.nband, seed=1)
    out = {}
    for key, pc, scale in (("hprsdft", 4, None), ("hybrid1", 6, 1.0), ("hybrid2", 6, 2.5)):
        if scale is not None:
            ctx.lpc_set_hybrid_scale(scale)
        ctx.upload_bands(u0)
        ctx.gram_schmidt()
        ctx.subspace_diag()
        out[key] = ctx.conjugate_gradient(ncg=4, pc_kind=pc, mloop=3)[0], ctx.download_bands()
    for key in ("hybrid1", "hybrid2"):
        np.testing.assert_allclose(out[key][0], out["hprsdft"][0], rtol=0, atol=1e-10)
        assert np.abs(out[key][1] - out["hprsdft"][1]).max() < 1e-8 * np.abs(out["hprsdft"][1]).max()
    assert ctx.lpc_fallbacks() == 0


def test_reject_limit_skips_a_rejected_network():
    """A silent network (P g = 0) fails the descent check in every block.
    With a rejection limit of 1 the first CG call tries it and falls back,
    the next call runs hprsdft without trying it, and setting the limit
    again clears the streak; every call's result is pc_kind 4's."""
    from rsdft_develop_amd import gpu

    cell = systems.silicon_supercell(1, ngrid_per_cell=24, nband=12, displacement=0.05, seed=4)
    v = systems.model_vloc(cell)
    ctx = gpu.Context().setup(cell, v)
    d = lpc.unpack(lpc.init_params(0))
    d["W3"] = np.zeros_like(d["W3"])
    d["b3"] = np.zeros_like(d["b3"])
    ctx.lpc_set_params(lpc.pack(d))
    ctx.lpc_set_potential(v)
    ctx.alloc_bands(cell.nband)
    u0 = systems.random_bands(cell.npoints, cell.nband, seed=1)

    def cg(pc):
        ctx.upload_bands(u0)
        ctx.gram_schmidt()
        ctx.subspace_diag()
        return ctx.conjugate_gradient(ncg=4, pc_kind=pc, mloop=3)[0], ctx.download_bands()

    ref = cg(4)
    ctx.lpc_set_reject_limit(1)
    seen = []
    for expect_fb, expect_skip in ((1, 0), (1, 1), (1, 2)):
        out = cg(5)
        seen.append((ctx.lpc_fallbacks(), ctx.lpc_reject_state()))
        np.testing.assert_allclose(out[0], ref[0], rtol=0, atol=1e-10)
        assert np.abs(out[1] - ref[1]).max() < 1e-8 * np.abs(ref[1]).max()
        assert ctx.lpc_fallbacks() == expect_fb and ctx.lpc_reject_state() == (1, expect_skip), seen
    ctx.lpc_set_reject_limit(1)  # a new streak: the network is tried again
    assert ctx.lpc_reject_state() == (0, 2)
    cg(5)
    assert ctx.lpc_fallbacks() == 2 and ctx.lpc_reject_state() == (1, 2)
    ctx.lpc_set_reject_limit(0)  # no limit: every call tries it
    for k in range(2):
        cg(5)
    assert ctx.lpc_fallbacks() == 4 and ctx.lpc_reject_state()[1] == 2


def test_trained_network_gain_over_no_preconditioner():
    """The shipped weights on a held-out Si64 cell (72^3, 160 bands): CG
    rounds to the residual tolerance hprsdft reaches in 8 rounds.  The
    network must reach it, and in fewer rounds than CG without a
    preconditioner; against hprsdft itself it needs 11 (recorded, not a
    gain)."""
    import os

    from rsdft_develop_amd import train_lpc

    path = os.path.join(os.path.dirname(lpc.__file__), "data", "lpc_si64.npz")
    cell = systems.silicon_supercell(2, displacement=0.05, seed=999)
    print("case: learned preconditioner rounds, held-out Si64", flush=True)
    ev = train_lpc.evaluate(lpc.load(path), cell)
    print({k: ev[k] for k in ("rounds_hprsdft", "rounds_learned", "rounds_none", "fallbacks")}, flush=True)
    assert ev["rounds_hprsdft"] == 8
    assert ev["reached_learned"] and ev["reached_none"]
    assert ev["rounds_learned"] < ev["rounds_none"]


def test_training_memory_of_a_large_batch(setup):
    """The quad layouts of the weight gradients stay within 1 GiB, whatever
    the batch: 648 samples of (17, 36, 36) would take 2.0 GiB.  They go
    through in groups (323, 323 and 2 samples); loss and gradients are the
    means over eight batches that need no groups.  Eight being a power of
    two, every dy and dz of the whole batch is the part's exactly, so only
    the order of the FP32 sums differs: chains of at most 409 additions,
    1.2e-6 of a chain's terms, 3e-8 of the sum of all terms over 2048
    chains; 1e-3 of the gradient leaves room for cancellation of 3e4."""
    import ctypes

    from rsdft_develop_amd import gpu, hip

    _, p, _, rng = setup
    n = (17, 36, 36)
    N, ns, parts = int(np.prod(n)), 648, 8
    ctx = gpu.Context()
    ctx.set_grid(n, np.diag([5.1, 10.8, 10.8]), 6)
    ctx.lpc_set_potential(0.3 * np.sin(np.arange(N) * 0.01))
    ctx.lpc_set_params(p)
    g = rng.standard_normal((N, ns), dtype=np.float32)
    t = np.float32(0.5) * g + np.float32(0.2)
    dg, dt = hip.DeviceArray.from_numpy(g), hip.DeviceArray.from_numpy(t)

    def free():
        a, b = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.runtime().hipMemGetInfo(ctypes.byref(a), ctypes.byref(b)) == 0
        return a.value

    print(f"case: {ns} training samples of {n}", flush=True)
    before = free()
    loss, grads = ctx.lpc_train_step(dg.ptr, dt.ptr, ns, want_grads=True)
    used = before - free()
    fields = N * ns * (4 + 32 + 32 + 4 + 2 + 32 + 32)  # two inputs, activations, y, dy, dz
    assert used < fields + 1.25 * 2 ** 30, (used, fields)
    step, losses, mean = ns // parts, [], 0.0
    for k in range(parts):
        o = k * step * N * 4
        lk, gk = ctx.lpc_train_step(dg.ptr + o, dt.ptr + o, step, want_grads=True)
        losses.append(lk)
        mean = mean + gk.astype(np.float64) / parts
    assert loss == pytest.approx(np.mean(losses), rel=1e-9)
    for k, want in lpc.unpack(mean).items():
        got = lpc.unpack(grads)[k]
        assert np.linalg.norm(got - want) < 1e-3 * np.linalg.norm(want), k
    dg.free()
    dt.free()
    ctx.close()


def test_planes_beyond_two_to_the_27_points(setup):
    """Sixteen channels of such a plane pass 2^31 values.  Input and potential
    of +-1 repeat every five rows, so that every norm is exact and the output
    repeats to the last bit: it is that of the five-row grid."""
    from rsdft_develop_amd import gpu, hip

    _, p, _, rng = setup
    rows = 5 * 52429
    assert 512 * rows > 2 ** 27
    sign = rng.permutation(np.repeat([-1.0, 1.0], 512 * 5 // 2)), rng.permutation(np.repeat([-1.0, 1.0], 512 * 5 // 2))
    out = []
    for n2 in (5, rows):
        N = 512 * n2
        ctx = gpu.Context()
        ctx.set_grid((512, n2, 1), np.diag([150.0, 0.3 * n2, 10.0]), 6)
        ctx.lpc_set_potential(np.tile(sign[0], n2 // 5))
        ctx.lpc_set_params(p)
        d = hip.DeviceArray.from_numpy(np.tile(sign[1].astype(np.float32), n2 // 5))
        o = hip.DeviceArray((N,), dtype=np.float32)
        print(f"case: network on a plane of {N} points", flush=True)
        ctx.lpc_apply_device(d.ptr, o.ptr, N, 1, dtype=np.float32)
        ctx.synchronize()
        out.append(o.to_numpy())
        d.free()
        o.free()
        ctx.close()
    assert np.abs(out[0]).max() > 0
    np.testing.assert_array_equal(out[1].reshape(-1, 512 * 5), np.broadcast_to(out[0], (rows // 5, 512 * 5)))


def _grads_with_the_gpu_roundings(op, g3, v3, t3, count, kappa):
    """Loss and gradients of one sample of a batch of `count` points in all,
    with the bfloat16 roundings of dy and dz that the kernels make."""
    q = lambda a: lo.bf16(a).astype(np.float64)  # noqa: E731
    _, c = lo.forward(op, g3, v3, bf16_storage=True)
    r = c["y"] - kappa * t3 / c["s"]
    dy = q(2.0 / count * r)
    dz2 = q(lo.conv_t(c["W3"], dy[None]) * (c["a2"] > 0))
    dz1 = q(lo.conv_t(c["W2"], dz2) * (c["a1"] > 0))
    return float((r * r).sum() / count), {
        "W1": lo.conv_dw(c["x"], dz1), "b1": dz1.reshape(16, -1).sum(1), "W2": lo.conv_dw(c["a1"], dz2),
        "b2": dz2.reshape(16, -1).sum(1), "W3": lo.conv_dw(c["a2"], dy[None]), "b3": np.array([dy.sum()])}


@pytest.mark.parametrize("n,ns", [((21, 13, 11), 3), ((18, 7, 9), 5), ((35, 5, 13), 3), ((16, 5, 10), 1),
                                  ((17, 6, 7), 3), ((3, 3, 3), 3), ((64, 3, 5), 1)])
def test_network_and_gradients_over_grids(setup, n, ns):
    """Lines that end in every place of a quad and of a 16-point chunk,
    z-runs of unequal length, planes that are no multiple of a tile, and
    point counts that leave the bias sums a tail; the targets weigh the line
    ends and the last points.  Forward: the tolerances of the test above.
    Gradients against a restatement with the same roundings: 5e-3 in norm.
    What is left are roundings that fall the other way on an FP32 difference
    (some 1 % of the activations, 4e-3 each: 4e-4 in norm) and, at the odd
    point, the sign of an activation near zero (2e-3 of the norm in a field
    of 5e5 values)."""
    from rsdft_develop_amd import gpu, hip

    _, p, _, _ = setup
    rng = np.random.default_rng(n[0] * 100 + ns)
    n1, n2, n3 = n
    N = n1 * n2 * n3
    ctx = gpu.Context()
    ctx.set_grid(n, np.diag([0.3 * k for k in n]), 6)
    v = 0.3 * np.sin(np.arange(N) * 0.7) + 0.1 * rng.standard_normal(N)
    ctx.lpc_set_potential(v)
    ctx.lpc_set_params(p)
    vn = ((v - v.mean()) / (np.sqrt(np.mean((v - v.mean()) ** 2)) + 1e-30)).astype(np.float32).reshape(n3, n2, n1)
    g = rng.standard_normal((N, ns)).astype(np.float32)
    t = (0.5 * g + 0.3).astype(np.float32)
    t.reshape(n3, n2, n1, ns)[:, :, [0, -1], :] += np.float32(2.0)
    t[-8:, -1] += np.float32(20.0)
    op = lpc.to_oracle(p)
    dg, dt, dp = hip.DeviceArray.from_numpy(g), hip.DeviceArray.from_numpy(t), hip.DeviceArray((N, ns), dtype=np.float32)
    print(f"case: network {n}, {ns} samples", flush=True)
    ctx.lpc_apply_device(dg.ptr, dp.ptr, N, ns, dtype=np.float32)
    ctx.synchronize()
    got = dp.to_numpy().astype(np.float64)
    loss, grads = ctx.lpc_train_step(dg.ptr, dt.ptr, ns, want_grads=True, kappa=1.7)
    want_loss, want = 0.0, {}
    for b in range(ns):
        g3 = g[:, b].astype(np.float64).reshape(n3, n2, n1)
        _, c = lo.forward(op, g3, vn, bf16_storage=True)
        err = np.abs(got[:, b] / c["s"] - c["y"].reshape(-1)) / np.abs(c["y"]).max()
        assert err.max() < 2e-2 and err.mean() < 2e-3, b
        lb, gb = _grads_with_the_gpu_roundings(op, g3, vn, t[:, b].astype(np.float64).reshape(n3, n2, n1), N * ns, 1.7)
        want_loss += lb
        want = {k: want.get(k, 0.0) + a for k, a in gb.items()}
    assert loss == pytest.approx(want_loss, rel=2e-3)
    gd = lpc.unpack(grads)
    for k, a in want.items():
        a = np.asarray(a).reshape(gd[k].shape)
        assert np.linalg.norm(gd[k] - a) < 5e-3 * np.linalg.norm(a), k
    for d in (dg, dt, dp):
        d.free()
    ctx.close()
