"""GPU tests of the solver's one-pass products and steps: lengths around the
16-byte groups, every history up to the one-pass limit and beyond, misaligned
parts of stacked vectors, and vectors that take each other's memory."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _fcg(a, d, niter, history, eps=0.0):
    """Flexible CG from zero on the diagonal rows [a; eps I] in FP64."""
    A = np.concatenate([a, np.full(a.size, eps)]) if eps else a
    n = a.size
    fwd = (lambda p: np.concatenate([a * p, eps * p])) if eps else (lambda p: a * p)
    adj = (lambda q: a * q[:n] + eps * q[n:]) if eps else (lambda q: a * q)
    rr = -(np.concatenate([d, np.zeros(n)]) if eps else d)
    m, S, SS, hist = np.zeros(n), [], [], [1.0]
    r0 = np.linalg.norm(rr)
    for _ in range(niter):
        g = adj(rr)
        gg = fwd(g)
        B = [gg] + SS
        M = np.array([[u @ v for v in B] for u in B])
        x = np.linalg.solve(M, -np.array([u @ rr for u in B]))
        s = x[0] * g + sum((xi * u for xi, u in zip(x[1:], S)), np.zeros(n))
        ss = x[0] * gg + sum((xi * u for xi, u in zip(x[1:], SS)), np.zeros(A.size))
        m, rr = m + s, rr + ss
        S, SS = ([s] + S)[:max(1, history)], ([ss] + SS)[:max(1, history)]
        hist.append(np.linalg.norm(rr) / r0)
    return m, hist


@pytest.mark.parametrize("n", [5, 1023, 4098, 262147])
@pytest.mark.parametrize("history", [0, 2, 8, 9, 16])
def test_solver_steps_against_fp64(dev, n, history):
    from sep_code_amd.operator import DeviceVector, IOp, RegSolver, SimpleSolver, WeightOp, cgstep
    r = np.random.default_rng(n + history)
    a = r.uniform(0.5, 2.0, n)
    d = r.standard_normal(n)
    wv = DeviceVector.from_array(dev, a)
    dv = DeviceVector.from_array(dev, d)
    a32, d32 = a.astype(np.float32).astype(np.float64), d.astype(np.float32).astype(np.float64)
    niter = min(3, n - 1)
    for eps in (0.0, 0.25):  # 0.25: a stacked range, its second part at n floats
        op = WeightOp(wv)
        sol = (RegSolver(cgstep(), dv, op, IOp(dev, n), eps, history=history) if eps else
               SimpleSolver(cgstep(), dv, op, history=history))
        res = sol.solve(niter)
        m, hist = _fcg(a32, d32, niter, history, eps)
        # FP32 vectors, FP64 scalars: a few roundings per step
        np.testing.assert_allclose(res.resid_hist, hist, rtol=2e-5)
        got = sol.return_model().numpy().astype(np.float64)
        assert np.linalg.norm(got - m) <= 2e-5 * np.linalg.norm(m)
        sol.close()


@pytest.mark.parametrize("n", [1, 3, 4, 7, 1000003])
def test_vector_kernels_at_odd_lengths(dev, n):
    from sep_code_amd.operator import DeviceVector
    r = np.random.default_rng(n)
    a, b = (r.standard_normal(n).astype(np.float32) for _ in range(2))
    va, vb = DeviceVector.from_array(dev, a), DeviceVector.from_array(dev, b)
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    # n FP64 additions of exact products
    assert abs(va.dot(vb) - a64 @ b64) <= n * 2.3e-16 * (np.abs(a64 * b64).sum() + 1e-300)
    want = (1.5 * a64 - 0.25 * b64).astype(np.float32)
    np.testing.assert_array_equal(va.clone().scale_add(1.5, vb, -0.25).numpy(), want)
    np.testing.assert_array_equal(va.clone().mult(vb).numpy(), a * b)


def test_new_vectors_are_zero_whatever_memory_they_take(dev):
    from sep_code_amd.operator import DeviceVector
    n = 100_000
    before = dev.device_bytes()
    for k in range(4):
        v = DeviceVector.from_array(dev, np.full(n - 10 * k, 3.0, np.float32))
        v.close()
        w = DeviceVector(dev, n - 10 * k)
        assert not w.numpy().any()
        w.close()
    # the memory kept for reuse is counted, and a new grid gives it back
    assert dev.device_bytes() >= before
    dev.create_space((10.0, 10.0, 10.0), 4.0, 0.0, (16, 16, 16))
    kept = dev.device_bytes()
    DeviceVector(dev, n).close()
    assert dev.device_bytes() >= kept + 4 * n
    dev.create_space((10.0, 10.0, 10.0), 4.0, 0.0, (16, 16, 16))
    assert dev.device_bytes() == kept


def test_history_change_restarts_from_no_previous_step(dev):
    """One flexible step, then cgstep: the scratch step it reads is empty, so
    it stops as a breakdown, as with freshly made vectors."""
    from sep_code_amd.operator import DeviceVector, SimpleSolver, WeightOp, cgstep
    n = 5000
    r = np.random.default_rng(3)
    wv = DeviceVector.from_array(dev, r.uniform(0.5, 2.0, n))
    dv = DeviceVector.from_array(dev, r.standard_normal(n))
    DeviceVector.from_array(dev, np.full(n, 7.0, np.float32)).close()  # dirty memory to take
    sol = SimpleSolver(cgstep(), dv, WeightOp(wv), history=4)
    sol.solve(1)
    sol.history = 0
    res = sol.solve(2)
    assert res.breakdown and res.iterations == 0
    sol.close()
