"""The rest of the drop-in boundary on the device: vmult_add / Tvmult /
Tvmult_add (schwarz_preconditioner.h:185-194), the multiplicative sweep with
the tiled 2^dim colors, and the error paths of the C ABI (non-finite output,
collapsed cells, CG without convergence)."""
import ctypes

import numpy as np
import pytest

import oracle as o
from test_gpu_parity import _tpss, dev, host, make, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,p,n,variant", [(2, 3, 7, 0), (2, 2, 6, 1), (3, 2, 4, 1), (3, 3, 4, 0)])
def test_vmult_add_and_transpose(dim, p, n, variant):
    t = _tpss()
    lv, sm, ref = make(dim, p, n, variant)
    src = o.splitmix_uniform(11, ref.N)
    d0 = o.splitmix_uniform(12, ref.N)
    Psrc = ref.precond_vmult(src)
    # vmult_add: dst += P src
    dst = dev(d0)
    sm.vmult_add(dst, dev(src))
    assert rel_err(host(dst), d0 + Psrc) < 1e-12
    # Tvmult: the reversed color sequence (the additive operator is symmetric)
    _, _, ref_t = make(dim, p, n, variant, reverse=True)
    dst = dev(np.zeros(ref.N))
    sm.Tvmult(dst, dev(src))
    PTsrc = host(dst)
    assert rel_err(PTsrc, ref_t.precond_vmult(src)) < 1e-12
    if variant == t.ADDITIVE:
        assert rel_err(PTsrc, Psrc) < 1e-12
    # adjoint identity <P^T x, y> = <x, P y>
    y = o.splitmix_uniform(13, ref.N)
    dy = dev(np.zeros(ref.N))
    sm.vmult(dy, dev(y))
    lhs, rhs = PTsrc @ y, src @ host(dy)
    assert abs(lhs - rhs) < 1e-12 * (np.abs(PTsrc).max() * np.abs(y).sum())
    # Tvmult_add
    dst = dev(d0)
    sm.Tvmult_add(dst, dev(src))
    assert rel_err(host(dst), d0 + PTsrc) < 1e-12


@pytest.mark.parametrize("dim,p,n,fused", [(2, 3, 8, True), (3, 3, 5, True), (3, 2, 6, False)])
def test_tiled_coloring_mvp_parity(dim, p, n, fused):
    """The multiplicative smoother with the 2^dim tiled colors (8 in 3D, the
    color count of the 64^3 Q3 configuration) against the oracle."""
    t = _tpss()
    lv, sm, ref = make(dim, p, n, t.MULTIPLICATIVE, coloring=t.COLOR_TILED)
    assert sm.n_colors == 2 ** dim == ref.n_colors
    np.testing.assert_array_equal(sm.color_ptr(), ref.color_ptr())
    sm.set_fused_residual(fused)
    src = o.splitmix_uniform(3, ref.N)
    dst = dev(np.zeros(ref.N))
    sm.precond_vmult(dst, dev(src))
    assert rel_err(host(dst), ref.precond_vmult(src)) < 1e-12
    x = dev(o.splitmix_uniform(4, ref.N))
    sm.vmult(x, dev(src))
    assert rel_err(host(x), ref.smoother_vmult(src)) < 1e-12


def test_nonfinite_output_is_reported():
    t = _tpss()
    lv, sm, ref = make(3, 2, 4, t.MULTIPLICATIVE)
    src = o.splitmix_uniform(3, ref.N)
    bad = src.copy()
    bad[17] = np.nan
    dst = dev(np.zeros(ref.N))
    # default mode: no synchronisation in the call, reported afterwards
    sm.vmult(dst, dev(bad))
    with pytest.raises(t.TPSSError) as e:
        sm.finite_status()
    assert e.value.code == t.E_NONFINITE
    sm.finite_status()  # the report clears the flag
    # reported by the next apply call once the check has run
    sm.vmult(dst, dev(bad))
    t.synchronize()
    with pytest.raises(t.TPSSError) as e:
        sm.vmult(dst, dev(src))
    assert e.value.code == t.E_NONFINITE
    sm.vmult(dst, dev(src))
    assert rel_err(host(dst), ref.smoother_vmult(src)) < 1e-12
    sm.finite_status()
    # synchronous mode reports in the call itself
    sm.set_check_finite(2)
    with pytest.raises(t.TPSSError) as e:
        sm.precond_vmult(dst, dev(bad))
    assert e.value.code == t.E_NONFINITE
    # off: nothing is reported
    sm.set_check_finite(0)
    sm.precond_vmult(dst, dev(bad))
    sm.finite_status()
    # Inf in an FP32 level vector
    lv32 = t.Level(2, 3, 5, precision=t.F32)
    sm32 = t.SchwarzSmoother(lv32, variant=t.ADDITIVE)
    b32 = np.ones(lv32.n_dofs, dtype=np.float32)
    b32[3] = np.inf
    d32 = dev(np.zeros(lv32.n_dofs, dtype=np.float32))
    sm32.precond_vmult(d32, dev(b32))
    with pytest.raises(t.TPSSError) as e:
        sm32.finite_status()
    assert e.value.code == t.E_NONFINITE


@pytest.mark.parametrize("dim,p,n", [(3, 3, 6), (3, 2, 4), (3, 3, 16), (3, 3, 19), (3, 1, 5), (3, 4, 3),
                                     (2, 3, 7), (2, 1, 9), (2, 4, 5)])
def test_nonfinite_check_of_the_residual_free_passes(dim, p, n):
    """The residual-free color passes check the values they store themselves
    (no separate pass over the output); the accumulating entry points keep the
    pass over the output.  3D Q3: colors of at most 256 patches (n = 6, 16) run
    the four-wave pass, larger ones (n = 19) one wave per patch."""
    t = _tpss()
    lv, sm, ref = make(dim, p, n, t.MULTIPLICATIVE)
    N = ref.N
    src = o.splitmix_uniform(3, N)
    # a NaN in the right-hand side of a Richardson step (read by the patches
    # holding that DoF) reaches the output
    b = src.copy()
    b[N // 2] = np.nan
    sm.step(dev(o.splitmix_uniform(4, N)), dev(b))
    with pytest.raises(t.TPSSError) as e:
        sm.finite_status()
    assert e.value.code == t.E_NONFINITE
    # Tvmult with an Inf in the source
    bad = src.copy()
    bad[N - 1] = np.inf
    dst = dev(np.zeros(N))
    sm.Tvmult(dst, dev(bad))
    with pytest.raises(t.TPSSError) as e:
        sm.finite_status()
    assert e.value.code == t.E_NONFINITE
    # vmult_add: the passes write a temporary; a NaN already in dst is found by
    # the pass over the output
    d = np.zeros(N)
    d[7] = np.nan
    sm.vmult_add(dev(d), dev(src))
    with pytest.raises(t.TPSSError) as e:
        sm.finite_status()
    assert e.value.code == t.E_NONFINITE
    # finite data: nothing reported, and the results are unchanged
    dst = dev(np.zeros(N))
    sm.precond_vmult(dst, dev(src))
    sm.finite_status()
    assert rel_err(host(dst), ref.precond_vmult(src)) < 1e-12


@pytest.mark.parametrize("dim,p,n,ras", [(2, 3, 5, 0), (2, 1, 6, 1), (2, 2, 5, 2), (3, 2, 4, 0), (3, 4, 3, 0),
                                         (3, 3, 4, 1), (3, 1, 5, 2)])
@pytest.mark.parametrize("prec", [0, 1])
def test_nonfinite_check_of_the_additive_slot_sum(dim, p, n, ras, prec):
    """The additive slot sum checks the values it stores (no separate pass over
    the output), also where it accumulates into dst."""
    t = _tpss()
    dt = np.float32 if prec else np.float64
    lv = t.Level(dim, p, n, precision=prec)
    N = lv.n_dofs
    src = o.splitmix_uniform(3, N).astype(dt)

    def reported(sm, call, x, b):
        call(dev(x, prec), dev(b, prec))
        try:
            sm.finite_status()
        except t.TPSSError as e:
            assert e.code == t.E_NONFINITE
            return True
        return False

    zero = np.zeros(N, dt)
    for kw in ({}, dict(n_steps=2), dict(damping_factor=0.8)):
        sm = t.SchwarzSmoother(lv, t.ADDITIVE, ras=ras, relaxation=0.2, **kw)
        calls = [sm.precond_vmult, sm.vmult_add, sm.Tvmult, sm.vmult, sm.step]
        for call in calls:
            assert not reported(sm, call, zero, src)
            for at, value in ((0, np.nan), (N // 2, np.inf), (N - 1, -np.inf)):
                bad = src.copy()
                bad[at] = value
                assert reported(sm, call, zero, bad)
                assert not reported(sm, call, zero, src)
                if call == sm.vmult_add:  # already in dst
                    assert reported(sm, call, bad, src)


def test_gmg_solve_reports_nonfinite_and_no_convergence():
    t = _tpss()
    g = t.GMGSolver(2, 2, 2, 3)
    b = o.splitmix_uniform(2, g.n_dofs)
    x = dev(np.zeros(g.n_dofs))
    with pytest.raises(t.TPSSError) as e:
        g.solve(x, dev(b), rel_tol=1e-14, max_iter=1)
    assert e.value.code == t.E_NOT_CONVERGED
    info, hist = g.solve(x, dev(b), rel_tol=1e-14, max_iter=1, raise_on_fail=False)
    assert len(hist) == 2 and hist[1] > 1e-14 * hist[0]
    bad = b.copy()
    bad[5] = np.nan
    with pytest.raises(t.TPSSError) as e:
        g.solve(x, dev(bad), rel_tol=1e-8, max_iter=10)
    assert e.value.code == t.E_NONFINITE


def test_collapsed_cell_is_singular():
    t = _tpss()
    V = o.uniform_vertices(2, 4).reshape(5, 5, 2).copy()
    V[:, 1, 0] = V[:, 2, 0]  # the column of cells between x-vertices 1 and 2 has zero width
    with pytest.raises(t.TPSSError) as e:
        t.Level(2, 2, 4, vertices=V.reshape(-1, 2))
    assert e.value.code == t.E_SINGULAR
    with pytest.raises(t.TPSSError) as e:
        t.GMGSolver(2, 2, 2, 2, vertices=V.reshape(-1, 2))
    assert e.value.code == t.E_SINGULAR


@pytest.mark.parametrize("variant,distorted", [(0, False), (1, True)])
def test_step_after_vmult_allocates_nothing(variant, distorted):
    """vmult from zero needs neither a residual nor a correction vector, but leaves them
    allocated: a caller may capture the launches of a step on the same handle"""
    t = _tpss()
    hip = ctypes.CDLL("libamdhip64.so.7")  # the runtime that the library has loaded
    p = ctypes.byref

    def free_bytes():
        free, total = ctypes.c_size_t(), ctypes.c_size_t()
        t.synchronize()
        assert hip.hipMemGetInfo(p(free), p(total)) == 0
        return free.value

    n = 28  # vectors of 4.7 MB, beyond the granularity of a device allocation
    V = o.distorted_vertices(3, n, 0.1, seed=3) if distorted else None
    lv = t.Level(3, 2, n, ip_factor=2.0, vertices=V)
    x0 = o.splitmix_uniform(4, lv.n_dofs)
    src, x, y = dev(o.splitmix_uniform(3, lv.n_dofs)), dev(x0), dev(x0)
    sm = t.SchwarzSmoother(lv, variant, relaxation=0.5)
    sm.vmult(x, src)
    before = free_bytes()
    sm.step(y, src)
    assert free_bytes() == before
    eager = host(y)
    # captured right after a vmult on a fresh handle, and replayed between eager steps
    sm = t.SchwarzSmoother(lv, variant, relaxation=0.5)
    sm.vmult(x, src)
    t.synchronize()
    stream, graph, ex = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_void_p()
    assert hip.hipStreamCreate(p(stream)) == 0
    assert hip.hipStreamBeginCapture(stream, 0) == 0
    sm.step(x, src, stream=stream.value)
    assert hip.hipStreamEndCapture(stream, p(graph)) == 0
    assert hip.hipGraphInstantiate(p(ex), graph, None, None, ctypes.c_size_t(0)) == 0
    for _ in range(3):
        x.upload(x0)
        assert hip.hipGraphLaunch(ex, stream) == 0
        np.testing.assert_array_equal(host(x), eager)
        x.upload(x0)
        sm.step(x, src)
        np.testing.assert_array_equal(host(x), eager)
    assert hip.hipGraphExecDestroy(ex) == 0 and hip.hipGraphDestroy(graph) == 0
    assert hip.hipStreamDestroy(stream) == 0
