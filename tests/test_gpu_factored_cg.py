"""CG-SR through the RBM factors against the stored O rows, bit for bit.

A gradient callback sends a step through the materialised O; with the
library's own gradient as that callback the rows are the ones the factored
products stand for, so every sum has the same terms in the same order and
the step's information and parameters must be equal to the last bit, at the
edges of the kernels' tiles: rows around 64, chunks around 128, sites and
hidden units around 16 and 32, hidden units of fewer than 8 sites, t staged
in one piece and in segments, and a vector too long for the one-workgroup
iteration.
"""
import ctypes

import numpy as np
import pytest

import scenarios
from spin_based_neural_network_amd.abi import (MarshallWrapper, SrInfo, config_defaults, fnptr,
                                               options_defaults)

pytestmark = pytest.mark.gpu

RBM, CRBM, TFIM = 5, 6, 0
REAL_CB = ctypes.CFUNCTYPE(ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p,
                           ctypes.c_int, ctypes.c_void_p)
HOLO_CB = ctypes.CFUNCTYPE(ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p,
                           ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p)


def _steps(hip, kind, N, M, B, chains, holo, precision, rows, steps=2, marshall=False):
    cfg = config_defaults(ansatz=kind, hamiltonian=TFIM, transverse_field=0.9, rbm_hidden_units=M,
                          rbm_init_scale=0.4, num_samples=B, num_thermalize=2 * N,
                          num_decorrelate=N, rng_seed=31 + N + M, learning_rate=1e-2,
                          sr_diag_shift=1e-3, sr_cg_max_iters=40, sr_cg_tol=1e-6)
    r = scenarios.Runner(hip, "nqs_")
    a = r.ansatz(cfg, N)
    fn, user = fnptr(hip, "nqs_ansatz_log_amp"), a
    if marshall:
        wrap = MarshallWrapper(fn, a, N, 1)
        fn, user = fnptr(hip, "nqs_marshall_log_amp"), ctypes.addressof(wrap)
    opt = options_defaults(num_chains=chains, periodic=1, precision=precision)
    s = hip.nqs_hip_sampler_create_ex(N, ctypes.byref(cfg), ctypes.byref(opt), fn, user)
    assert s
    hip.nqs_sampler_thermalize(s)
    cb = None
    if rows:
        cb = (HOLO_CB(lambda u, x, sp, n, re, im:
                      hip.nqs_ansatz_logpsi_gradient_complex(x, sp, n, re, im)) if holo else
              REAL_CB(lambda u, x, sp, n, g: hip.nqs_ansatz_logpsi_gradient(x, sp, n, g)))
    step = hip.nqs_sr_step_holomorphic_full if holo else hip.nqs_sr_step_custom_full
    out = []
    for _ in range(steps):
        info = SrInfo()
        assert step(ctypes.byref(cfg), N, 1, a, s, fn, user, ctypes.cast(cb, ctypes.c_void_p), None,
                    ctypes.byref(info)) == 0
        out.append((info.as_dict(), r.params(a)))
    hip.nqs_sampler_free(s)
    hip.nqs_ansatz_free(a)
    return out


@pytest.mark.parametrize("kind,holo,N,M,B,chains", [
    (CRBM, True, 24, 96, 320, 64), (CRBM, True, 4, 9, 200, 40), (CRBM, True, 9, 1, 63, 21),
    (CRBM, True, 16, 16, 129, 43), (CRBM, True, 33, 31, 128, 32), (CRBM, True, 12, 300, 65, 13),
    (CRBM, True, 40, 210, 40, 40), (CRBM, False, 15, 47, 257, 64), (CRBM, False, 64, 20, 100, 50),
    (RBM, True, 10, 33, 191, 30), (RBM, True, 3, 5, 64, 16),
])
def test_factored_cg_equals_stored_rows(hip, kind, holo, N, M, B, chains):
    print("factored CG:", kind, holo, N, M, B, flush=True)
    got = _steps(hip, kind, N, M, B, chains, holo, 0, False)
    ref = _steps(hip, kind, N, M, B, chains, holo, 0, True)
    for (gi, gp), (ri, rp) in zip(got, ref):
        assert gi == ri
        assert np.array_equal(gp, rp)


# more than 64 sites, hidden units past one staging with enough rows for the
# factored route; the real-projected step of a real RBM (with a sign rule on its
# amplitude, which keeps it out of the batched path)
@pytest.mark.parametrize("kind,holo,N,M,B,chains", [
    (CRBM, True, 65, 16, 70, 14), (CRBM, True, 81, 20, 100, 50), (CRBM, True, 100, 33, 129, 43),
    (CRBM, True, 128, 31, 191, 30), (CRBM, True, 256, 3, 64, 16), (CRBM, False, 65, 15, 257, 64),
    (CRBM, False, 127, 8, 128, 32), (CRBM, False, 200, 5, 300, 60), (CRBM, False, 5, 150, 200, 40),
    (RBM, False, 15, 31, 63, 21), (RBM, False, 16, 32, 64, 32), (RBM, False, 17, 33, 65, 13),
    (RBM, False, 31, 16, 127, 127), (RBM, False, 33, 15, 129, 43), (RBM, False, 64, 20, 128, 64),
    (RBM, False, 100, 17, 300, 60), (RBM, False, 3, 1, 40, 8),
])
def test_factored_cg_equals_stored_rows_wide(hip, kind, holo, N, M, B, chains):
    print("factored CG:", kind, holo, N, M, B, flush=True)
    marshall = kind == RBM
    c, ms = ctypes.c_longlong(), ctypes.c_double()
    hip.nqs_hip_kernel_timing(b"frows_rowdot")
    got = _steps(hip, kind, N, M, B, chains, holo, 0, False, marshall=marshall)
    assert hip.nqs_hip_kernel_stats(b"frows_rowdot", ctypes.byref(c), ctypes.byref(ms)) == 0 and c.value > 0
    hip.nqs_hip_kernel_timing(None)
    ref = _steps(hip, kind, N, M, B, chains, holo, 0, True, marshall=marshall)
    for (gi, gp), (ri, rp) in zip(got, ref):
        assert gi == ri
        assert np.array_equal(gp, rp)


@pytest.mark.parametrize("kind,holo", [(CRBM, True), (CRBM, False), (RBM, False)])
def test_factored_cg_single_precision_factors(hip, kind, holo):
    """FP32 factors are widened exactly: the step stays within the FP32
    amplitudes' error of the FP64 one (about 1e-6 in t, times the solve's
    1 / shift on an update of a few hundredths)."""
    f32 = _steps(hip, kind, 12, 24, 480, 60, holo, 1, False, steps=1)[0]
    f64 = _steps(hip, kind, 12, 24, 480, 60, holo, 0, False, steps=1)[0]
    assert abs(f32[0]["mean_energy"] - f64[0]["mean_energy"]) < 1e-4 * abs(f64[0]["mean_energy"])
    assert np.abs(f32[1] - f64[1]).max() < 2e-3 * f64[0]["update_norm"] + 1e-6


@pytest.mark.parametrize("holo", [True, False])
def test_stored_rows_stop_with_their_eight(hip, holo):
    """A solve that converges within eight iterations launches nothing past
    them where its products read stored rows: as many launches as one that is
    limited to eight."""
    def launches(iters):
        cfg = config_defaults(ansatz=CRBM, hamiltonian=TFIM, transverse_field=0.9, rbm_hidden_units=4,
                              num_samples=256, num_thermalize=8, num_decorrelate=2, rng_seed=5,
                              learning_rate=1e-2, sr_diag_shift=10.0, sr_cg_max_iters=iters,
                              sr_cg_tol=1e-2)
        r = scenarios.Runner(hip, "nqs_")
        a, fn = r.ansatz(cfg, 6), fnptr(hip, "nqs_ansatz_log_amp")
        opt = options_defaults(num_chains=32, periodic=1)
        s = hip.nqs_hip_sampler_create_ex(6, ctypes.byref(cfg), ctypes.byref(opt), fn, a)
        assert s
        hip.nqs_sampler_thermalize(s)
        cb = (HOLO_CB(lambda u, x, sp, n, re, im:
                      hip.nqs_ansatz_logpsi_gradient_complex(x, sp, n, re, im)) if holo else
              REAL_CB(lambda u, x, sp, n, g: hip.nqs_ansatz_logpsi_gradient(x, sp, n, g)))
        step = hip.nqs_sr_step_holomorphic_full if holo else hip.nqs_sr_step_custom_full
        info, before = SrInfo(), hip.nqs_hip_device_launches()
        assert step(ctypes.byref(cfg), 6, 1, a, s, fn, a, ctypes.cast(cb, ctypes.c_void_p), None,
                    ctypes.byref(info)) == 0
        n = hip.nqs_hip_device_launches() - before
        hip.nqs_sampler_free(s)
        hip.nqs_ansatz_free(a)
        return n, info.cg_iterations, info.converged

    launches(8)   # buffers and tables once
    few, many = launches(8), launches(100)
    assert many[2] == 1 and many[1] <= 8
    assert few == many


@pytest.mark.parametrize("kind,holo,N,M,B,factored", [
    (CRBM, False, 9, 100, 16, True), (CRBM, False, 16, 64, 80, False), (CRBM, False, 16, 64, 81, True),
    (CRBM, False, 64, 20, 340, False), (CRBM, False, 64, 20, 341, True),
    (CRBM, False, 24, 96, 1280, False), (CRBM, False, 24, 96, 1281, True),
    (CRBM, True, 36, 100, 16, True), (CRBM, True, 64, 120, 16, False), (CRBM, True, 64, 120, 17, True),
    (CRBM, True, 64, 90, 64, False), (CRBM, True, 64, 90, 65, True), (CRBM, True, 64, 130, 16, True),
    (RBM, True, 36, 100, 16, True),
])
def test_few_rows_are_stored(hip, kind, holo, N, M, B, factored):
    """Few samples of many parameters go through stored rows, which take less
    there, on either side of the lines; with the same bits.  (From 512 samples
    on theta comes from a product of its own, which a callback's rows do not
    see: the route alone.)"""
    print("route:", kind, holo, N, M, B, flush=True)
    c, ms = ctypes.c_longlong(), ctypes.c_double()
    hip.nqs_hip_kernel_timing(b"frows_rowdot")
    got = _steps(hip, kind, N, M, B, 16, holo, 0, False)
    on = hip.nqs_hip_kernel_stats(b"frows_rowdot", ctypes.byref(c), ctypes.byref(ms)) == 0 and c.value > 0
    hip.nqs_hip_kernel_timing(None)
    assert on == factored
    if B >= 512:
        return
    ref = _steps(hip, kind, N, M, B, 16, holo, 0, True)
    for (gi, gp), (ri, rp) in zip(got, ref):
        assert gi == ri
        assert np.array_equal(gp, rp)
