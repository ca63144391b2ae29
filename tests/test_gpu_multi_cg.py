"""Batched CG at the edges of its kernels' tiles and splits.

* A batch of one against the same step through the stored O rows (the
  library's own gradient as callback): three CG iterations, which 64 bits
  determine, so the two summation orders agree to rounding times the
  amplification of three iterations.  Sizes around the 16-row and 16-site
  tiles, the 32-site words, the 64-row sums and the 256-element slices;
  samples around the 16-sample tiles, one slot and many, slots that hold no
  sample, more samples in a workgroup than it has in hand.
* The cooperative launch against the launch sequence, bit for bit, for
  batches with fewer workgroups than the vectors want (vectors in memory) and
  with more problems than CUs (no cooperative launch; its problems in smaller
  batches have it).
"""
import ctypes

import numpy as np
import pytest

import scenarios
from spin_based_neural_network_amd.abi import SrInfo, config_defaults, fnptr, options_defaults

pytestmark = pytest.mark.gpu

RBM, TFIM = 5, 0
GRAD_CB = ctypes.CFUNCTYPE(ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p,
                           ctypes.c_int, ctypes.c_void_p)


def _problem(hip, r, N, M, B, chains, iters, seed):
    cfg = config_defaults(ansatz=RBM, hamiltonian=TFIM, transverse_field=0.9, rbm_hidden_units=M,
                          rbm_init_scale=0.3, num_samples=B, num_thermalize=N, num_decorrelate=2,
                          rng_seed=seed, learning_rate=1e-2, sr_diag_shift=1e-2,
                          sr_cg_max_iters=iters, sr_cg_tol=1e-10)
    a = r.ansatz(cfg, N)
    fn = fnptr(hip, "nqs_ansatz_log_amp")
    opt = options_defaults(num_chains=chains, periodic=1)
    s = hip.nqs_hip_sampler_create_ex(N, ctypes.byref(cfg), ctypes.byref(opt), fn, a)
    assert s
    return dict(cfg=cfg, N=N, a=a, s=s, fn=fn)


def _free(hip, probs):
    for p in probs:
        hip.nqs_sampler_free(p["s"])
        hip.nqs_ansatz_free(p["a"])


@pytest.mark.parametrize("N,M,B,chains", [
    (2, 1, 1, 1), (3, 5, 17, 17), (15, 15, 64, 16), (16, 16, 65, 13), (17, 31, 130, 10),
    (31, 33, 1000, 100), (32, 63, 200, 50), (63, 64, 2050, 205), (64, 65, 300, 60),
    (96, 129, 128, 64), (4, 300, 3000, 100), (128, 256, 33, 33), (200, 20, 516, 129),
])
def test_one_problem_equals_stored_rows(hip, N, M, B, chains):
    print("batch of one:", N, M, B, flush=True)
    r = scenarios.Runner(hip, "nqs_")
    out = []
    for rows in (False, True):
        p = _problem(hip, r, N, M, B, chains, 3, 7 + N + M)
        cb = GRAD_CB(lambda u, x, sp, n, g: hip.nqs_ansatz_logpsi_gradient(x, sp, n, g)) if rows else None
        p0, info = r.params(p["a"]), SrInfo()
        assert hip.nqs_sr_step_custom_full(ctypes.byref(p["cfg"]), N, 1, p["a"], p["s"], p["fn"],
                                           p["a"], ctypes.cast(cb, ctypes.c_void_p), None,
                                           ctypes.byref(info)) == 0
        out.append((r.params(p["a"]) - p0, info.mean_energy, info.cg_iterations))
        _free(hip, [p])
    (got, e, it), (ref, e_ref, it_ref) = out
    assert abs(e - e_ref) <= 1e-12 * abs(e_ref) and it == it_ref
    # |delta| is subtracted from parameters of order 1: 2^-52 each, and the
    # products' sums over B samples and P terms enter three times
    tol = 3 * 2.0 ** -52 * (B + N * M) * np.abs(ref).max() + 2.0 ** -50
    assert np.abs(got - ref).max() <= tol, (np.abs(got - ref).max(), tol)


@pytest.mark.parametrize("split", [8, 256])
@pytest.mark.parametrize("n,N,M,B,group", [(160, 64, 64, 48, 160), (300, 6, 8, 64, 100),
                                           (40, 20, 90, 520, 40)])
def test_cooperative_launch_equals_launch_sequence(hip, monkeypatch, n, N, M, B, group, split):
    """One batch as a launch sequence, and `group` problems at a time in the
    cooperative launch, both at the same split target (4 and 8 slots for the
    520 samples; timed targets may differ from batch to batch)."""
    print("cooperative launch:", n, N, M, B, split, flush=True)
    monkeypatch.setenv("NQS_HIP_MULTI_SPLIT", str(split))
    r = scenarios.Runner(hip, "nqs_")
    params = []
    for on in (0, 1):
        probs = [_problem(hip, r, N + i % 2, M + i % 3, B, 16, 12, 5 + i) for i in range(n)]
        for k in range(0, n, group if on else n):
            part = probs[k:k + (group if on else n)]
            g = len(part)
            cfgs = (type(part[0]["cfg"]) * g)(*[p["cfg"] for p in part])
            m = hip.nqs_hip_multi_create(g, cfgs, (ctypes.c_int * g)(*[p["N"] for p in part]),
                                         (ctypes.c_int * g)(*[1] * g),
                                         (ctypes.c_void_p * g)(*[p["a"] for p in part]),
                                         (ctypes.c_void_p * g)(*[p["s"] for p in part]))
            assert m
            assert hip.nqs_hip_multi_use_persistent(m, on) == 0
            info = (SrInfo * g)()
            count, ms = ctypes.c_longlong(), ctypes.c_double()
            hip.nqs_hip_kernel_timing(b"multi_cg")
            for _ in range(2):
                assert hip.nqs_hip_multi_step(m, info) == 0
            assert hip.nqs_hip_kernel_stats(b"multi_cg", ctypes.byref(count), ctypes.byref(ms)) == 0
            hip.nqs_hip_kernel_timing(None)
            assert count.value == (2 if on else 0)
            assert hip.nqs_hip_multi_sync(m) == 0
            hip.nqs_hip_multi_free(m)
        params.append([r.params(p["a"]) for p in probs])
        _free(hip, probs)
    for p, q in zip(*params):
        assert np.array_equal(p, q)


def test_workgroups_that_do_not_meet(hip, monkeypatch, capfd):
    """A cooperative launch that gives its meetings up at once (no look at the
    counter: every workgroup of a problem that has several leaves): the step
    ends on the launch sequence, with its bits, and so do the later ones."""
    monkeypatch.setenv("NQS_HIP_MULTI_SPLIT", "64")
    r = scenarios.Runner(hip, "nqs_")
    out = []
    for polls, on in (("0", 1), (None, 0)):
        if polls:
            monkeypatch.setenv("NQS_HIP_MULTI_POLLS", polls)
        else:
            monkeypatch.delenv("NQS_HIP_MULTI_POLLS")
        probs = [_problem(hip, r, N, M, B, 16, 12, 3 + N) for N, M, B in
                 ((20, 40, 512), (6, 5, 64), (64, 128, 256))]
        n = len(probs)
        cfgs = (type(probs[0]["cfg"]) * n)(*[p["cfg"] for p in probs])
        m = hip.nqs_hip_multi_create(n, cfgs, (ctypes.c_int * n)(*[p["N"] for p in probs]),
                                     (ctypes.c_int * n)(*[1] * n),
                                     (ctypes.c_void_p * n)(*[p["a"] for p in probs]),
                                     (ctypes.c_void_p * n)(*[p["s"] for p in probs]))
        assert m
        assert hip.nqs_hip_multi_use_persistent(m, on) == 0
        info, steps = (SrInfo * n)(), []
        for _ in range(3):
            assert hip.nqs_hip_multi_step(m, info) == 0
            assert hip.nqs_hip_multi_sync(m) == 0
            steps.append(([i.as_dict() for i in info], [r.params(p["a"]) for p in probs]))
        out.append(steps)
        hip.nqs_hip_multi_free(m)
        _free(hip, probs)
        assert capfd.readouterr().err.count("did not meet") == (1 if on else 0)
    for (gi, gp), (ri, rp) in zip(*out):
        assert gi == ri
        assert all(np.array_equal(g, q) for g, q in zip(gp, rp))


@pytest.mark.parametrize("N,M,B", [(130, 130, 33), (64, 260, 500), (255, 65, 129), (20, 1000, 64), (128, 512, 16),
                                   (200, 100, 1300)])
def test_shared_rows_equal_one_share(hip, monkeypatch, N, M, B):
    """Few samples of many parameters share the rows of p over workgroups, in the
    cooperative launch and in the launch sequence: the bits of a batch that leaves
    each problem too few workgroups for that (256 problems; others beside it)."""
    print("shared rows:", N, M, B, flush=True)
    monkeypatch.setenv("NQS_HIP_MULTI_SPLIT", "64")
    r = scenarios.Runner(hip, "nqs_")
    out = []
    for on, beside in ((1, 0), (0, 0), (0, 300)):
        probs = [_problem(hip, r, N, M, B, 16, 6, 9)]
        probs += [_problem(hip, r, 4, 3, 128, 16, 6, 20 + i) for i in range(beside)]
        n = len(probs)
        cfgs = (type(probs[0]["cfg"]) * n)(*[p["cfg"] for p in probs])
        m = hip.nqs_hip_multi_create(n, cfgs, (ctypes.c_int * n)(*[p["N"] for p in probs]),
                                     (ctypes.c_int * n)(*[1] * n),
                                     (ctypes.c_void_p * n)(*[p["a"] for p in probs]),
                                     (ctypes.c_void_p * n)(*[p["s"] for p in probs]))
        assert m
        assert hip.nqs_hip_multi_use_persistent(m, on) == 0
        info = (SrInfo * n)()
        for _ in range(2):
            assert hip.nqs_hip_multi_step(m, info) == 0
        assert hip.nqs_hip_multi_sync(m) == 0
        out.append((info[0].as_dict(), r.params(probs[0]["a"])))
        hip.nqs_hip_multi_free(m)
        _free(hip, probs)
    for i, p in out[1:]:
        assert i == out[0][0]
        assert np.array_equal(p, out[0][1])


@pytest.mark.parametrize("on,tag,part", [(1, b"multi_cg", 0.47), (0, b"multi_gemm_z", 0.75)])
def test_few_samples_take_less(hip, monkeypatch, on, tag, part):
    """66049 parameters, an eighth of the samples: a third of an iteration's time
    in the cooperative launch, half of the row weights' as a launch (0.61 and
    0.98 where every workgroup went over all parameters for 16 samples)."""
    monkeypatch.setenv("NQS_HIP_MULTI_SPLIT", "64")
    r, us = scenarios.Runner(hip, "nqs_"), []
    for B in (512, 4096):
        p = _problem(hip, r, 256, 256, B, 256, 20, 3)
        p["cfg"].sr_cg_tol = 0.0
        m = hip.nqs_hip_multi_create(1, ctypes.byref(p["cfg"]), (ctypes.c_int * 1)(256), (ctypes.c_int * 1)(1),
                                     (ctypes.c_void_p * 1)(p["a"]), (ctypes.c_void_p * 1)(p["s"]))
        assert m
        assert hip.nqs_hip_multi_use_persistent(m, on) == 0
        hip.nqs_hip_multi_use_graph(m, 0)
        info, best = (SrInfo * 1)(), 1e9
        for _ in range(4):
            count, ms = ctypes.c_longlong(), ctypes.c_double()
            hip.nqs_hip_kernel_timing(tag)
            assert hip.nqs_hip_multi_step(m, info) == 0
            assert hip.nqs_hip_kernel_stats(tag, ctypes.byref(count), ctypes.byref(ms)) == 0
            hip.nqs_hip_kernel_timing(None)
            best = min(best, 1e3 * ms.value / info[0].cg_iterations)
        us.append(best)
        hip.nqs_hip_multi_free(m)
        _free(hip, [p])
    print("us an iteration:", us, flush=True)
    assert us[0] < part * us[1], us
