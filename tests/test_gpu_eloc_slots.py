"""Real-RBM local energies of device batches against the oracle at the edges of
the term octets and tiles: groups of one (flips), two and four terms that share
a site, octets with empty slots, hidden units around the tile of 8 and the
rescaling groups of 4, samples around one and two a lane, FP32.  The FP32
bound is the oracle's own formula evaluated with 2^-24 in each of the M
factors and in theta."""
import ctypes
import time

import numpy as np
import pytest

import scenarios
from spin_based_neural_network_amd.abi import config_defaults, fnptr, options_defaults, ptr

pytestmark = pytest.mark.gpu

RBM, TFIM, HEIS, J1J2, KAGOME = 5, 0, 1, 2, 6


@pytest.mark.parametrize("ham,Lx,Ly,per,M,B,scale", [
    (TFIM, 3, 1, 1, 1, 1, 0.3), (TFIM, 9, 1, 0, 7, 63, 0.5), (TFIM, 16, 1, 1, 33, 4096, 0.2),
    (HEIS, 3, 1, 0, 8, 64, 0.5), (HEIS, 4, 4, 1, 9, 65, 0.4), (HEIS, 5, 7, 0, 31, 129, 2.0),
    (J1J2, 3, 3, 1, 4, 200, 0.3), (J1J2, 6, 6, 1, 12, 7400, 0.3), (J1J2, 8, 8, 1, 130, 70, 0.2),
    (KAGOME, 2, 2, 1, 16, 127, 0.4), (KAGOME, 2, 3, 0, 5, 128, 4.0),
])
@pytest.mark.parametrize("precision", [0, 1])
def test_real_local_energies(hip, orc, ham, Lx, Ly, per, M, B, scale, precision):
    print("real E_loc:", ham, Lx, Ly, per, M, B, scale, precision, flush=True)
    N = 3 * Lx * Ly if ham == KAGOME else Lx * Ly
    cfg = config_defaults(ansatz=RBM, hamiltonian=ham, rbm_hidden_units=M, rbm_init_scale=scale,
                          j2_coupling=0.5, transverse_field=0.7, rng_seed=41 + M, kagome_pbc=per)
    ah, ao = hip.nqs_ansatz_create(ctypes.byref(cfg), N), orc.orc_ansatz_create(ctypes.byref(cfg), N)
    s = scenarios.spins_random(B, N, 5 + N, sz0=False)
    e = [np.zeros(B) for _ in range(4)]
    opt = options_defaults(periodic=per, precision=precision)
    assert hip.nqs_hip_local_energy_batch_ex(ctypes.byref(cfg), Lx, Ly, ctypes.byref(opt), ptr(s), B,
                                             fnptr(hip, "nqs_ansatz_log_amp"), ah, ptr(e[0]),
                                             ptr(e[1])) == 0
    orc.orc_local_energy_batch_ex(ctypes.byref(cfg), Lx, Ly, per, ptr(s), B,
                                  fnptr(orc, "orc_ansatz_log_amp"), ao, ptr(e[2]), ptr(e[3]))
    unit = 2.0 ** -24 if precision else 2.0 ** -53
    # theta is a sum of N + 1 terms of size `scale`, a ratio a product of M
    # factors; the oracle differences two log amplitudes of size M theta
    tol = 16 * unit * (M + 4) * (1.0 + scale * (N + 1)) * max(1.0, np.abs(e[2]).max())
    assert np.abs(e[0] - e[2]).max() <= tol, (np.abs(e[0] - e[2]).max(), tol)
    assert not e[1].any()
    hip.nqs_ansatz_free(ah)
    orc.orc_ansatz_free(ao)


@pytest.mark.parametrize("kind", [RBM, 6])
def test_alternating_hamiltonians(hip, kind):
    """Two Hamiltonians in turn cost a caller their upload (about 0.1 ms for 1024
    pairs), not a millisecond of grouping terms on the host at every call."""
    L, B = 16, 1
    cfgs = [config_defaults(ansatz=kind, hamiltonian=J1J2, rbm_hidden_units=2, rbm_init_scale=0.1,
                            j2_coupling=j2, rng_seed=3) for j2 in (0.4, 0.5)]
    a = hip.nqs_ansatz_create(ctypes.byref(cfgs[0]), L * L)
    s = scenarios.spins_random(B, L * L, 5, sz0=True)
    e, opt = [np.zeros(B), np.zeros(B)], options_defaults(periodic=1)

    def call(cfg):
        t = time.perf_counter()
        assert hip.nqs_hip_local_energy_batch_ex(ctypes.byref(cfg), L, L, ctypes.byref(opt), ptr(s), B,
                                                 fnptr(hip, "nqs_ansatz_log_amp"), a, ptr(e[0]),
                                                 ptr(e[1])) == 0
        return time.perf_counter() - t

    same = min(call(cfgs[0]) for _ in range(40))
    turn = min(call(cfgs[i & 1]) for i in range(1, 41))
    hip.nqs_ansatz_free(a)
    print("same / in turn:", same, turn, flush=True)
    assert turn - same < 2.5e-4, (same, turn)
