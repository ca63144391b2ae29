"""Small dense products and solves: Grams whose 128 x 128 tiles leave CUs idle
(64 x 64 tiles) around the tile edges, inner lengths around the chunks of 32,
and triangular solves around the 64-, 256- and 512-row blocks."""
import numpy as np
import pytest

from spin_based_neural_network_amd.abi import ptr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,P", [(255, 64), (256, 64), (257, 65), (300, 95), (511, 97), (640, 300),
                                 (1921, 128)])
def test_gram(hip, B, P):
    print("gram:", B, P, flush=True)
    rng = np.random.default_rng(B + P)
    O = np.ascontiguousarray(rng.standard_normal((B, P)))
    T = np.zeros((B, B))
    assert hip.nqs_hip_gram(ptr(O), B, P, 1.0 / B, ptr(T)) == 0
    # P products of standard normals in one chain, on both sides
    assert np.abs(T - O @ O.T / B).max() <= 2.0 ** -53 * (P + 8) * 4 * P / B


@pytest.mark.parametrize("n", [1, 15, 63, 65, 127, 129, 255, 256, 257, 319, 320, 511, 513, 769, 1030])
def test_cholesky_solve(hip, n):
    print("solve:", n, flush=True)
    rng = np.random.default_rng(n)
    G = rng.standard_normal((n, n + 20))
    A = np.ascontiguousarray(G @ G.T / n + 0.1 * np.eye(n))
    b = rng.standard_normal(n)
    Aw, x = A.copy(), np.zeros(n)
    assert hip.nqs_hip_cholesky_solve(ptr(Aw), n, ptr(b), ptr(x)) == 1
    # normwise backward error of a Cholesky solve: a small multiple of n units
    # of |A| |x| (the blocks' inverses add their condition, here below 100)
    res = np.abs(A @ x - b).max()
    assert res <= 100 * 2.0 ** -53 * (n + 8) * np.linalg.norm(A, np.inf) * np.abs(x).max()
