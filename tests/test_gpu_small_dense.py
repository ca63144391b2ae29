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


@pytest.mark.parametrize("o", [0, 64, 128, 512, 576])
@pytest.mark.parametrize("past", [1, 46, 300])
def test_panel_sum_order(hip, o, past):
    """The rank-16 updates inside a diagonal block: sums from zero over the even
    and over the odd columns, subtracted once.  Pivots of 1, so the factor's
    entries are those sums: 2^-53 is lost eight times over where it is added to
    a 1, and kept where its own sum is added."""
    print("panel sums:", o, past, flush=True)
    n = o + 18 + past
    A, w = np.eye(n), 2.0 ** -53
    A[o + 16, o:o + 16] = 1.0
    A[o + 16, o + 16] = 17.0
    A[o + 17, o:o + 16] = [1.0, w] + [0.0, w] * 7
    A[o + 17, o + 17] = A[o + 18, o + 18] = 64.0
    A[o + 18, o:o + 16] = -w
    A[o + 18, o + 16] = 1.0
    A = np.ascontiguousarray(A + np.tril(A, -1).T)
    x = np.zeros(n)
    assert hip.nqs_hip_cholesky_solve(ptr(A), n, ptr(np.ones(n)), ptr(x)) == 1
    assert np.array_equal(A[o + 16, o:o + 17], np.ones(17))
    assert A[o + 17, o + 16] == -(1.0 + 8 * w), float(A[o + 17, o + 16]).hex()
    assert A[o + 18, o + 16] == 1.0 + 16 * w, float(A[o + 18, o + 16]).hex()
