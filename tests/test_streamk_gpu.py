"""fp32 products whose last round has fewer stream-K steps than workgroups
(few tiles past the whole rounds, short K): every output against float64."""
import numpy as np
import pytest

from test_kat_gpu import U, gemm, kat  # noqa: F401 (kat is the fixture)

pytestmark = pytest.mark.gpu


# 786 tiles (18 past three rounds of 256) of 8 steps and 516 (4 past two) of 32;
# 530 tiles, whose last 18 x 24 steps do fill the 256 workgroups
@pytest.mark.parametrize("M,N,K", [(132, 50257, 256), (257, 21900, 1024), (1280, 6700, 768)])
def test_few_steps_past_the_whole_rounds(kat, M, N, K):  # noqa: F811
    rng = np.random.default_rng(K)
    X = rng.standard_normal((M, K)).astype(np.float32)
    W = rng.standard_normal((N, K)).astype(np.float32)
    b = np.zeros(N, np.float32)
    # what an unwritten partial slot would add: the previous product's tiles
    gemm(kat, X, W, b, M, N, K, 0, 0)
    Y = gemm(kat, X, W, b, M, N, K, 0, 0)
    rows = np.r_[0:M:17, M - 1]
    want = X[rows].astype(np.float64) @ W.T.astype(np.float64)
    mag = np.abs(X[rows]).astype(np.float64) @ np.abs(W).T.astype(np.float64)
    assert (np.abs(Y[rows] - want) <= (K + 4) * U * mag).all()
