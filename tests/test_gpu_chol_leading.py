"""The factor's leading block depends on the matrix's leading block alone, and
its bits with it: an element's sums are taken in the same order, and in the
same parts, in a factorisation of 8,704 rows as in one of 2,560, whatever
tiles the updates of the larger one take."""
import numpy as np
import pytest

import sopgpu as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [S.CHOL_BF16X3, S.CHOL_F32], ids=["split-bf16", "fp32"])
def test_leading_block(mode):
    n, k = 8704, 2560
    rng = np.random.default_rng(5)
    A = rng.standard_normal((n, n), dtype=np.float32) * np.float32(0.1 / np.sqrt(n))
    A = A + A.T
    A[np.arange(n), np.arange(n)] = 1.0
    print("case: orders %d and %d, mode %d" % (n, k, mode), flush=True)
    large = S.chol_factor(A, mode, 0)[0][:k, :k]
    small = S.chol_factor(np.ascontiguousarray(A[:k, :k]), mode, 0)[0]
    np.testing.assert_array_equal(large, small)
