"""The blocked factorisation where its launches change: one 64-row block,
padding rows, a last panel narrower than the others, the tile sizes of the
next panel's and the trailing updates (128x64, 128x128, 256x256) and their
ragged last tiles.  L L^T against the matrix in FP64, and the one-stream
and two-stream schedules against each other bit for bit."""
import numpy as np
import pytest

import sopgpu as S

pytestmark = pytest.mark.gpu


def _matrix(n, seed):
    """A well-conditioned SPD matrix with entries of both signs everywhere."""
    import torch

    g = torch.Generator(device="cuda").manual_seed(seed)
    B = torch.randn(n, 96, generator=g, device="cuda", dtype=torch.float64)
    A = B @ B.T / 96.0
    A += torch.eye(n, device="cuda", dtype=torch.float64)
    return A.float()


@pytest.mark.parametrize("mode", [S.CHOL_BF16X3, S.CHOL_F32], ids=["bf16x3", "f32"])
@pytest.mark.parametrize("n", [1, 64, 65, 513, 577, 1088, 1700, 4001, 6913, 9025])
def test_factor_at_the_edges_of_its_launches(n, mode):
    import torch

    A = _matrix(n, 7 + n)
    mp = (n + 63) // 64 * 64
    buf = torch.full((mp, mp), float("nan"), device="cuda")
    buf[:n, :n] = A
    torch.cuda.synchronize()
    print("case: order %d, mode %d" % (n, mode), flush=True)
    rc = S.lib.sop_chol_factor_noalloc(0, n, buf.data_ptr(), mp, mode, torch.cuda.current_stream().cuda_stream)
    assert rc == 0, S.lib.sop_last_error()
    torch.cuda.synchronize()
    L = buf[:n, :n].tril()
    D = A.double()
    err = (torch.linalg.norm(L.double() @ L.double().T - D) / torch.linalg.norm(D)).item()
    print("case: order %d, mode %d: covariance error %.2e" % (n, mode, err), flush=True)
    assert err < 1e-5
    if n > 1:  # the upper triangle is left as it was
        assert torch.equal(buf[:n, :n].triu(1), A.triu(1))
    if n <= 7000:
        two, _ = S.chol_factor(A.cpu().numpy(), mode)
        np.testing.assert_array_equal(two, L.cpu().numpy())
