"""The batched Crank-Nicolson solve at the edges of its segment counts (4, 8,
16 or 32 segments of 9 rows) and of a block's systems (needs an MI355X).

NY is the last row of one segment count and the first of the next, and the
shortest; the numbers of systems leave a block of every size partly empty.
The outer couplings sl[0] and su[ny-1] are non-zero here and must be dropped.
FP64 residuals ||Ax - b|| / ||b|| <= 1e-14 and FP32 <= 2e-6: the systems are
diagonally dominant with condition number < 50, so a stable solve leaves a
few roundings (2^-53, 2^-24) times that; a wrong neighbour, row or coupling
leaves O(1) in its rows."""
import numpy as np
import pytest
import torch

from diablo_amd import batched

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nsys", [1, 67])
@pytest.mark.parametrize("ny", [2, 36, 37, 72, 73, 144, 145, 288])
def test_cn_solve_at_segment_edges(ny, nsys):
    print(f"[batched] cn solve ny={ny} systems={nsys}", flush=True)
    sl, su = batched.cn_rows(ny)
    sl[0], su[ny - 1] = 0.7, 0.9
    sl[ny - 1], su[0] = 0.4, 0.3
    alpha, rhs = batched.cn_inputs(ny, nsys, 1)
    sl_d, su_d, al_d, b = (torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (sl, su, alpha, rhs))
    for fp32, bar in ((False, 1e-14), (True, 2e-6)):
        rhs_d = b.to(torch.complex64) if fp32 else b
        x = torch.empty_like(rhs_d)
        batched.cn_solve(sl_d, su_d, al_d, rhs_d, x, fp32=fp32)
        torch.cuda.synchronize()
        d = rhs_d.to(torch.complex128)
        r = batched.cn_matrix_apply(sl_d, su_d, al_d, x.to(torch.complex128)) - d
        res = (torch.linalg.vector_norm(r, dim=0) / torch.linalg.vector_norm(d, dim=0)).max()
        assert float(res) <= bar
