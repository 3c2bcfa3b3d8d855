"""matmul_mat for few rows of deep matrices: K in ranges over workgroups that meet in memory (gemm_rows.hip), at the edges of the rule and of the ranges."""
import numpy as np
import pytest

from test_gpu_ops import EXACT, Q4, Q8, make_weight

pytestmark = pytest.mark.gpu

# four, two and one range; a last tile of each number of row groups; ragged columns; depths whose steps don't divide by the ranges, an odd number of blocks
SHAPES = [(2, 8192, 2048), (8, 8192, 2048), (9, 8192, 2048), (31, 8192, 2080), (32, 8192, 4096), (32, 8192, 4097), (33, 8192, 2048), (64, 8192, 2048), (64, 8192, 2049), (65, 8192, 2048),
          (17, 8224, 33), (40, 8256, 100), (5, 16384, 40), (3, 8160, 64)]


@pytest.mark.parametrize("wd", [Q8, Q4])
@pytest.mark.parametrize("M,K,N", SHAPES)
def test_against_the_order_faithful_form(fh, torch_gpu, wd, M, K, N):
    """Block sums are the same integers: 1e-3 of |value| + the row's root mean square for the order of the 32-bit sums, as for every product in fast mode; and which range arrives last changes no bit."""
    torch = torch_gpu
    w = fh.ops.QWeight(wd, make_weight(fh, wd, N, K, M + K + N), K, N)
    x = torch.randn(M, K, generator=torch.Generator().manual_seed(M)).cuda()
    want = fh.ops.matmul_mat_q(w, x, EXACT).cpu().numpy().astype(np.float64)
    first = fh.ops.matmul_mat_q(w, x).cpu().numpy()
    unit = np.abs(want) + np.sqrt((want ** 2).mean(axis=1, keepdims=True))
    assert np.all(np.abs(first - want) <= 1e-3 * unit)
    for _ in range(4):
        assert np.array_equal(fh.ops.matmul_mat_q(w, x).cpu().numpy(), first)
    w.close()


def test_recorded_into_a_graph(fh, torch_gpu):
    torch = torch_gpu
    M, K, N = 20, 8192, 2048
    w = fh.ops.QWeight(Q8, make_weight(fh, Q8, N, K, 5), K, N)
    x = torch.randn(M, K, device="cuda")
    fh.ops.matmul_mat_q(w, x)                        # the scratch is there
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        y = fh.ops.matmul_mat_q(w, x)
    for seed in range(4):
        x.copy_(torch.randn(M, K, generator=torch.Generator().manual_seed(seed)))
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, fh.ops.matmul_mat_q(w, x)), seed
    w.close()
