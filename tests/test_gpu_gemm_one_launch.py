"""matmul_mat for few rows in one launch: its workgroups quantise the activations for each other (gemm_rows.hip).  The bits are those of the
two launches that a result over a part of the activations takes, and that a graph records."""
import ctypes as C
import hashlib
import os
import subprocess
import sys

import numpy as np
import pytest

from test_gpu_ops import Q4, Q8, make_weight

pytestmark = pytest.mark.gpu

# both sides of every line of the rule: tiles, groups of 8 rows, pieces that end inside a row, one and two of them a wave, matrix sizes
SHAPES = [(1, 32, 33), (2, 2048, 8192), (8, 8192, 2048), (9, 8192, 96), (7, 608, 96), (8, 3072, 8192), (16, 2048, 100), (17, 2048, 100), (16, 3072, 1024), (31, 544, 1000), (32, 2048, 2048), (33, 576, 576),
          (40, 96, 4100), (128, 2048, 2048), (130, 416, 2100), (200, 576, 1536)]


def _overlapping(fh, torch, w, x, M, K, N):
    """The result, begun in the last element of a copy of the activations: two launches."""
    buf = torch.empty(M * K + M * N, device="cuda")
    buf[:M * K] = x.view(-1)
    y = buf[M * K - 1:M * K - 1 + M * N]
    fh.check(fh.lib().forge_hip_gemm_q(w._h, C.c_void_p(buf.data_ptr()), M, C.c_void_p(y.data_ptr()), 0, C.c_void_p(torch.cuda.current_stream().cuda_stream)))
    return y.clone().view(M, N)


def _run(fh, torch, wd):
    digest = hashlib.sha256()
    for M, K, N in SHAPES:
        w = fh.ops.QWeight(wd, make_weight(fh, wd, N, K, M + K + N), K, N)
        for seed in range(3):                        # other activations in the same scratch, one after the other
            x = torch.randn(M, K, generator=torch.Generator().manual_seed(seed)).cuda() * 10.0 ** (seed - 1)
            one, two = fh.ops.matmul_mat_q(w, x), _overlapping(fh, torch, w, x, M, K, N)
            assert torch.equal(one.view(torch.int32), two.view(torch.int32)), (M, K, N, seed)
            digest.update(one.cpu().numpy().tobytes())
        w.close()
    return digest.hexdigest()


@pytest.mark.parametrize("wd", [Q8, Q4])
def test_one_launch_has_the_bits_of_two(fh, torch_gpu, wd):
    _run(fh, torch_gpu, wd)


@pytest.mark.parametrize("wd", [Q8, Q4])
def test_a_wait_that_ends_early_costs_time_only(fh, torch_gpu, wd):
    """Pieces that are not there when the wait ends are quantised by everybody who misses them: the same bits."""
    code = "import sys; sys.path[:0] = %r\nimport torch\nfrom __graft_entry__ import load_package\nimport test_gpu_gemm_one_launch as t\nprint(t._run(load_package(), torch, %d))" % (
        [os.path.dirname(os.path.abspath(__file__)), os.path.dirname(os.path.dirname(os.path.abspath(__file__)))], wd)
    r = subprocess.run([sys.executable, "-c", code], env=dict(os.environ, FORGE_HIP_PD_SPIN_LIMIT="1"), capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr
    assert r.stdout.split()[-1] == _run(fh, torch_gpu, wd)


def test_recorded_into_a_graph(fh, torch_gpu):
    torch = torch_gpu
    M, K, N = 16, 2048, 2048
    w = fh.ops.QWeight(Q4, make_weight(fh, Q4, N, K, 5), K, N)
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


def test_rows_with_infinities_and_no_number(fh, torch_gpu):
    torch = torch_gpu
    M, K, N = 5, 64, 40
    w = fh.ops.QWeight(Q8, make_weight(fh, Q8, N, K, 6), K, N)
    x = torch.randn(M, K)
    x[1, 3], x[2, 40], x[3, 7], x[4] = torch.inf, torch.nan, 1e-42, 0.0
    x = x.cuda()
    one, two = fh.ops.matmul_mat_q(w, x).cpu().numpy(), _overlapping(fh, torch, w, x, M, K, N).cpu().numpy()
    assert np.array_equal(one.view(np.uint32), two.view(np.uint32))
    w.close()
