"""A prompt's rows in fast mode: the norm that keeps a row in registers, at the edges of its widths, and Q6_K products that read pairs of activation blocks twice, in each form of tile."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

Q8, Q6K, EXACT = 8, 14, 1


@pytest.mark.parametrize("hidden", [64, 1024, 1056, 2048, 2080, 4096, 4128, 8192, 8224])
def test_norm_of_prompt_rows(fh, torch_gpu, hidden):
    """One layer, fast against order-faithful mode.  Five vectors are rounded to 8 bits on the way (both norms, attention, feed-forward, final norm); the rounding of a block of normal
    values, whose largest of 32 is about 2.5 standard deviations, is 2.5 / 127 / sqrt(12) = 0.6 % of them, and where all codes come out otherwise two such errors stand against each
    other: 0.6 % * sqrt(2 * 5) = 1.8 %, times 1.7 for the blocks with larger ones.  A row, a weight or a tail taken wrongly is of the size of the result."""
    cfg = fh.synth.tiny(wdtype=Q8, max_seq=640, hidden=hidden, inter=64, layers=1, heads=2, kv_heads=1, head_dim=64, vocab=64)
    blob = fh.synth.make_weights_blob(cfg, seed=3, std=0.05)
    ids = fh.synth.uniform_ids(7, 33, 64)
    out = []
    for flags in (0, EXACT):
        cfg["flags"] = flags
        m = fh.HipModel(cfg, blob)
        out.append(np.asarray(m.forward_prefill(ids), np.float64))
        m.close()
    assert np.sqrt(((out[0] - out[1]) ** 2).mean()) <= 0.03 * np.sqrt((out[1] ** 2).mean())


@pytest.mark.parametrize("M,K,N", [(2, 256, 64), (33, 2048, 130), (65, 256, 2048), (200, 1024, 512), (300, 2048, 512), (700, 512, 1030), (1030, 8192, 300), (2000, 256, 2048)])
def test_q6_k_rows_against_their_order_faithful_form(fh, torch_gpu, M, K, N):
    """Only 32-bit sums are rounded: a step of the biased sums (12582912 times a block's scale S) by up to 0.75 S, 0.43 S rms, where these matrices' block sums are about 400 S: 1e-3 of the
    row's root mean square after any number of blocks, and 5e-3 is five times that."""
    rng = np.random.default_rng(M + K)
    raw = fh.synth.kquant_blocks(rng, Q6K, N * K // 256)
    w = fh.ops.QWeight(Q6K, raw, K, N)
    x = rng.normal(0, 1, (M, K)).astype(np.float32)
    x[M // 2, 32:64] = 0.0
    xd = torch_gpu.from_numpy(x).cuda()
    fast, exact = (fh.ops.matmul_mat_q(w, xd, f).cpu().numpy().astype(np.float64).reshape(M, N) for f in (0, EXACT))
    unit = np.abs(exact) + np.sqrt((exact ** 2).mean(axis=1, keepdims=True))
    assert np.all(np.abs(fast - exact) <= 5e-3 * unit)
