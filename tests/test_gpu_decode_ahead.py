"""The resident decode kernel of models of up to 2048 channels (decode_ahead.hip): order-faithful against the kernel sequence, bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

Q8, Q4, EXACT = 8, 2, 1


def same_bits(got, want):
    got, want = np.ascontiguousarray(got, np.float32), np.ascontiguousarray(want, np.float32)
    diff = got.view(np.uint32) != want.view(np.uint32)
    assert not diff.any(), f"{diff.sum()} of {diff.size} differ in bits; max abs err {np.max(np.abs(got - want)):.3e}"


def pair(fh, monkeypatch, cfg, seed):
    """(the kernel, the kernel sequence) over the same weights."""
    blob = fh.synth.make_weights_blob(cfg, seed=seed, threads=16)
    one = fh.HipModel(cfg, blob)
    monkeypatch.setenv("FORGE_HIP_PD_AHEAD", "0")
    seq = fh.HipModel(cfg, blob)
    monkeypatch.delenv("FORGE_HIP_PD_AHEAD")
    return one, seq


def shape(fh, wd, hidden, inter, heads, kv_heads, head_dim, vocab, layers=3, lm=None, max_seq=1024):
    cfg = fh.synth.tiny(wdtype=wd, max_seq=max_seq, hidden=hidden, inter=inter, layers=layers, heads=heads, kv_heads=kv_heads, head_dim=head_dim, vocab=vocab)
    return dict(cfg, flags=EXACT, lm_head_dtype=lm or wd)


# (format, hidden, inter, heads, kv heads, head dim, vocab, lm_head format): widths whose rows end inside a wave's and a workgroup's share, depths that are
# no multiple of a group of products (24) or of a norm accumulator's (12), the widest and the narrowest vectors, one wave's rows per matrix, a vocabulary of a
# few tiles and of a ragged number of them
SHAPES = {
    "smollm2": (Q8, 576, 1536, 9, 3, 64, 49152, None),
    "narrow": (Q8, 64, 64, 1, 1, 64, 100, None),
    "q4_ragged": (Q4, 608, 1056, 9, 1, 64, 4100, None),
    "widest": (Q8, 768, 2048, 8, 2, 96, 3004, Q4),
    "hd128": (Q4, 352, 736, 6, 2, 128, 1000, Q8),
    # the wide form: the 1B shape, one block of channels above the narrow form, ragged depths and few tiles
    "wide_1b": (Q8, 2048, 8192, 32, 8, 64, 8000, None),
    "wide_least": (Q4, 800, 1088, 12, 4, 64, 1000, Q8),
    "wide_hd128": (Q8, 1184, 3040, 9, 3, 128, 2052, Q4),
    "wide_hd96": (Q4, 1536, 4096, 16, 4, 96, 4000, None),
}


@pytest.mark.parametrize("name", sorted(SHAPES))
def test_equals_the_kernel_sequence(fh, torch_gpu, monkeypatch, name):
    """Contexts that end inside a block of 64 keys, at its last key and at the first of the next, with one and with several blocks: logits, greedy tokens, cache."""
    wd, *rest, lm = SHAPES[name]
    cfg = shape(fh, wd, *rest, layers=2 if name == "smollm2" else 3, lm=lm)
    one, seq = pair(fh, monkeypatch, cfg, 7)
    toks = fh.synth.uniform_ids(8, 400, cfg["vocab"])
    for n in (1, 60, 126, 380 if cfg["hidden"] <= 768 else 188):
        one.reset(); seq.reset()
        same_bits(one.forward_prefill(toks[:n]), seq.forward_prefill(toks[:n]))
        assert one.decode_launches == 1 and seq.decode_launches > 1
        for t in toks[n:n + 4]:
            assert one.forward_greedy(int(t)) == seq.forward_greedy(int(t))
        for t in toks[n + 4:n + 7]:
            same_bits(one.forward(int(t)), seq.forward(int(t)))
    for layer in range(cfg["layers"]):
        for which in (0, 1):
            assert np.array_equal(one.read_kv(layer, which), seq.read_kv(layer, which))
    one.close(); seq.close()


@pytest.mark.parametrize("hidden,head_dim,line", [(256, 64, 768), (256, 128, 768), (800, 64, 256)])
def test_across_its_last_context_with_a_penalty(fh, torch_gpu, monkeypatch, hidden, head_dim, line):
    """From the kernel to the sequence where the context outgrows a workgroup's blocks, and back after a reset, the repeat penalty's counts shared by both."""
    cfg = shape(fh, Q8, hidden, 512, 4, 2, head_dim, 1000)
    one, seq = pair(fh, monkeypatch, cfg, 17)
    toks = fh.synth.uniform_ids(18, 770, cfg["vocab"])
    for turn in range(2):
        for m in (one, seq):
            m.reset()
            m.set_repeat_penalty(1.3)
            m.forward_prefill(toks[:line - 4])
        t = 5
        for _ in range(8):
            a, b = one.forward_greedy(t), seq.forward_greedy(t)
            assert a == b
            t = a
        same_bits(one.forward(t), seq.forward(t))
    one.close(); seq.close()


@pytest.mark.parametrize("hidden", [256, 800])
def test_rewinds_its_tags_and_gives_up_instead_of_hanging(fh, torch_gpu, monkeypatch, hidden):
    """Tags that are about to wrap, and a poll limit of 1: a step that gave up has not happened and can be fed again."""
    cfg = shape(fh, Q8, hidden, 512, 4, 2, 64, 1000)
    monkeypatch.setenv("FORGE_HIP_PD_TAG_START", str(0xF0000000 - 40))
    one, seq = pair(fh, monkeypatch, cfg, 27)
    monkeypatch.delenv("FORGE_HIP_PD_TAG_START")
    toks = [int(t) for t in fh.synth.uniform_ids(28, 24, cfg["vocab"])]
    for m in (one, seq):
        m.set_repeat_penalty(1.2)
        m.forward_prefill(toks[:4])
    for t in toks[4:12]:
        assert one.forward_greedy(t) == seq.forward_greedy(t)
    one.set_poll_limit(1)
    failed = False
    for t in toks[12:18]:
        before = one.pos
        try:
            one.forward_greedy(t)
        except fh.ForgeHipError as e:
            assert e.code == fh.ERR_HIP and "gave up waiting" in str(e) and one.pos == before
            failed = True
            break
        seq.forward_greedy(t)
    assert failed, "no step gave up with a poll limit of 1"
    one.set_poll_limit(0)
    assert one.forward_greedy(t) == seq.forward_greedy(t)
    for t in toks[18:]:
        same_bits(one.forward(t), seq.forward(t))
    one.close(); seq.close()


@pytest.mark.parametrize("hidden,flags,prompt", [(256, EXACT, 30), (800, EXACT, 30), (800, 0, 300)])
def test_cooperative_launches(fh, torch_gpu, monkeypatch, hidden, flags, prompt):
    """FORGE_HIP_PD_COOP=1: the same tokens from launches that check residency."""
    cfg = dict(shape(fh, Q8, hidden, 512, 4, 4, 64, 1000), flags=flags)
    blob = fh.synth.make_weights_blob(cfg, seed=87)
    toks = fh.synth.uniform_ids(88, prompt, cfg["vocab"])
    plain = fh.HipModel(cfg, blob)
    monkeypatch.setenv("FORGE_HIP_PD_COOP", "1")
    coop = fh.HipModel(cfg, blob)
    assert coop.generate_greedy(toks, 12) == plain.generate_greedy(toks, 12)
    assert coop.decode_launches == plain.decode_launches == 1
    same_bits(coop.forward(3), plain.forward(3))
    coop.close(); plain.close()


@pytest.mark.parametrize("hidden", [256, 800])
def test_order_faithful_steps_that_give_up_run_as_the_sequence(fh, torch_gpu, monkeypatch, hidden):
    """Other users of the GPU do not make a step of the order-faithful mode fail: what gives up is the kernel sequence's, with its bits, until a poll limit is set."""
    cfg = shape(fh, Q8, hidden, 512, 4, 2, 64, 1000)
    monkeypatch.setenv("FORGE_HIP_PD_SPIN_LIMIT", "1")
    left = []
    toks = [int(t) for t in fh.synth.uniform_ids(78, 40, cfg["vocab"])]
    for first in ("greedy", "logits", "profile"):
        one, seq = pair(fh, monkeypatch, cfg, 77)
        for m in (one, seq):
            m.set_repeat_penalty(1.2)
            m.forward_prefill(toks[:6])
        assert one.decode_launches == 1
        at = 6
        for t in toks[6:12]:                                 # a step may get through if every hand-over is on time
            if first == "greedy":
                assert one.forward_greedy(t) == seq.forward_greedy(t)
            elif first == "logits":
                same_bits(one.forward(t), seq.forward(t))
            else:
                a, b = one.forward_profile(t), seq.forward_profile(t)
                if one.decode_launches > 1:
                    assert [n for _, n in a.values()] == [n for _, n in b.values()]
            at += 1
            if one.decode_launches > 1:
                break
        left.append(one.decode_launches)
        for t in toks[at:at + 6]:
            assert one.forward_greedy(t) == seq.forward_greedy(t) and one.pos == seq.pos
        one.set_poll_limit(0)
        assert one.decode_launches == 1
        for t in toks[at + 6:at + 10]:
            same_bits(one.forward(t), seq.forward(t))
        assert one.decode_launches == 1
        one.close(); seq.close()
    assert min(left) > 1, "no step gave up with a poll limit of 1"


@pytest.mark.parametrize("hidden", [256, 800])
def test_a_failed_step_keeps_the_count_that_the_other_kernel_made(fh, torch_gpu, monkeypatch, hidden):
    """Fast mode, a penalty: the token at position 0 is counted by decode_step_kernel's step, the one at position 1 is the first of decode_ahead_kernel, which gives up.
    The first count stays: without it the token, whose row of the output matrix is 64 times the others, would be the next one."""
    cfg = dict(shape(fh, Q8, hidden, 512, 4, 2, 64, 1000), flags=0)
    blob = fh.synth.make_weights_blob(cfg, seed=67)
    often, row = 7, hidden // 32 * 34
    blocks = blob[len(blob) - 1000 * row:][often * row:(often + 1) * row].reshape(-1, 34)
    blocks[:, :2] = (np.ascontiguousarray(blocks[:, :2]).view(np.float16) * np.float16(64)).view(np.uint8)
    one = fh.HipModel(cfg, blob)
    assert one.decode_launches == 1

    def after(x):
        one.reset()
        one.forward_greedy(often)
        return one.forward_greedy(x)

    x = next(x for x in range(500, 600) if after(x) == often)
    one.set_repeat_penalty(1000.0)
    want = after(x)
    assert want != often
    for _ in range(8):                                       # a step may get through if every hand-over is on time
        one.reset()
        one.forward_greedy(often)
        one.set_poll_limit(1)
        try:
            one.forward_greedy(often)
        except fh.ForgeHipError as e:
            assert "gave up waiting" in str(e) and one.pos == 1
            break
        finally:
            one.set_poll_limit(0)
    assert one.pos == 1, "no step gave up with a poll limit of 1"
    assert one.forward_greedy(x) == want
    one.close()


@pytest.mark.parametrize("name", ["narrow_form", "wide_1b", "wide_least", "wide_hd128"])
def test_fast_mode_takes_it_too(fh, oracle, torch_gpu, name):
    """Fast mode, token by token: the narrow form is the order-faithful one, the wide form adds up in another order.  Rounding moves single codes of the
    8-bit activations, which random weights amplify from layer to layer: two layers, and the loose bound that the other kernels' fast mode is held to."""
    wd, *rest, lm = SHAPES[name] if name in SHAPES else (Q8, 256, 512, 4, 2, 64, 1000, None)
    cfg = shape(fh, wd, *rest, layers=2, lm=lm)
    blob = fh.synth.make_weights_blob(cfg, seed=37, threads=16)
    fast, om = fh.HipModel(dict(cfg, flags=0), blob), oracle.Model(cfg, blob, 0, 1)
    toks = fh.synth.uniform_ids(38, 70, cfg["vocab"])
    fast.forward(int(toks[0])); om.forward(int(toks[0]))
    assert fast.decode_launches == 1
    for t in toks[1:]:
        a, b = fast.forward(int(t)), om.forward(int(t))
    assert np.all(np.isfinite(a)) and np.corrcoef(a, b)[0, 1] > 0.99
    # correlation sees neither scale nor offset.  Eight 8-bit vectors, 0.6% of the norm each and twice, over caches that differ as much
    assert np.linalg.norm(a - b) < 0.1 * np.linalg.norm(b)
    fast.close()


@pytest.mark.parametrize("name", ["narrow_form", "wide_1b", "wide_least", "wide_hd96", "wide_hd128"])
def test_short_contexts_of_fast_mode(fh, torch_gpu, monkeypatch, name):
    """Single steps from identical state, one layer, against decode_step_kernel: the bounds of test_longer_contexts_of_fast_mode."""
    wd, *rest, lm = SHAPES[name] if name in SHAPES else (Q8, 256, 512, 4, 2, 64, 1000, None)
    cfg = dict(shape(fh, wd, *rest, layers=1, lm=lm), flags=0)
    one, streamed = pair(fh, monkeypatch, cfg, 117)
    toks = fh.synth.uniform_ids(118, 260, cfg["vocab"])
    rel = []
    for n in (1, 2, 62, 63, 64, 126, 127, 128, 190, 191, 192, 253, 254):
        for m in (one, streamed):
            m.reset()
            m.forward_prefill_batch(toks[:n])
        a, b = one.forward(int(toks[n])), streamed.forward(int(toks[n]))
        assert one.decode_launches == 1 and np.all(np.isfinite(a))
        rel.append(np.linalg.norm(a - b) / np.linalg.norm(b))
    assert max(rel) < 2e-2 and np.median(rel) < 1e-5, rel
    one.close(); streamed.close()


@pytest.mark.parametrize("head_dim", [64, 96, 128])
@pytest.mark.parametrize("page_rows", [64, 256])
def test_narrow_models_over_pages(fh, torch_gpu, head_dim, page_rows):
    """Contexts across the edges of blocks and pages, up to the narrow form's last and past it: the flat cache's bits."""
    cfg = dict(shape(fh, Q8, 256, 512, 4, 2, head_dim, 1000), flags=0)
    blob = fh.synth.make_weights_blob(cfg, seed=127)
    flat, paged = fh.HipModel(cfg, blob), fh.HipModel(cfg, blob)
    paged.set_kv_pages(page_rows, np.random.default_rng(128).permutation(cfg["max_seq"] // page_rows).astype(np.uint32))
    toks = fh.synth.uniform_ids(129, 780, cfg["vocab"])
    for n in (1, 62, 127, 254, 510, 700, 764):
        for m in (flat, paged):
            m.reset()
            m.forward_prefill_batch(toks[:n])
        for t in toks[n:n + 6]:
            same_bits(paged.forward(int(t)), flat.forward(int(t)))
    for layer in range(cfg["layers"]):
        for which in (0, 1):
            assert np.array_equal(paged.read_kv(layer, which), flat.read_kv(layer, which))
    flat.close(); paged.close()


# (hidden, inter, heads, kv heads, head dim, contexts whose next steps cross a line): from the short form; from one round of requested keys to two and to three; from
# two rounds (two KV heads), five (10 splits) and six (heads of 128) to the other kernel.  Groups of 4, of 7 (waves with a second head) and of 3 heads, heads that fill their lanes and heads that do not
LONG = {"1b": (2048, 8192, 32, 8, 64, (254, 800, 2557, 5117)), "groups_of_7": (896, 4864, 14, 2, 64, (254, 318, 2557, 5117)),
        "hd96": (1536, 4096, 16, 4, 96, (254, 800, 1277, 2557)), "hd128": (1024, 3072, 12, 4, 128, (254, 318, 1277, 2557, 7677)), "splits_10": (800, 512, 24, 24, 64, (254, 798, 3997))}


@pytest.mark.parametrize("name", sorted(LONG))
def test_longer_contexts_of_fast_mode(fh, torch_gpu, monkeypatch, name):
    """Splits of the context: the same sums in another order, so outputs agree to rounding (a sum of
    a few thousand terms: 1e-5) unless a code of an 8-bit vector falls to its neighbour; each of the four vectors carries a rounding of 1/127 of a block's
    largest value, 0.6% of its norm, twice (both kernels'): under 2% of the output's."""
    hidden, inter, heads, kv_heads, hd, contexts = LONG[name]
    cfg = dict(shape(fh, Q8, hidden, inter, heads, kv_heads, hd, 1000, layers=1, max_seq=5248 if contexts[-1] < 5200 else 7808), flags=0)
    one, streamed = pair(fh, monkeypatch, cfg, 57)
    toks = fh.synth.uniform_ids(58, cfg["max_seq"] - 48, cfg["vocab"])
    rel = []
    for n in contexts:
        for m in (one, streamed):
            m.reset()
            m.forward_prefill(toks[:n])
        for t in toks[n:n + 5]:
            a, b = one.forward(int(t)), streamed.forward(int(t))
            assert one.decode_launches == 1 and np.all(np.isfinite(a))
            rel.append(np.linalg.norm(a - b) / np.linalg.norm(b))
    assert max(rel) < 2e-2 and np.median(rel) < 1e-5, rel
    # the same rows in pages all over the pool: the same bits
    paged = fh.HipModel(cfg, fh.synth.make_weights_blob(cfg, seed=57, threads=16))
    for page_rows, starts in ((64, (200, contexts[-1])), (128, (254, contexts[-2]))):
        paged.reset()
        paged.set_kv_pages(page_rows, np.random.default_rng(59).permutation(cfg["max_seq"] // page_rows).astype(np.uint32))
        for n in starts:
            for m in (one, paged):
                m.reset()
                m.forward_prefill(toks[:n])
            for t in toks[n:n + 3]:
                same_bits(paged.forward(int(t)), one.forward(int(t)))
    paged.close()
    # a step that gives up has not happened
    for m in (one, streamed):
        m.reset()
        m.forward_prefill(toks[:400])
    one.set_poll_limit(1)
    with pytest.raises(fh.ForgeHipError, match="gave up waiting"):
        for t in toks[400:410]:
            one.forward(int(t))
            streamed.forward(int(t))
    one.set_poll_limit(0)
    assert one.pos == streamed.pos
    a, b = one.forward(int(toks[420])), streamed.forward(int(toks[420]))
    assert np.linalg.norm(a - b) < 2e-2 * np.linalg.norm(b)
    one.close(); streamed.close()


# formats of q, k, v, o, gate, up, down and the lm_head, then hidden, inter, heads, kv heads, head dim: v of its own format at the edge of a wave's rows, all of one
# format, each format everywhere; depths whose last round of blocks is half a wave's
Q4K, Q6K = 12, 14
KQ = {"1b": ((Q4K, Q4K, Q6K, Q4K, Q4K, Q4K, Q6K), Q6K, 2048, 8192, 32, 8, 64), "all_q6": ((Q6K,) * 7, Q6K, 1024, 2048, 8, 4, 128), "all_q4": ((Q4K,) * 7, Q4K, 1536, 4096, 16, 4, 96),
      "turned": ((Q6K, Q6K, Q4K, Q6K, Q6K, Q6K, Q4K), Q4K, 1280, 2304, 20, 4, 64)}


@pytest.mark.parametrize("name", sorted(KQ))
def test_kquant_models_of_fast_mode(fh, torch_gpu, monkeypatch, name):
    """Single steps from identical state, one layer, against decode_step_kernel: the same whole sums and products of them, added up in another order, so the bounds of
    test_longer_contexts_of_fast_mode; over pages the same bits; a penalty's counts are both kernels'."""
    formats, lm, hidden, inter, heads, kv_heads, hd = KQ[name]
    cfg = dict(shape(fh, Q8, hidden, inter, heads, kv_heads, hd, 1004, layers=1, lm=lm, max_seq=2048), flags=0)
    blob = fh.synth.make_weights_blob_mixed(cfg, formats, seed=67, std=0.05)
    one = fh.HipModel(cfg, blob, proj_dtypes=formats)
    paged = fh.HipModel(cfg, blob, proj_dtypes=formats)
    monkeypatch.setenv("FORGE_HIP_PD_AHEAD", "0")
    streamed = fh.HipModel(cfg, blob, proj_dtypes=formats)
    monkeypatch.delenv("FORGE_HIP_PD_AHEAD")
    paged.set_kv_pages(128, np.random.default_rng(69).permutation(cfg["max_seq"] // 128).astype(np.uint32))
    toks = fh.synth.uniform_ids(68, 2000, cfg["vocab"])
    rel, differ = [], 0
    for n in (1, 63, 64, 190, 254, 255, 700, 1990):
        for m in (one, streamed, paged):
            m.reset()
            m.set_repeat_penalty(1.1)
            m.forward_prefill(toks[:n])
        for t in toks[n:n + 3]:
            a, b = one.forward(int(t)), streamed.forward(int(t))
            same_bits(paged.forward(int(t)), a)
            assert one.decode_launches == 1 and np.all(np.isfinite(a))
            rel.append(np.linalg.norm(a - b) / np.linalg.norm(b))
            differ += not np.array_equal(a, b)
        assert one.forward_greedy(5) == streamed.forward_greedy(5)
    assert max(rel) < 2e-2 and np.median(rel) < 1e-5, rel
    assert differ, "the same bits throughout: both ran the same kernel"
    one.close(); streamed.close(); paged.close()


@pytest.mark.parametrize("head_dim,which,channel", [(64, "v", 5), (96, "v", 5), (128, "v", 127), (96, "k", 95), (128, "k", 127)])
def test_an_infinite_value_in_the_first_row_of_a_long_context(fh, torch_gpu, monkeypatch, head_dim, which, channel):
    """The first row stands in for keys that are not there and its last channels for those past a head's: neither may count.  The first token's embedding has one channel, and
    one row of k or v is that channel alone, by a factor that takes it past what the 16-bit cache holds and leaves every other token's there."""
    hidden, heads, kv = 800, 4, 2
    cfg = dict(shape(fh, Q8, hidden, 512, heads, kv, head_dim, 1000, layers=1), flags=0)
    blob = fh.synth.make_weights_blob(cfg, seed=107)
    row, first, at = hidden // 32 * 34, 11, 3
    embed = blob[:1000 * hidden * 4].view(np.float32).reshape(1000, hidden)
    embed[first] = 0
    embed[first, at] = 1
    norm = blob[1000 * hidden * 4:][:hidden * 4].view(np.float32)
    matrix = 1001 * hidden * 4 + (heads * head_dim + (kv * head_dim if which == "v" else 0)) * row
    blocks = blob[matrix + channel * row:matrix + (channel + 1) * row].reshape(-1, 34)
    blocks[:] = 0
    blocks[0, :2] = np.array([1.4e5 / (127 * hidden ** 0.5 * abs(norm[at]))], np.float16).view(np.uint8)
    blocks[0, 2 + at] = 127
    one = fh.HipModel(cfg, blob)
    monkeypatch.setenv("FORGE_HIP_PD_AHEAD", "0")
    streamed = fh.HipModel(cfg, blob)
    toks = fh.synth.uniform_ids(108, 340, 1000)
    toks[toks == first] = 12
    toks[0] = first
    for m in (one, streamed):
        m.forward_prefill_batch(toks[:300])
    cached = one.read_kv(0, 0 if which == "k" else 1)
    cached = cached.view(np.float16).reshape(300, kv * head_dim)
    assert np.isinf(cached[0, channel]) and np.isfinite(cached[1:]).all()
    for t in toks[300:310]:
        a, b = one.forward(int(t)), streamed.forward(int(t))
        assert one.decode_launches == 1
        assert np.array_equal(np.isfinite(a), np.isfinite(b))
        if np.isfinite(b).all():
            assert np.linalg.norm(a - b) < 2e-2 * np.linalg.norm(b)
    one.close(); streamed.close()


@pytest.mark.parametrize("name,flags,prompt", [("smollm2", EXACT, 100), ("wide_1b", EXACT, 100), ("wide_1b", 0, 100), ("wide_1b", 0, 600), ("wide_hd128", 0, 600)])
def test_profile_gives_every_phase_its_time(fh, torch_gpu, name, flags, prompt):
    """The phases' times: none is shorter than a hand-over between workgroups takes (0.7 us measured; half of it is asked for), the merge of a long context
    is the quantise stage's, and they add up to what the kernel takes."""
    wd, *rest, lm = SHAPES[name]
    cfg = dict(shape(fh, wd, *rest, layers=4, lm=lm), flags=flags)
    m = fh.HipModel(cfg, fh.synth.make_weights_blob(cfg, seed=97, threads=16))
    m.forward_prefill_batch(fh.synth.uniform_ids(98, prompt, cfg["vocab"]))
    m.forward_profile(1)
    assert m.decode_launches == 1
    stages = {k: v for k, v in m.forward_profile(2).items() if v[1]}
    for stage, (ms, n) in stages.items():
        if stage == "quantize_act" and prompt < 256:
            assert ms == 0
        elif stage != "argmax":
            assert ms / n > 0.35e-3, (stage, ms, n)
    assert sum(ms for ms, _ in stages.values()) < 1.0
    m.close()


def test_models_of_several_threads_take_turns(fh, torch_gpu):
    """Two models step at the same time: each kernel needs the whole device, so their launches follow one another, and the tokens are those of a model alone."""
    import threading
    cfg = shape(fh, Q8, 256, 512, 4, 2, 64, 1000)
    blob = fh.synth.make_weights_blob(cfg, seed=47)
    prompt = fh.synth.uniform_ids(48, 30, cfg["vocab"])

    def generate(m):
        m.reset()
        return m.generate_greedy(prompt, 200)

    models = [fh.HipModel(cfg, blob) for _ in range(2)]
    want = generate(models[0])
    got = [None, None]

    def work(i):
        got[i] = generate(models[i])

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert got[0] == want and got[1] == want
    for m in models:
        m.close()
