"""The resident decode kernel of small bfloat16 block networks: against the 64-bit oracle at the edges of what its registers hold and of how it shares out a context, against the kernel
sequence where the oracle would take too long, and what it does when a step is given up."""
import numpy as np
import pytest

from folder_model import Case, check

pytestmark = pytest.mark.gpu


def configs(fh):
    s = fh.synth
    lay, vab = s.vabirax_layer, s.vabirax_config
    att, gla, kak = s.kakirax_attention, s.kakirax_gla, s.kakirax_config
    return {
        # latent attention: heads dim rot vdim q_rank kv_rank ff window
        "latent_largest": ("vabirax_oracle", vab(768, 70, [lay(5, 64, 32, 64, 192, 128, 1536, 130)] * 2, loop=(0, 1, 2))),
        "latent_ragged": ("vabirax_oracle", vab(90, 203, [lay(3, 20, 6, 44, 50, 70, 77, None, rot_dims=4)] * 3, loop=(1, 2, 2), embedding_scale=1.7, eps=3e-3)),
        "latent_many_heads": ("vabirax_oracle", vab(64, 80, [lay(24, 32, 32, 32, 33, 64, 51, None)] * 2)),
        # linear (heads dim vdim ff) and grouped attention (heads kv_heads dim vdim ff)
        "mixed_largest": ("kakirax_oracle", kak(768, 70, [gla(6, 64, 128, 1536), att(12, 3, 64, 64, 1536), 0], embedding_scale=20.0)),
        "mixed_ragged": ("kakirax_oracle", kak(90, 203, [gla(5, 20, 60, 77, tau=3.0), att(6, 2, 20, 44, 77, rot_dims=12), 0, 1], embedding_scale=9.5, eps=3e-3, cap=7.0)),
        "grouped_many_heads": ("kakirax_oracle", kak(64, 80, [att(24, 24, 32, 32, 51)] * 2, embedding_scale=8.0)),
        # layers that registers do not hold: the wide form
        "wide_largest": ("kakirax_oracle", kak(2048, 70, [gla(16, 64, 128, 8192), att(32, 8, 64, 64, 8192)], embedding_scale=45.0)),
        "wide_ragged": ("kakirax_oracle", kak(1000, 203, [gla(5, 20, 60, 2077, tau=3.0), att(6, 2, 20, 44, 2077, rot_dims=12), 0, 1], embedding_scale=9.5, eps=3e-3, cap=7.0)),
        "wide_deep": ("kakirax_oracle", kak(90, 80, [att(24, 24, 32, 32, 1601), gla(48, 16, 32, 1601), 0], embedding_scale=8.0)),
        # records of parts over many waves' strips of LDS; more parts than linear heads
        "grouped_few_heads": ("kakirax_oracle", kak(64, 80, [att(9, 3, 64, 64, 51)] * 3, embedding_scale=8.0)),
        "mixed_few_heads": ("kakirax_oracle", kak(64, 80, [att(12, 3, 64, 64, 51), gla(2, 32, 32, 51), 0, 0], embedding_scale=8.0)),
        "wide_few_heads": ("kakirax_oracle", kak(90, 80, [att(8, 2, 64, 64, 1601), 0, gla(2, 32, 32, 1601), 0], embedding_scale=8.0)),
        # an odd number of heads of 32 values: rows of the input product that no head reads
        "latent_odd": ("vabirax_oracle", vab(64, 61, [lay(3, 32, 32, 32, 64, 64, 51, None)] * 2)),
        "grouped_odd": ("kakirax_oracle", kak(64, 61, [att(3, 1, 32, 32, 51)] * 2, embedding_scale=8.0)),
        "wide_odd": ("kakirax_oracle", kak(64, 61, [gla(3, 32, 32, 1601), att(3, 1, 32, 32, 1601)], embedding_scale=8.0)),
        "linear_only": ("kakirax_oracle", kak(70, 61, [gla(3, 16, 32, 40), 0], embedding_scale=8.0)),
    }


@pytest.fixture(scope="module")
def get(fh, torch_gpu, tmp_path_factory):
    made, known = {}, configs(fh)

    def case(name):
        if name not in made:
            print("case", name, flush=True)
            oracle, cfg = known[name]
            tensors = None
            if oracle == "kakirax_oracle":           # a rank of the decays' maps that the kernel covers
                tensors = fh.synth.folder_tensors(cfg, 5, fh.synth.kakirax_shapes(cfg, 11))
            made[name] = Case(fh, getattr(__import__("oracle." + oracle), oracle), tmp_path_factory.mktemp(name), cfg, tensors)
        return made[name]
    return case


@pytest.mark.parametrize("name", ["latent_largest", "latent_ragged", "latent_many_heads", "mixed_largest", "mixed_ragged", "grouped_many_heads", "linear_only", "wide_largest", "wide_ragged", "wide_deep"])
def test_against_the_oracle(get, name):
    """Token by token over the first tiles of keys, the window's edge and the change from one workgroup a head to parts (384 keys)."""
    c = get(name)
    ids = c.ids(400, seed=3)
    want = c.oracle.forward(ids)[0]
    scale = np.sqrt((want ** 2).mean())
    m = c.model(max_seq=400, dtype="bfloat16")
    for start, steps in ((1, 37), (120, 15), (376, 24)):
        m.reset()
        m.forward_prefill(ids[:start])
        assert m.decode_launches == 1
        got = np.stack([m.forward(int(t)) for t in ids[start:start + steps]])
        check(got, want[start:start + steps], "bfloat16", scale)
        assert m.pos == start + steps and m.decode_launches == 1          # no step was given up
    m.close()


@pytest.mark.parametrize("name", ["latent_many_heads", "grouped_many_heads", "wide_deep"])
def test_contexts_of_several_rounds(get, name, monkeypatch):
    """24 heads leave each eight or nine workgroups of twelve waves of 32 keys: four waves, eight, twelve, and a second round.  The wide form: ten of four waves, up to three rounds."""
    c = get(name)
    ids = c.ids(3700, seed=4)
    m = c.model(max_seq=3700, dtype="bfloat16")
    monkeypatch.setenv("FORGE_HIP_PERSIST", "0")
    sequence = c.model(max_seq=3700, dtype="bfloat16")
    for start in (640, 1500, 2600, 3690):
        for x in (m, sequence):
            x.reset()
            x.forward_prefill(ids[:start])
        assert m.decode_launches == 1 and sequence.decode_launches > 1
        for t in ids[start:start + 3]:
            check(m.forward(int(t)), sequence.forward(int(t)).astype(np.float64), "bfloat16")
        assert m.decode_launches == 1
    m.close()
    sequence.close()


@pytest.mark.parametrize("name", ["grouped_few_heads", "mixed_few_heads", "wide_few_heads"])
def test_parts_over_the_strips_of_all_waves(get, name, monkeypatch):
    """A key / value head's parts, up to 64 of them, lie where its workgroup's waves keep transposed values: at four, eight and twelve waves that attend (up to 8192 rows of context, up to 16384,
    beyond) the records reach the strips of waves without a part in adding them up, which are free for the next layer at once."""
    c = get(name)
    ids = c.ids(16700, seed=7)
    m = c.model(max_seq=16700, dtype="bfloat16")
    monkeypatch.setenv("FORGE_HIP_PERSIST", "0")
    sequence = c.model(max_seq=16700, dtype="bfloat16")
    for start in (1300, 2700, 8300, 16500):
        for x in (m, sequence):
            x.reset()
            x.forward_prefill(ids[:start])
        assert m.decode_launches == 1 and sequence.decode_launches > 1
        for t in ids[start:start + 12]:
            check(m.forward(int(t)), sequence.forward(int(t)).astype(np.float64), "bfloat16")
        assert m.decode_launches == 1
    m.close()
    sequence.close()


@pytest.mark.parametrize("name", ["latent_odd", "grouped_odd", "linear_only", "wide_odd"])
def test_rows_that_no_head_reads(get, name, monkeypatch):
    """The last rows of an input product pad it; no workgroup has only those to do (none would wait for it, and it would find its own input overwritten and give up)."""
    c = get(name)
    ids = c.ids(500, seed=11)
    m = c.model(max_seq=500, dtype="bfloat16")
    monkeypatch.setenv("FORGE_HIP_PERSIST", "0")
    sequence = c.model(max_seq=500, dtype="bfloat16")
    for x in (m, sequence):
        x.forward_prefill(ids[:2])
    assert m.decode_launches == 1 and sequence.decode_launches > 1
    for t in ids[2:]:
        check(m.forward(int(t)), sequence.forward(int(t)).astype(np.float64), "bfloat16")
    assert m.decode_launches == 1
    m.close()
    sequence.close()


@pytest.mark.parametrize("ff", [51, 1601])
def test_a_normed_row_beyond_bfloat16(fh, torch_gpu, tmp_path, ff, monkeypatch):
    """An element of a normed row between bfloat16's largest number and 32-bit's is finite in the kernel sequence's 32-bit row, and would be no number in its planes: the model keeps the sequence.
    Everything but the gates is blind to it, and they close."""
    from oracle import kakirax_oracle
    s, c = fh.synth, 3
    cfg = s.kakirax_config(64, 61, [s.kakirax_gla(2, 32, 32, ff), s.kakirax_attention(2, 1, 32, 32, ff)])
    t = s.folder_tensors(cfg, 5)
    t["embed"][:, c] = s.to_bf16([1.0])                                  # the same for all tokens, nearly so when normed
    for name in ("q", "k", "v", "a1", "g"):
        t["l0.mix." + name][:, c] = s.to_bf16([-1.0 if name == "g" else 0.0])
    x = s.from_bf16(t["embed"]).astype(np.float64)
    z = (x[:, c] - x.mean(1)) / np.sqrt(x.var(1) + 1e-5)
    t["l0.norm1"][c:c + 1], t["l0.norm1.b"][c] = s.to_bf16([1.0e36 / np.median(z)]), 0x7F7F
    y = z * s.from_bf16(t["l0.norm1"][c]) + s.from_bf16(t["l0.norm1.b"][c])
    ids = np.flatnonzero((y > 3.3965e38) & (y < 3.402e38))
    assert ids.size >= 20
    case = Case(fh, kakirax_oracle, tmp_path, cfg, t)
    m = case.model(dtype="bfloat16")
    monkeypatch.setenv("FORGE_HIP_PERSIST", "0")
    sequence = case.model(dtype="bfloat16")
    for i, token in enumerate(ids):
        got, want = m.forward(int(token)), sequence.forward(int(token))
        assert m.decode_launches == sequence.decode_launches > 1
        check(got, want.astype(np.float64), "bfloat16")
    m.close()
    sequence.close()


@pytest.mark.parametrize("name,at", [("latent_ragged", "head"), ("latent_ragged", "l1.mix.uk"), ("latent_ragged", "loop.in"), ("latent_ragged", "l2.norm1.b"), ("latent_ragged", "l0.mix.dkv.norm"),
                                     ("mixed_ragged", "l0.mlp.down"), ("mixed_ragged", "l0.mix.norm"), ("mixed_ragged", "l1.norm2"), ("wide_ragged", "l1.mix.o"), ("wide_ragged", "l1.mix.k.norm")])
def test_weights_of_any_size(get, name, at, tmp_path):
    """A model with a weight past 2^32, infinite or NaN keeps the kernel sequence; one with a weight of 2^32 does not."""
    c = get(name)
    for value, one in ((0x7F80, False), (0xFF80, False), (0x7FC0, False), (0x7F7F, False), (0xCF81, False), (0x4F80, True), (0xCF80, True)):
        t = dict(c.tensors)
        t[at] = t[at].copy()
        t[at].reshape(-1)[-1] = value
        c.fh.synth.write_model_folder(str(tmp_path), c.cfg, t)
        m = c.fh.HipModel.from_folder(str(tmp_path), 16, "bfloat16")
        m.forward(1)
        assert (m.decode_launches == 1) == one, hex(value)
        m.close()


def bits(x):
    return x.view(np.uint32)


@pytest.mark.parametrize("name", ["latent_ragged", "mixed_ragged", "wide_ragged"])
def test_a_step_that_is_given_up(get, fh, name, monkeypatch):
    """With a poll limit of 1 a step that gives up has not happened, states of linear layers included; with the library's own limit it runs as the kernel sequence.  Tags wrap."""
    c = get(name)
    ids = c.ids(40, seed=6)
    plain = c.model(dtype="bfloat16")
    monkeypatch.setenv("FORGE_HIP_PD_TAG_START", str(0xF0000000 - 40))
    m = c.model(dtype="bfloat16")
    monkeypatch.delenv("FORGE_HIP_PD_TAG_START")
    for x in (plain, m):
        x.forward_prefill(ids[:9])
    failed = 0
    for t in ids[9:]:
        before = m.pos
        m.set_poll_limit(1)
        for _ in range(3):
            try:
                got = m.forward(int(t))
                break
            except fh.ForgeHipError as e:
                assert e.code == fh.ERR_HIP and "gave up waiting" in str(e) and m.pos == before
                failed += 1
        else:
            m.set_poll_limit(0)
            got = m.forward(int(t))
        assert np.array_equal(bits(got), bits(plain.forward(int(t))))
    assert failed, "no step gave up with a poll limit of 1"
    m.close()
    monkeypatch.setenv("FORGE_HIP_PERSIST", "0")
    sequence = c.model(dtype="bfloat16")
    monkeypatch.delenv("FORGE_HIP_PERSIST")
    monkeypatch.setenv("FORGE_HIP_PD_SPIN_LIMIT", "1")
    m = c.model(dtype="bfloat16")
    for x in (sequence, m):
        x.forward_prefill(ids[:9])
    same = 0
    for t in ids[9:]:
        left = m.decode_launches > 1
        a, b = m.forward(int(t)), sequence.forward(int(t))
        check(a, b.astype(np.float64), "bfloat16")
        same += left and m.decode_launches == sequence.decode_launches
    assert same, "no step gave up with a poll limit of 1"
    for x in (plain, sequence, m):
        x.close()


@pytest.mark.parametrize("name", ["latent_ragged", "mixed_ragged", "wide_ragged"])
def test_greedy_with_a_repeat_penalty(get, fh, name):
    """The token that a greedy step returns is the last maximum of the penalised logits of the same step."""
    c = get(name)
    ids = c.ids(6, seed=8)
    a, b = c.model(dtype="bfloat16"), c.model(dtype="bfloat16")
    b.set_repeat_penalty(1.7)
    for x in (a, b):
        x.forward_prefill(ids)
    fed, token = list(ids), 5
    for _ in range(30):
        fed.append(token)
        p = a.forward(token).copy()
        fh.ops.apply_repeat_penalty(p, np.array(fed, np.uint32), 1.7)
        token = b.forward_greedy(token)
        assert token == p.size - 1 - int(np.argmax(p[::-1]))
    a.close()
    b.close()
