"""Prompts of block networks whose products reach each form of tile and the depth in ranges, at the edges of the rules that choose them, against the 64-bit restatement."""
import numpy as np
import pytest

from folder_model import DTYPES, Case, check

pytestmark = pytest.mark.gpu


def configs(fh):
    s = fh.synth
    return {
        # every epilogue, sizes that no tile divides: tiles of 32 x 32 throughout
        "ragged": ("vabirax_oracle", s.vabirax_config(200, 150, [s.vabirax_layer(5, 20, 6, 44, 50, 70, 333, None, rot_dims=4)] * 2)),
        # 8192 rows of [gate; up]: the edges between 32 x 32, 64 x 32 and larger tiles; a depth of 4096 in 8 ranges
        "broad": ("kakirax_oracle", s.kakirax_config(256, 70, [s.kakirax_attention(4, 2, 32, 32, 4096)], embedding_scale=16.0)),
        # ranges by tiles of 64 x 32 (up to 160 rows), 64 x 64 (up to 512) and 128 x 128, and residual tiles of 32 x 64 (from 1025, the shallow product)
        "deep": ("kakirax_oracle", s.kakirax_config(1024, 70, [s.kakirax_attention(4, 2, 32, 32, 4096)], embedding_scale=32.0)),
        # the depth's stages don't divide by the ranges
        "odd_depth": ("kakirax_oracle", s.kakirax_config(130, 70, [s.kakirax_attention(4, 2, 32, 32, 4200)], embedding_scale=11.0)),
    }


@pytest.fixture(scope="module")
def get(fh, torch_gpu, tmp_path_factory):
    made, known = {}, configs(fh)

    def case(name):
        if name not in made:
            oracle, cfg = known[name]
            c = Case(fh, getattr(__import__("oracle." + oracle), oracle), tmp_path_factory.mktemp(name), cfg)
            most = 1030 if name == "deep" else 330
            made[name] = c, c.ids(most, seed=4), {}
        return made[name]
    return case


ROWS = {"ragged": (2, 31, 32, 33, 65, 200), "broad": (32, 33, 64, 65, 96, 97, 129, 320, 321), "deep": (33, 160, 161, 512, 513, 1030), "odd_depth": (2, 70)}


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name,rows", [(n, r) for n, rs in ROWS.items() for r in rs])
def test_prompt(get, name, rows, dtype):
    c, ids, known = get(name)
    if "all" not in known:
        known["all"] = c.oracle.forward(ids)[0]
    want = known["all"][:rows]
    scale = np.sqrt((known["all"] ** 2).mean())
    at = np.unique(np.linspace(0, rows - 1, min(rows, 64)).astype(int))
    m = c.model(max_seq=1030, dtype=dtype)
    first = m.prefill_logits(ids[:rows], at)
    check(first, want[at], dtype, scale)
    for _ in range(3):           # which workgroup arrives last changes no bit
        m.reset()
        assert np.array_equal(m.prefill_logits(ids[:rows], at), first)
    m.close()
