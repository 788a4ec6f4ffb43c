"""Long rows of a step (portions of prompts) on the attention launch that shares K and V pages between the tokens of a
workgroup, against the same tokens fed eight at a time, which the one-wave items attend."""
import numpy as np
import pytest

from retrograd_amd import engine as E
from retrograd_amd import synth

pytestmark = pytest.mark.gpu

# head width, query heads, kv heads: 1 to 16 query heads per kv head, column tiles that divide sixteen and that do not
HEADS = {"32x4": (32, 16, 4), "64x1": (64, 8, 8), "64x8": (64, 16, 2), "128x4": (128, 8, 2), "128x7": (128, 7, 1), "128x16": (128, 16, 1), "64x3": (64, 9, 3)}


@pytest.mark.parametrize("kv", [E.KV_F16, E.KV_Q8_0, E.KV_Q4_0])
@pytest.mark.parametrize("heads", list(HEADS))
def test_long_rows_match_the_same_tokens_in_pieces(tmp_path, heads, kv):
    """Rows of 12 (the shortest), 31, 33, 100 and 333 tokens behind 0 to 700 resident ones, beside a decode row; the end of a
    row, of a tile of tokens and of a page fall everywhere. One layer; queries and probabilities carry 22 bits and sums are
    f32, which leaves about 1e-6 of the logits: 1e-5 is asked of nine rows in ten. A row's own keys and values come from
    products over other numbers of tokens, so one of them may sit on the other side of a rounding boundary of the cache's
    type: no row is further off than one such step (2^-11 of a value, 1/127 or 1/8 of the largest of a block) in one
    dimension of a head whose whole weight lies on that token."""
    dim, n_head, n_kv = HEADS[heads]
    shape = synth.scaled(synth.TINY_LLAMA, n_layer=1, n_embd=512, n_head=n_head, n_head_kv=n_kv, head_dim=dim, n_ff=512, name="wide-%s" % heads)
    path = tmp_path / "m.gguf"
    synth.write_model(path, shape, seed=3, device="cpu", std=0.08)
    eng = E.Engine(path, E.EngineConfig(n_ctx=8192, n_seq_max=8, n_batch=1024, n_ubatch=1024, kv_dtype=kv))
    rng = np.random.default_rng(8)
    rows = [(0, 700, 12), (1, 65, 100), (2, 0, 333), (3, 640, 31), (4, 1, 33), (5, 95, 1)]
    tokens = [rng.integers(0, shape.n_vocab, before + n) for _, before, n in rows]

    def fill():
        for (slot, before, _), t in zip(rows, tokens):
            eng.seq_rm(slot)
            for at in range(0, before, 8):
                eng.step_logits([(slot, t[at:min(at + 8, before)], at)], [])

    fill()
    want = [(i, j) for i, (_, _, n) in enumerate(rows) for j in range(n)]
    got = eng.step_logits([(slot, t[before:], before) for (slot, before, _), t in zip(rows, tokens)], want)
    fill()
    pieces = []
    for (slot, before, n), t in zip(rows, tokens):
        for at in range(before, before + n, 8):
            part = t[at:min(at + 8, before + n)]
            pieces.append(eng.step_logits([(slot, part, at)], [(0, j) for j in range(len(part))]))
    pieces = np.concatenate(pieces)
    assert np.isfinite(got).all()
    worst = np.linalg.norm(got - pieces, axis=1) / np.linalg.norm(pieces, axis=1)
    print("%s kv %d: nine of ten %.2e, worst row %.2e" % (heads, kv, np.quantile(worst, 0.9), worst.max()), flush=True)
    step = {E.KV_F16: 2.0 ** -11, E.KV_Q8_0: 1 / 127, E.KV_Q4_0: 1 / 8}[kv]
    assert np.quantile(worst, 0.9) <= 1e-5
    assert worst.max() <= step / np.sqrt(dim / 3)          # values of a head spread evenly over +-1: norm sqrt(dim / 3)
    eng.close()
